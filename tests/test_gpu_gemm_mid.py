"""The prefill kernels for calls with few output tiles (gemm_mid.hip, and gemm_few.hip for a few
rows) against the one for many (gemm.hip): a row has the same bits whichever of them its call
runs, at the edges of the row tiles (8, 16, 32 and 64 rows) and of the few-row kernel's range
(256 tiles of 32 x 32), with a ragged N (tiles of 16, 32 and 128 features cut), an odd number
of groups (the last pair half empty), more bias steps than run ahead of the K loop, a split K,
bf16 scales, ACCUM and every native codebook; and the rows match the fp64 product."""

import numpy as np
import pytest

import oracle as O
from tests.qdata import make_layer, make_x, sample_cols, to_dev, upload

pytestmark = pytest.mark.gpu
TOL = 1e-3

# K, N, scales, rows of the call whose 128 x 256 tiles fill the chip (gemm.hip); the third
# splits K in two
SHAPES = [(1024, 1000, "f16", 16384), (1088, 300, "bf16", 16384), (8192, 1000, "f16", 4352), (320, 1500, "bf16", 16384),
          (320, 40, "f16", 40000), (9216, 4200, "bf16", 4352)]
ROWS = [9, 16, 17, 31, 32, 33, 64, 65, 127, 224, 257, 300]


@pytest.mark.parametrize("K,N,sd,M", SHAPES)
def test_same_bits_as_the_full_kernel(gpu, K, N, sd, M):
    import torch

    from raceline_amd import ops

    q, s, b = make_layer(K + N, N, K, sd)
    wt = upload(q, s, b, sd, gpu)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(K)
    x = torch.randn((M, K), generator=gen, device=gpu).to(torch.float16)
    h = torch.randn((M, N), generator=gen, device=gpu)
    full = ops.linear(x, wt, kernel=2)
    full_acc = ops.linear(x, wt, out=h.clone(), accum=True, kernel=2)
    cols = sample_cols(N, min(N, 128), seed=K)
    for r in ROWS:
        r0 = (7 * r) % (M - r)
        y = ops.linear(x[r0:r0 + r], wt, kernel=2)
        assert torch.equal(y, full[r0:r0 + r]), f"{r} rows"
        wide = torch.full((r, N + 5), -3.0, device=gpu)          # a row stride that is not N
        wide[:, :N] = h[r0:r0 + r]
        ops.linear(x[r0:r0 + r], wt, out=wide, accum=True, kernel=2)
        assert torch.equal(wide[:, :N], full_acc[r0:r0 + r]), f"{r} rows, ACCUM"
        assert (wide[:, N:] == -3.0).all(), "wrote past the last column"
        ref = O.linear_affine_f64(x[r0:r0 + r].cpu().numpy(), q[cols], s[cols], b[cols], sd)
        O.check_close(y.cpu().numpy()[:, cols], ref, TOL, f"{r} rows K={K} N={N}")


@pytest.mark.parametrize("book", ["int15", "int16", "fp4"])
def test_native_same_bits_as_the_full_kernel(gpu, book):
    import torch

    from raceline_amd import ops

    K, N, M = 1088, 1000, 16384
    rng = np.random.default_rng(K)
    q = rng.integers(0, 16, size=(N, K), dtype=np.uint8)
    s_row = rng.uniform(0.002, 0.02, size=N).astype(np.float32)
    nw = ops.pack_native(to_dev(O.pack_nibbles_u32(q).view(np.int32), gpu), to_dev(s_row, gpu), book)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(K)
    x = torch.randn((M, K + 64), generator=gen, device=gpu).to(torch.float16)[:, :K]   # a row stride that is not K
    full = ops.linear_native(x, nw, kernel=2)
    cols = sample_cols(N, 128, seed=K)
    for r in ROWS:
        y = ops.linear_native(x[5:5 + r], nw, kernel=2)
        assert torch.equal(y, full[5:5 + r]), f"{r} rows"
        ref = O.linear_native_f64(x[5:5 + r].cpu().numpy(), q[cols], s_row[cols], book)
        O.check_close(y.cpu().numpy()[:, cols], ref, TOL, f"{book} {r} rows")


def test_replays_in_a_graph_with_a_split(gpu):
    """A split call captured in a graph gives the eager bits on every replay (its arrival
    counters are left zero), with eager calls of other sizes between the replays."""
    import torch

    from raceline_amd import ops, synth

    K, N, M = 8192, 1024, 70
    wt = synth.random_affine(N, K, 3, gpu)
    x = synth.random_activations(M, K, 4, gpu)
    want = ops.linear(x, wt)
    y = torch.zeros((M, N), device=gpu)
    ops.linear(x, wt, out=y)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.linear(x, wt, out=y)
    for k in range(4):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {k}"
        ops.linear(x[:20 + k], wt)
