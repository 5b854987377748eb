"""The prefill kernels (gemm.hip, gemm_mid.hip at 32 and 64 rows, gemm_few.hip), each named in
the call: a row has the same bits whichever of them runs, at the edges of their row tiles (8,
16, 32, 64 and 128 rows), with a ragged N (tiles of 16, 32, 128 and 256 features cut), an odd
number of groups (the last pair half empty), a single group, more bias steps than run ahead of
the K loop, a split K, bf16 scales, ACCUM and every native codebook; and the rows match the
fp64 product. The cases that test_gpu_linear.py, test_gpu_native.py and test_gpu_precision.py
run on the kernel a call's sizes choose run here on each kernel."""

import numpy as np
import pytest

import oracle as O
from tests import routes as R
from tests.qdata import make_layer, make_x, sample_cols, to_dev, upload
from tests.test_gpu_linear import GEMM_CASES, SPLIT_GEMM_CASES
from tests.test_gpu_precision import GEMM_SHAPES, mixed_x, scaled_x

pytestmark = pytest.mark.gpu
TOL = 1e-3

# 8192, 8256 (an odd number of groups), 9216 and 32960 inputs split K in two; 32960 (odd too)
# goes through the prep pass that walks a row twice
SHAPES = [(1024, 1000, "f16"), (1088, 300, "bf16"), (320, 1500, "bf16"), (320, 40, "f16"), (64, 48, "bf16"),
          (8192, 1000, "f16"), (8256, 1000, "bf16"), (9216, 2100, "bf16"), (32960, 40, "f16"), (32960, 40, "bf16")]
ROWS = [9, 16, 17, 31, 32, 33, 64, 65, 127, 224, 257, 300]
M_ALL = 400


def _compare(x, h, w, kernels, ref, cols, what):
    """Calls of some of x's rows on each kernel against the full-tile kernel's over all of them
    (its last row tile ragged), plain and added into h, whose rows have a stride of their own."""
    import torch

    M, N = h.shape
    full = R.linear_on(R.FULL, x, w)
    full_acc = R.linear_on(R.FULL, x, w, out=h.clone(), accum=True)
    O.check_close(full.cpu().numpy()[:, cols], ref, TOL, what)
    O.check_close(full_acc.cpu().numpy()[:, cols], ref + h.cpu().numpy()[:, cols], TOL, f"{what}, ACCUM")
    for r in ROWS:
        r0 = (7 * r) % (M - r)
        for k in kernels:
            name = f"{what}: {r} rows on {R.NAMES[k]}"
            assert torch.equal(R.linear_on(k, x[r0:r0 + r], w), full[r0:r0 + r]), name
            wide = torch.full((r, N + 5), -3.0, device=h.device)
            wide[:, :N] = h[r0:r0 + r]
            R.linear_on(k, x[r0:r0 + r], w, out=wide, accum=True)
            assert torch.equal(wide[:, :N], full_acc[r0:r0 + r]), f"{name}, ACCUM"
            assert (wide[:, N:] == -3.0).all(), f"{name} wrote past the last column"


@pytest.mark.parametrize("K,N,sd", SHAPES)
def test_same_bits_on_every_kernel(gpu, K, N, sd):
    import torch

    q, s, b = make_layer(K + N, N, K, sd)
    x_np = make_x(K, M_ALL, K, outliers=0.01)
    h = to_dev(np.random.default_rng(K + 1).standard_normal((M_ALL, N)).astype(np.float32), gpu)
    cols = sample_cols(N, min(N, 128), seed=K)
    ref = O.linear_affine_f64(x_np, q[cols], s[cols], b[cols], sd)
    x = to_dev(x_np, gpu)
    wide = torch.zeros((M_ALL, K + 64), dtype=torch.float16, device=gpu)     # a row stride that is not K
    wide[:, :K] = x
    _compare(wide[:, :K], h, upload(q, s, b, sd, gpu), R.AFFINE, ref, cols, f"K={K} N={N} {sd}")


@pytest.mark.parametrize("book", ["int15", "int16", "fp4"])
@pytest.mark.parametrize("K,N", [(1088, 1000), (64, 48), (320, 300), (8256, 1000)])
def test_native_same_bits_on_every_kernel(gpu, book, K, N):
    import torch

    from raceline_amd import ops

    rng = np.random.default_rng(K)
    q = rng.integers(0, 16, size=(N, K), dtype=np.uint8)
    s_row = rng.uniform(0.002, 0.02, size=N).astype(np.float32)
    w = ops.pack_native(to_dev(O.pack_nibbles_u32(q).view(np.int32), gpu), to_dev(s_row, gpu), book)
    x_np = make_x(K + 3, M_ALL, K)
    h = to_dev(rng.standard_normal((M_ALL, N)).astype(np.float32), gpu)
    cols = sample_cols(N, min(N, 128), seed=K)
    ref = O.linear_native_f64(x_np, q[cols], s_row[cols], book)
    wide = torch.zeros((M_ALL, K + 64), dtype=torch.float16, device=gpu)
    wide[:, :K] = to_dev(x_np, gpu)
    _compare(wide[:, :K], h, w, R.NATIVE, ref, cols, f"{book} K={K} N={N}")


@pytest.mark.parametrize("kernel", R.AFFINE)
@pytest.mark.parametrize("M,K,N", GEMM_CASES)
def test_prefill_cases(gpu, kernel, M, K, N):
    """The shapes of test_gemm_parity on each kernel, with outlier activations."""
    sd = "f16" if (M + N) % 2 else "bf16"
    q, s, b = make_layer(M * 7 + N, N, K, sd)
    x = make_x(M + K, M, K, outliers=0.01)
    y = R.linear_on(kernel, to_dev(x, gpu), upload(q, s, b, sd, gpu)).cpu().numpy()
    cols = sample_cols(N, 256, seed=K)
    O.check_close(y[:, cols], O.linear_affine_f64(x, q[cols], s[cols], b[cols], sd), TOL, f"M={M} K={K} N={N}")


@pytest.mark.parametrize("kernel", R.AFFINE)
@pytest.mark.parametrize("M,K,N,sd", [c for c in SPLIT_GEMM_CASES if c[2] <= 2048] + [(200, 1024, 384, "f16")])
def test_split_and_accumulate_cases(gpu, kernel, M, K, N, sd):
    """The split and ACCUM shapes of test_gpu_linear.py on each kernel; a repeat call gives the
    same bits (a split call leaves its counters zero)."""
    import torch

    q, s, b = make_layer(M + K + N, N, K, sd)
    x_np = make_x(M + 5, M, K, outliers=0.01)
    w, x = upload(q, s, b, sd, gpu), to_dev(x_np, gpu)
    cols = sample_cols(N, 256, seed=K)
    ref = O.linear_affine_f64(x_np, q[cols], s[cols], b[cols], sd)
    y = R.linear_on(kernel, x, w)
    assert torch.equal(R.linear_on(kernel, x, w), y)
    O.check_close(y.cpu().numpy()[:, cols], ref, TOL, f"M={M} K={K} N={N}")
    y0 = np.random.default_rng(M).standard_normal((M, N)).astype(np.float32)
    ya = R.linear_on(kernel, x, w, out=to_dev(y0, gpu), accum=True).cpu().numpy()
    O.check_close(ya[:, cols], ref + y0[:, cols], TOL, f"ACCUM M={M} K={K} N={N}")


@pytest.mark.parametrize("kernel", R.AFFINE)
@pytest.mark.parametrize("M,K,N", GEMM_SHAPES)
def test_small_and_mixed_activations(gpu, kernel, M, K, N):
    """The precision shapes of test_gpu_precision.py on each kernel: rows of 1e-4, rows that mix
    1e-4 with O(1) entries (held to the bar row by row), entries near 60000, a row of subnormals
    and an all-zero row."""
    sd = "f16" if M % 3 else "bf16"
    q, s, b = make_layer(M + K + N, N, K, sd)
    x = np.concatenate([scaled_x(K + M, M // 2, K, 1e-4), mixed_x(K, M - M // 2, K)])
    rng = np.random.default_rng(71)
    x[0] = np.clip(rng.standard_normal(K) * 5e3, -6e4, 6e4)
    x[0, 5] = 60000.0
    x[1] = rng.integers(-1023, 1024, size=K) * 2.0 ** -24
    x[2] = 0.0
    y = R.linear_on(kernel, to_dev(x, gpu), upload(q, s, b, sd, gpu)).cpu().numpy()
    ref = O.linear_affine_f64(x, q, s, b, sd)
    assert (y[2] == 0).all()
    for m in range(M):
        if m != 2:
            O.check_close(y[m:m + 1], ref[m:m + 1], TOL, f"row {m} on {R.NAMES[kernel]}")


@pytest.mark.parametrize("kernel", R.AFFINE)
@pytest.mark.parametrize("sd", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N", [(40, 2048, 272), (33, 8256, 1000)])
def test_one_hot_rows(gpu, kernel, sd, M, K, N):
    """x = e_k on each kernel gives the dequantized weight exactly, with biases below fp16's
    normal range among them."""
    rng = np.random.default_rng(80 + M + K)
    q = rng.integers(0, 16, size=(N, K), dtype=np.uint8)
    sf = rng.uniform(0.001, 0.012, size=(N, K // 64)).astype(np.float32)
    bf = (-7.5 * sf + rng.uniform(-0.01, 0.01, size=sf.shape)).astype(np.float32)
    bf = np.where(rng.random(sf.shape) < 0.25, rng.uniform(-2.0 ** -15, 2.0 ** -15, size=sf.shape), bf)
    s, b = O.scale_from_f32(sf, sd), O.scale_from_f32(bf.astype(np.float32), sd)
    ks = rng.choice(K, size=M, replace=False)
    ks[0], ks[1] = K - 1, 64 * (K // 128) + 1
    x = np.zeros((M, K), np.float16)
    x[np.arange(M), ks] = 1.0
    y = R.linear_on(kernel, to_dev(x, gpu), upload(q, s, b, sd, gpu)).cpu().numpy()
    ref = O.dequant_affine(q, s, b, sd)[:, ks].T.astype(np.float32)
    np.testing.assert_array_equal(y.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("book", [None, "int15", "int16", "fp4"])
@pytest.mark.parametrize("K", [320, 1024])   # an odd number of groups; one that fills the ring exactly
def test_infinities_and_nans_stay_in_their_rows(gpu, book, K):
    """Rows that hold an infinity or a NaN give the same values on every kernel, and leave the
    other rows' bits alone: what pads a tile's rows, the last pair or the ring past the last
    pair adds nothing."""
    import torch

    from raceline_amd import ops

    M, N = 70, 300
    q, s, b = make_layer(K, N, K)
    w = upload(q, s, b, "f16", gpu)
    if book:
        w = ops.pack_native(to_dev(O.pack_nibbles_u32(q).view(np.int32), gpu), torch.full((N,), 0.01, device=gpu), book)
    clean = make_x(K, M, K)
    x_np = clean.copy()
    bad = [1, 8, 33, 69]
    x_np[1, 5], x_np[8, K - 1], x_np[33, 64], x_np[69, 2] = np.inf, -np.inf, np.nan, np.inf
    x_np[69, 3] = -np.inf
    kernels = R.NATIVE if book else R.AFFINE
    want = R.linear_on(R.FULL, to_dev(x_np, gpu), w).cpu().numpy()
    plain = R.linear_on(R.FULL, to_dev(clean, gpu), w).cpu().numpy()
    good = [m for m in range(M) if m not in bad]
    np.testing.assert_array_equal(want[good], plain[good])
    assert not np.isfinite(want[bad]).any()
    for k in kernels:
        got = R.linear_on(k, to_dev(x_np, gpu), w).cpu().numpy()
        np.testing.assert_array_equal(got, want, err_msg=R.NAMES[k])     # NaNs compare equal here


@pytest.mark.parametrize("book,M,K,N", [(0, 27, 4096, 4096), (0, 300, 5120, 7168), (0, 2048, 5120, 34816),
                                        (1, 64, 4096, 4096), (3, 64, 4096, 24576), (3, 2048, 4096, 24576)])
def test_chosen_kernel_runs(gpu, book, M, K, N):
    """A call that names no kernel gives the bits of the one its sizes choose (layer sizes)."""
    import torch

    from raceline_amd import ops, synth

    x = synth.random_activations(M, K, 5, gpu)
    if book == 0:
        w = synth.random_affine(N, K, 3, gpu)
        y = ops.linear(x, w)
    else:
        g = torch.Generator(device=gpu)
        g.manual_seed(3)
        codes = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), generator=g, device=gpu, dtype=torch.int32)
        w = ops.pack_native(codes, torch.full((N,), 0.004, device=gpu), {1: "int15", 3: "fp4"}[book])
        y = ops.linear_native(x, w)
    assert torch.equal(y, R.linear_on(R.chosen(book, M, K, N), x, w))
    assert torch.equal(y, R.linear_on(R.FULL, x, w))


@pytest.mark.parametrize("kernel", R.AFFINE)
def test_replays_in_a_graph_with_a_split(gpu, kernel):
    """A split call captured in a graph gives the eager bits on every replay (its arrival
    counters are left zero), with eager calls of other sizes between the replays."""
    import torch

    from raceline_amd import ops, synth

    K, N, M = 8192, 1024, 70
    wt = synth.random_affine(N, K, 3, gpu)
    x = synth.random_activations(M, K, 4, gpu)
    want = R.linear_on(kernel, x, wt)
    y = torch.zeros((M, N), device=gpu)
    R.linear_on(kernel, x, wt, out=y)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        R.linear_on(kernel, x, wt, out=y)
    for k in range(4):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {k}"
        ops.linear(x[:20 + k], wt)
