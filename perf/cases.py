"""The work this library is used for, as a list of cases that can be timed and checked.

Every case is one pass of a model layer, or of one of its blocks, through the public entry
points (raceline_amd.ops, raceline_amd.model): the four linears of a transformer layer, the
output head, a mixture of experts, the engine's MLP step. Sizes are the ones of
raceline_amd.configs (a 9B and a 27B dense layer, a 35B-A3B-style mixture of experts, a
248,320-row head); row counts run from one token to a 2048-token prompt chunk, over what
serving meets: single-token decode, a draft's verification, batched decode, short prompts,
prompt chunks.

listed() names the cases, draw() gives more of the same ranges, prepare() makes the inputs
and packs the weights (what a program keeps), run() is one pass, exact() the same pass in 64
bits in plain torch.
"""

from __future__ import annotations

import math
import os
import tempfile

import torch

GROUP = 64
STD = 0.02                      # weights N(0, STD), as the checkpoints the format comes from
SCALES = {"f16": torch.float16, "bf16": torch.bfloat16}
BOOKS = {"int15": [float(v) for v in (0, 1, 2, 3, 4, 5, 6, 7, -8, -7, -6, -5, -4, -3, -2, -1)],
         "fp4": [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]}
BOOKS["int16"] = [v + 0.5 for v in BOOKS["int15"]]

# (name, K, N) of a layer's linears in the order a layer runs them; "o" and "down" add into
# the residual stream
LAYERS = {"9b": [("qkv", 4096, 6144), ("o", 4096, 4096), ("gate_up", 4096, 24576), ("down", 12288, 4096)],
          "27b": [("qkv", 5120, 7168), ("o", 5120, 5120), ("gate_up", 5120, 34816), ("down", 17408, 5120)]}
RESIDUAL = ("o", "down")
HEAD_K, HEAD_N = 4096, 248320
MOE_H, MOE_I, MOE_E, MOE_TOPK = 2048, 512, 256, 8
MLP_H, MLP_I = 4096, 12288


def listed():
    return [
        # the smallest call: one token through one 4096 x 4096 projection
        dict(name="linear_m1", kind="linear", M=1, K=4096, N=4096, scales="f16"),
        # single-token decode of a 9B layer
        dict(name="layer_9b_m1", kind="layer", layer="9b", M=1, scales="f16"),
        # eight tokens of a 27B layer: a draft's verification, or eight users; bf16 scales, as
        # .rlm files store them
        dict(name="layer_27b_m8", kind="layer", layer="27b", M=8, scales="bf16"),
        # 27 users decoding together, or a very short prompt
        dict(name="layer_9b_m27", kind="layer", layer="9b", M=27, scales="f16"),
        # a short prompt, or the ragged last chunk of a longer one
        dict(name="layer_27b_m300", kind="layer", layer="27b", M=300, scales="bf16"),
        # a full prompt chunk with outlier activations: the largest call
        dict(name="layer_27b_m2048", kind="layer", layer="27b", M=2048, scales="f16", outliers=0.01),
        # the output head over the 16 rows one engine step may ask logits for
        dict(name="head_m16", kind="linear", M=16, K=HEAD_K, N=HEAD_N, scales="bf16"),
        # native-format (codebook) weights on a prompt of 64 tokens
        dict(name="native_fp4_9b_m64", kind="native", layer="9b", M=64, book="fp4"),
        # one token through a mixture of experts: launches and latency
        dict(name="moe_t1", kind="moe", T=1, scales="f16"),
        # batched decode through native-format experts
        dict(name="moe_int15_t24", kind="moe_native", T=24, book="int15"),
        # a prompt chunk through a mixture of experts
        dict(name="moe_t512", kind="moe", T=512, scales="f16"),
        # the engine's whole MLP step (norm, gate/up, SwiGLU, down into the residual) of a 9B
        # layer from a model file, on a prompt of 200 tokens
        dict(name="mlp_9b_t200", kind="mlp", T=200),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "layer", "layer", "head", "native", "native", "moe", "moe",
                       "moe_native", "mlp"])
    scales = rng.choice(["f16", "bf16"])
    if kind == "linear":       # projections of other models: K a multiple of the group, any N
        return dict(kind="linear", M=_log_int(rng, 1, 2048), K=GROUP * _log_int(rng, 8, 192),
                    N=_log_int(rng, 256, 16384), scales=scales)
    if kind == "layer":
        layer = rng.choice(["9b", "27b"])
        return dict(kind="layer", layer=layer, M=_log_int(rng, 1, 2048 if layer == "9b" else 1600), scales=scales,
                    outliers=rng.choice([0.0, 0.01]))
    if kind == "head":
        return dict(kind="linear", M=rng.randint(1, 16), K=HEAD_K, N=HEAD_N - 16 * rng.randint(0, 6000) - rng.randint(0, 9),
                    scales=scales)
    if kind == "native":
        return dict(kind="native", layer="9b", M=_log_int(rng, 1, 1024), book=rng.choice(["int15", "int16", "fp4"]))
    if kind == "moe":
        return dict(kind="moe", T=_log_int(rng, 1, 2048), scales=scales)
    if kind == "moe_native":
        return dict(kind="moe_native", T=_log_int(rng, 1, 1024), book=rng.choice(["int15", "fp4"]))
    return dict(kind="mlp", T=_log_int(rng, 1, 1024))


# ------------------------------------------------------------------ inputs

def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + stream)
    return g


def _affine(gen, N, K, dtype):
    """N(0, STD) weights in 4-bit affine groups of 64 along K: codes [N][K] uint8, scales and
    biases [N][K/64] (round to nearest from the stored scale and bias)."""
    qs, ss, bs = [], [], []
    for r0 in range(0, N, 16384):
        r = min(16384, N - r0)
        W = torch.randn((r, K // GROUP, GROUP), generator=gen, device="cuda") * STD
        lo, hi = W.amin(-1), W.amax(-1)
        s, b = ((hi - lo) / 15).to(dtype), lo.to(dtype)
        q = ((W - b.float().unsqueeze(-1)) / s.float().unsqueeze(-1)).round_().clamp_(0, 15)
        qs.append(q.to(torch.uint8).view(r, K))
        ss.append(s)
        bs.append(b)
    return torch.cat(qs), torch.cat(ss), torch.cat(bs)


def _native(gen, N, K):
    """Codes uniform over the codebook and one fp32 scale per row."""
    q = torch.randint(0, 16, (N, K), generator=gen, device="cuda", dtype=torch.uint8)
    s = torch.rand(N, generator=gen, device="cuda") * 0.004 + 0.002
    return q, s


def _words(q):
    """Codes [N][K] -> 32-bit words [N][K/8], code k at bits 4 (k % 8)."""
    N, K = q.shape
    out = torch.empty((N, K // 8), dtype=torch.int32, device=q.device)
    shifts = torch.arange(0, 32, 4, device=q.device, dtype=torch.int32)
    for r0 in range(0, N, 65536):
        part = q[r0:r0 + 65536].view(-1, K // 8, 8).to(torch.int32)
        out[r0:r0 + 65536] = (part << shifts).sum(-1, dtype=torch.int32)
    return out


def _acts(gen, M, K, outliers=0.0, scale=1.0):
    x = torch.randn((M, K), generator=gen, device="cuda") * scale
    if outliers:
        x = torch.where(torch.rand((M, K), generator=gen, device="cuda") < outliers, x * 20.0, x)
    return x.to(torch.float16)


def _layer_inputs(case, seed):
    """The activations of each linear of a layer and the residual stream."""
    g = _gen(seed, 1)
    M, out = case["M"], case.get("outliers", 0.0)
    xs = {name: _acts(g, M, K, out) for name, K, N in LAYERS[case["layer"]]}
    h = torch.randn((M, LAYERS[case["layer"]][1][2]), generator=g, device="cuda")
    return xs, h


def _moe_inputs(case, seed):
    g = _gen(seed, 1)
    T = case["T"]
    x = _acts(g, T, MOE_H)
    logits = torch.randn((T, MOE_E + 1), generator=g, device="cuda") * 1.5
    h = torch.randn((T, MOE_H), generator=g, device="cuda")
    return x, logits, h


def _mlp_inputs(case, seed):
    g = _gen(seed, 1)
    h = torch.randn((case["T"], MLP_H), generator=g, device="cuda")
    post = torch.rand(MLP_H, generator=g, device="cuda") + 0.5
    return h, post


def _mlp_weights(seed):
    g = _gen(seed, 2)
    return _affine(g, 2 * MLP_I, MLP_H, torch.bfloat16), _affine(g, MLP_H, MLP_I, torch.bfloat16)


class _MlpStep:
    """An open engine over a one-layer model file, closed with the state that holds it."""

    def __init__(self, engine, h):
        self.engine, self.h = engine, h

    def __del__(self):
        try:
            self.engine.close()
        except Exception:
            pass


def _open_mlp(case, seed):
    from raceline_amd import rlm, synth
    from raceline_amd.model import Engine

    h, post = _mlp_inputs(case, seed)
    gu, dn = _mlp_weights(seed)

    def blocked(q, s, b, parts):
        N, K = q.shape                       # N a multiple of the format's 256-row block
        two = q.view(N // 256, 128, 2, K)
        w = (two[:, :, 0] | (two[:, :, 1] << 4)).transpose(1, 2).contiguous()
        sb = [v.view(torch.int16).view(N // 256, 256, K // GROUP).transpose(1, 2).contiguous().cpu().numpy().view("uint16")
              for v in (s, b)]
        spans = [(i * (N // parts), N // parts) for i in range(parts)]
        return w.cpu().numpy(), sb[0], sb[1], N, spans

    fd, path = tempfile.mkstemp(suffix=".rlm")
    os.close(fd)
    try:
        w = rlm.Writer(path)
        w.begin("layer.0")
        w.add_float("layers.0.post_norm", post.cpu().numpy())
        w.add_blocked_packed("layers.0.mlp.gate_up", ["gate", "up"], blocked(*gu, 2))
        w.add_blocked_packed("layers.0.mlp.down", ["out"], blocked(*dn, 1))
        w.end()
        w.finish(rlm.affine_meta(synth.model_config(MLP_H, 1, MLP_I, 1024)))
        return _MlpStep(Engine(path, max_chunk=max(8, case["T"])), h)
    finally:
        os.unlink(path)


def prepare(case, seed):
    from raceline_amd import ops

    kind = case["kind"]
    if kind == "mlp":
        return _open_mlp(case, seed)
    if kind == "linear":
        q, s, b = _affine(_gen(seed, 2), case["N"], case["K"], SCALES[case["scales"]])
        return dict(kind=kind, x=_acts(_gen(seed, 1), case["M"], case["K"]), w=ops.pack_affine(_words(q), s, b))
    if kind in ("layer", "native"):
        xs, h = _layer_inputs(case, seed)
        ws = {}
        for i, (name, K, N) in enumerate(LAYERS[case["layer"]]):
            if kind == "layer":
                q, s, b = _affine(_gen(seed, 2 + i), N, K, SCALES[case["scales"]])
                ws[name] = ops.pack_affine(_words(q), s, b)
            else:
                q, s = _native(_gen(seed, 2 + i), N, K)
                ws[name] = ops.pack_native(_words(q), s, case["book"])
            del q
        return dict(kind=kind, x=xs, w=ws, h=h)
    x, logits, h = _moe_inputs(case, seed)
    E1, H, I = MOE_E + 1, MOE_H, MOE_I
    if kind == "moe":
        dt = SCALES[case["scales"]]
        gq, gs, gb = _affine(_gen(seed, 2), E1 * 2 * I, H, dt)
        dq, ds, db = _affine(_gen(seed, 3), E1 * H, I, dt)
        w = ops.pack_moe((_words(gq), gs, gb), (_words(dq), ds, db), MOE_E, H, I)
        return dict(kind=kind, x=x, logits=logits, h=h, w=w)
    gq, gs = _native(_gen(seed, 2), E1 * 2 * I, H)
    dq, ds = _native(_gen(seed, 3), E1 * H, I)
    gu = ops.pack_moe_native(_words(gq), gs, 2 * I, case["book"])
    dn = ops.pack_moe_native(_words(dq), ds, H, case["book"])
    cs = torch.rand(I, generator=_gen(seed, 4), device="cuda") * 0.5 + 0.75
    return dict(kind=kind, x=x, logits=logits, h=h, gu=gu, dn=dn, cs=cs,
                slots=torch.arange(E1, dtype=torch.int32, device="cuda"))


# ------------------------------------------------------------------ one pass

def run(state):
    from raceline_amd import ops

    if isinstance(state, _MlpStep):
        return {"h": state.engine.mlp(0, state.h)}
    kind = state["kind"]
    if kind == "linear":
        return {"y": ops.linear(state["x"], state["w"])}
    if kind in ("layer", "native"):
        linear = ops.linear if kind == "layer" else ops.linear_native
        x, w, h = state["x"], state["w"], state["h"]
        qkv = linear(x["qkv"], w["qkv"])
        linear(x["o"], w["o"], out=h, accum=True)
        gate_up = linear(x["gate_up"], w["gate_up"])
        linear(x["down"], w["down"], out=h, accum=True)
        return {"qkv": qkv, "gate_up": gate_up, "h": h}
    if kind == "moe":
        return {"h": ops.moe(state["x"], state["logits"], state["w"], MOE_TOPK, state["h"])}
    return {"h": ops.moe_native(state["x"], state["logits"], state["gu"], state["dn"], state["slots"], MOE_TOPK,
                                state["h"], cs=state["cs"])}


# ------------------------------------------------------------------ the same in 64 bits

def _mm64(x, q, s, b):
    """x [M][K] times the dequantized rows, in 64 bits, by blocks of rows."""
    N, K = q.shape
    x = x.double()
    out = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device)
    for r0 in range(0, N, 16384):
        r1 = min(N, r0 + 16384)
        W = (q[r0:r1].view(-1, K // GROUP, GROUP).double() * s[r0:r1].double().unsqueeze(-1)
             + b[r0:r1].double().unsqueeze(-1))
        out[:, r0:r1] = x @ W.view(r1 - r0, K).t()
    return out


def _mm64_native(x, q, s, book):
    levels = torch.tensor(BOOKS[book], dtype=torch.float64, device=x.device)
    N = q.shape[0]
    x = x.double()
    out = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device)
    for r0 in range(0, N, 16384):
        r1 = min(N, r0 + 16384)
        W = levels[q[r0:r1].long()] * s[r0:r1].double().unsqueeze(-1)
        out[:, r0:r1] = x @ W.t()
    return out


def _silu(v):
    return v / (1 + torch.exp(-v))


def _moe64(x, logits, h, gate_up, down, cs=None):
    """h plus the routed experts' and the shared expert's MLPs of x; gate_up(e, rows) and
    down(e, act) are the products with expert e's matrices."""
    T = x.shape[0]
    l = logits.double()
    top, sel = torch.topk(l[:, :MOE_E], MOE_TOPK, dim=1)
    w = torch.softmax(top, dim=1)
    out = h.double()
    for e in range(MOE_E + 1):
        if e < MOE_E:
            tok, slot = torch.nonzero(sel == e, as_tuple=True)
            if tok.numel() == 0:
                continue
            we = w[tok, slot]
        else:
            tok = torch.arange(T, device=x.device)
            we = torch.sigmoid(l[:, MOE_E])
        g = gate_up(e, x[tok])
        act = _silu(g[:, :MOE_I]) * g[:, MOE_I:]
        if cs is not None:
            act = act * cs.double()
        out.index_add_(0, tok, down(e, act) * we.unsqueeze(-1))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        h, post = _mlp_inputs(case, seed)
        gu, dn = _mlp_weights(seed)
        h, post = h.double(), post.double()
        xn = h / torch.sqrt((h * h).mean(-1, keepdim=True) + 1e-6) * post
        g = _mm64(xn, *gu)
        return {"h": h + _mm64(_silu(g[:, :MLP_I]) * g[:, MLP_I:], *dn)}
    if kind == "linear":
        q, s, b = _affine(_gen(seed, 2), case["N"], case["K"], SCALES[case["scales"]])
        return {"y": _mm64(_acts(_gen(seed, 1), case["M"], case["K"]), q, s, b)}
    if kind in ("layer", "native"):
        xs, h = _layer_inputs(case, seed)
        out = {"h": h.double()}
        for i, (name, K, N) in enumerate(LAYERS[case["layer"]]):
            if kind == "layer":
                y = _mm64(xs[name], *_affine(_gen(seed, 2 + i), N, K, SCALES[case["scales"]]))
            else:
                y = _mm64_native(xs[name], *_native(_gen(seed, 2 + i), N, K), case["book"])
            if name in RESIDUAL:
                out["h"] += y
            else:
                out[name] = y
        return out
    x, logits, h = _moe_inputs(case, seed)
    E1, H, I = MOE_E + 1, MOE_H, MOE_I
    if kind == "moe":
        dt = SCALES[case["scales"]]
        gu = _affine(_gen(seed, 2), E1 * 2 * I, H, dt)
        dn = _affine(_gen(seed, 3), E1 * H, I, dt)

        def rows(m, e, n):
            return [v[e * n:(e + 1) * n] for v in m]

        return {"h": _moe64(x, logits, h, lambda e, a: _mm64(a, *rows(gu, e, 2 * I)),
                            lambda e, a: _mm64(a, *rows(dn, e, H)))}
    gq, gs = _native(_gen(seed, 2), E1 * 2 * I, H)
    dq, ds = _native(_gen(seed, 3), E1 * H, I)
    cs = torch.rand(I, generator=_gen(seed, 4), device="cuda") * 0.5 + 0.75
    return {"h": _moe64(x, logits, h,
                        lambda e, a: _mm64_native(a, gq[e * 2 * I:(e + 1) * 2 * I], gs[e * 2 * I:(e + 1) * 2 * I], case["book"]),
                        lambda e, a: _mm64_native(a, dq[e * H:(e + 1) * H], ds[e * H:(e + 1) * H], case["book"]), cs)}


# ------------------------------------------------------------------ what a pass cannot do without

def _linear_work(M, K, N, residual=False, native=False):
    weights = K * N // 2 + (4 * N if native else 4 * N * (K // GROUP))
    return weights + 2 * M * K + (8 if residual else 4) * M * N, 2 * M * N * K


def work(case):
    kind = case["kind"]
    if kind == "linear":
        parts = [_linear_work(case["M"], case["K"], case["N"])]
    elif kind in ("layer", "native"):
        parts = [_linear_work(case["M"], K, N, name in RESIDUAL, kind == "native")
                 for name, K, N in LAYERS[case["layer"]]]
    elif kind == "mlp":
        T = case["T"]
        # the residual rows in and out; both matrices once
        parts = [(2 * MLP_I * MLP_H // 2 + 4 * 2 * MLP_I * (MLP_H // GROUP) + 8 * T * MLP_H, 4 * T * MLP_I * MLP_H),
                 (MLP_I * MLP_H // 2 + 4 * MLP_H * (MLP_I // GROUP), 2 * T * MLP_I * MLP_H)]
    else:
        T, H, I = case["T"], MOE_H, MOE_I
        experts = 1 + MOE_E * (1 - (1 - MOE_TOPK / MOE_E) ** T)      # distinct experts T tokens are expected to pick
        per_group = 4 if kind == "moe" else 0
        one = 3 * H * I // 2 + per_group * 3 * H * I // GROUP + (0 if kind == "moe" else 4 * (2 * I + H))
        parts = [(experts * one + T * (2 * H + 4 * (MOE_E + 1) + 8 * H), 2 * T * (MOE_TOPK + 1) * 3 * H * I)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """About four times the largest error seen against exact(), per kind of case."""
    kind = case["kind"]
    if kind == "native":
        # fp16 products of exact levels summed in fp32: 3e-7
        return {"rel": 1.2e-6, "max": 2e-5}
    if kind in ("linear", "layer"):
        # affine: the matrix cores' sums over exact 4-bit codes as fp16 subnormals, 1e-5; with
        # outlier activations 3.6e-5 (residual rows, where the terms of a sum cancel most)
        return {"rel": 1.5e-4, "max": 1.5e-3}
    if kind in ("moe", "moe_native"):
        # the experts' SwiGLU outputs pass through fp16: 3.2e-5 of the residual row
        return {"rel": 1.3e-4, "max": 2e-3}
    # the engine's step also rounds the normed rows to fp16: 3.4e-4
    return {"rel": 1.4e-3, "max": 1.4e-2}
