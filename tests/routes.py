"""Running one named prefill kernel (include/rlq.h, rlq_prefill_route): the three of them give
a row the same bits, and which one a call runs depends on its sizes."""

FULL, MID32, MID64, FEW = 1, 2, 3, 4
NAMES = {FULL: "full", MID32: "mid32", MID64: "mid64", FEW: "few"}
AFFINE = (FULL, MID32, MID64, FEW)
NATIVE = (FULL, MID32, MID64)


def chosen(book, M, K, N, scale_dtype=0):
    """The kernel a call of these sizes runs; book: 0 (affine) or the native codebook's code."""
    from raceline_amd import lib

    return lib.call("rlq_prefill_route", book, scale_dtype, M, K, N)


def linear_on(route, x, w, out=None, accum=False):
    """ops.linear, or ops.linear_native for a NativeWeight, on one prefill kernel."""
    import torch

    from raceline_amd import lib, ops

    M, K, N = x.shape[0], w.K, w.N
    if out is None:
        out = torch.empty((M, N), dtype=torch.float32, device=x.device)
    ws = ops._WS.get(x.device, ops.workspace_bytes(M, K, N))
    tail = (out.data_ptr(), out.stride(0), int(accum), ws.data_ptr(), ws.numel(), ops._stream())
    if isinstance(w, ops.NativeWeight):
        lib.call("rlq_linear_native_prefill", route, x.data_ptr(), x.stride(0), M, K, N, w.packed.data_ptr(),
                 w.s_row.data_ptr(), w.code, *tail)
    else:
        lib.call("rlq_linear_affine_prefill", route, x.data_ptr(), x.stride(0), M, K, N, w.packed.data_ptr(), w.code,
                 *tail)
    return out
