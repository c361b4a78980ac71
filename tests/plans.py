"""The library's own choice of fp32-activation GEMM kernel, for tests that are
about one of them: the internal planners, which need no GPU (without one they
plan for the MI355X's 256 CUs)."""
import ctypes

_Z = ctypes.c_size_t


class SkinnyPlan(ctypes.Structure):
    _fields_ = [("ks", ctypes.c_uint32), ("nw", ctypes.c_uint32), ("us", ctypes.c_double)]


class SplitPlan(ctypes.Structure):
    _fields_ = [("wn", ctypes.c_int), ("ks", ctypes.c_uint32), ("blocks", ctypes.c_uint32), ("us", ctypes.c_double)]


def _function(zq, name, result, *args):
    f = getattr(zq.lib(), name)
    f.restype, f.argtypes = result, list(args)
    return f


def takes_split(zq, fmt, m, n, k, ws_bytes=None):
    """Whether a call goes to the split kernels (else to the few-token kernel):
    the comparison launch_gemm_f32_batch makes, for a caller's workspace of
    ws_bytes or, without, for the library's own buffers (the host calls)."""
    if ws_bytes is None:
        use = _function(zq, "_ZN2zq19gemm_f32_best_bytesEimmm", _Z, ctypes.c_int, _Z, _Z, _Z)(fmt, m, n, k)
    else:
        use = min(ws_bytes, zq.gemm_workspace_bytes(fmt, m, n, k, zq.ACT_F32))
    skinny = _function(zq, "_ZN2zq20plan_gemm_skinny_f32Eimmmm", SkinnyPlan, ctypes.c_int, _Z, _Z, _Z, _Z)
    split = _function(zq, "_ZN2zq13gemm_split_usEimmmPKvm", ctypes.c_double, ctypes.c_int, _Z, _Z, _Z, ctypes.c_void_p, _Z)
    return skinny(fmt, m, n, k, use // (m * n * 4)).us > split(fmt, m, n, k, 256 if use else None, use)


def skinny_waves(zq, fmt, m, n, k):
    """Waves of the few-token kernel's workgroups, without a workspace (m > 32)."""
    return _function(zq, "_ZN2zq20plan_gemm_skinny_f32Eimmmm", SkinnyPlan, ctypes.c_int, _Z, _Z, _Z, _Z)(fmt, m, n, k, 0).nw


def split_bytes(zq, fmt, m, k):
    """Workspace of the split activations of m tokens."""
    return _function(zq, "_ZN2zq16gemm_split_bytesEimm", _Z, ctypes.c_int, _Z, _Z)(fmt, m, k)


def split_plan(zq, fmt, m, n, k, planes):
    """(tile columns, K splits) of the split kernels with room for `planes` planes."""
    f = _function(zq, "_ZN2zq15plan_gemm_splitEimmmm", SplitPlan, ctypes.c_int, _Z, _Z, _Z, _Z)
    p = f(fmt, m, n, k, planes)
    return 64 * p.wn, p.ks


def launch_split(zq, fmt, w, X, Y, ws, ws_bytes, m, n, k):
    """The split kernels whatever the dispatch would take, on device tensors and
    the default stream; the number of launches."""
    p = ctypes.c_void_p
    f = _function(zq, "_ZN2zq17launch_gemm_splitEiPKhPKfPfPvmmmmP12ihipStream_tPj", ctypes.c_int, ctypes.c_int, p, p, p, p,
                  _Z, _Z, _Z, _Z, p, ctypes.POINTER(ctypes.c_uint32))
    assert w.numel() >= zq.weight_bytes(fmt, n, k) and X.numel() >= m * k and Y.numel() >= m * n and ws.numel() >= ws_bytes
    launches = ctypes.c_uint32()
    e = f(fmt, w.data_ptr(), X.data_ptr(), Y.data_ptr(), ws.data_ptr(), ws_bytes, m, n, k, None, ctypes.byref(launches))
    assert e == 0, f"hipError {e}"
    return launches.value
