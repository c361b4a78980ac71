"""The streaming GEMVs on rows that are not whole 16-byte units: Q6_K of any
number of super-blocks and Q8_0 / Q4_0 of any number of blocks -- each remainder
and count of slices, every start of a row within 16 bytes, one task and several,
and Q6_K's paired gate|up form."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.tolerance import assert_close

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda:0"


def place(zq, fmt, w, rows, cols, fill):
    """The weights with `fill` in the tail pad, which no result may depend on."""
    buf = torch.full((zq.weight_bytes(fmt, rows, cols),), fill, dtype=torch.uint8, device=DEV)
    buf[: w.size] = torch.from_numpy(w).to(DEV)
    return buf


def check(zq, orc, fmt, cols, rows, seed):
    x = orc.gen_normal(seed, cols)
    xd = torch.from_numpy(x).to(DEV)
    ws = [orc.gen_weights(fmt, seed + 10 + i, r, cols) for i, r in enumerate(rows)]
    got = []
    for fill in (0, 255):
        ys = [torch.full((r + 16,), 7.0, device=DEV) for r in rows]
        ds = [place(zq, fmt, w, r, cols, fill) for w, r in zip(ws, rows)]
        if len(rows) == 1:
            zq.gemv_dev(fmt, ds[0], xd, ys[0], rows[0], cols)
        else:
            zq.gemv_batch_dev(fmt, xd, [(d, y, r) for d, y, r in zip(ds, ys, rows)], cols)
        got.append([y.cpu().numpy() for y in ys])
    for w, r, y, y2 in zip(ws, rows, *got):
        assert np.all(y[r:] == 7.0) and np.array_equal(y, y2)
        assert_close(y[:r], orc.gemv_f32(fmt, w, x, r, cols), f"fmt={fmt} cols={cols} rows={r}")


# super-blocks per row: under one slice, one more and one less than whole
# slices, the most; rows: fewer than a step, odd, and past the 2-rows-per-step line
@pytest.mark.parametrize("sb", (1, 2, 5, 7, 9, 15, 20, 27, 33, 43, 54, 63))
@pytest.mark.parametrize("rows", ((1,), (17,), (4099,), (33, 7, 130)))
def test_any_number_of_super_blocks(zq, orc, sb, rows):
    check(zq, orc, O.Q6_K, 256 * sb, rows, 1000 + sb)


# blocks per row: one, odd and even, around one, two and four slices of 64
# pairs, the most; rows: fewer than a step, 8 and 16 waves a workgroup
@pytest.mark.parametrize("blocks", (1, 2, 3, 9, 63, 90, 127, 129, 130, 253, 257, 345, 449, 510, 511))
@pytest.mark.parametrize("rows", ((1,), (19,), (4099,), (33, 7, 130)))
@pytest.mark.parametrize("fmt", (O.Q8_0, O.Q4_0))
def test_any_number_of_blocks(zq, orc, fmt, blocks, rows):
    check(zq, orc, fmt, 32 * blocks, rows, 1100 + blocks)


def streamed(zq, fmt, cols, rows):
    """The library's own rule for which rows the streaming kernels take."""
    f = zq.lib()._ZN2zq13gemv_streamedEijj
    f.restype, f.argtypes = ctypes.c_bool, [ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32]
    return f(fmt, cols, rows)


# blocks (Q6_K: super-blocks) per row as above, with rows enough for the streaming
# kernels: past the two-rows-per-step line with a last partial block of rows, 8
# waves a workgroup, three tasks; and the few rows that long odd ones take
@pytest.mark.parametrize("fmt,blocks,rows", [
    *((O.Q6_K, b, r) for b in (2, 3, 4) for r in ((8190,), (4090,), (4000, 7, 4183))),
    *((f, b, (8190,)) for f in (O.Q8_0, O.Q4_0) for b in (23, 29, 63, 90, 127, 129, 130, 253, 257, 345, 449, 510, 511)),
    *((f, b, (4000, 7, 4183)) for f in (O.Q8_0, O.Q4_0) for b in (63, 90, 257)),
    *((f, b, (2045,)) for f in (O.Q8_0, O.Q4_0) for b in (127, 130, 257)),
    *((f, b, (67,)) for f in (O.Q8_0, O.Q4_0) for b in (225, 511))])
def test_rows_that_are_streamed(zq, orc, fmt, blocks, rows):
    cols = (256 if fmt == O.Q6_K else 32) * blocks
    assert streamed(zq, fmt, cols, sum(rows))
    check(zq, orc, fmt, cols, rows, 1200 + blocks)


@pytest.mark.parametrize("sb", (1, 3, 20))
def test_an_infinity_reaches_every_row(zq, orc, sb):
    """A code times an infinity is one, or NaN where the code is 0: no row is finite."""
    cols, rows = 256 * sb, 40
    w = orc.gen_weights(O.Q6_K, 1020, rows, cols)
    x = orc.gen_normal(1021, cols)
    x[cols - 1] = np.inf
    y = torch.empty(rows, device=DEV)
    zq.gemv_dev(O.Q6_K, place(zq, O.Q6_K, w, rows, cols, 255), torch.from_numpy(x).to(DEV), y, rows, cols)
    assert not np.isfinite(y.cpu().numpy()).any()


@pytest.mark.parametrize("hidden,ffn", [(256, 768), (256, 8192), (2304, 2816), (5120, 1280)])
def test_paired_gate_up(zq, orc, hidden, ffn):
    """ffn_residual_fused against separate calls (as for the other formats: the
    SiLU's expf and orders of addition, within the GEMV bar)."""
    aw = 256
    shapes = {"o": (hidden, aw), "g": (ffn, hidden), "u": (ffn, hidden), "d": (hidden, ffn)}
    w = {k: orc.gen_weights(O.Q6_K, 1030 + i, r, c) for i, (k, (r, c)) in enumerate(shapes.items())}
    dev = {k: place(zq, O.Q6_K, w[k], r, c, 255) for k, (r, c) in shapes.items()}
    x, nw, a = (torch.from_numpy(orc.gen_normal(s, n)).to(DEV) for s, n in ((1034, hidden), (1035, hidden), (1036, aw)))
    wsb = zq.ffn_residual_workspace_bytes(hidden, ffn)
    ws, out = torch.empty(wsb, dtype=torch.uint8, device=DEV), torch.empty(hidden, device=DEV)
    zq.ffn_residual_fused_dev(O.Q6_K, dev["o"], dev["g"], dev["u"], dev["d"], nw, x, a, out, hidden, aw, ffn, 1e-5, ws, wsb)
    t0, h2, g, u, d = (torch.empty(n, device=DEV) for n in (hidden, hidden, ffn, ffn, hidden))
    zq.gemv_dev(O.Q6_K, dev["o"], a, t0, hidden, aw)
    h1 = t0 + x
    zq.rms_norm_dev(h1, nw, h2, 1, hidden, 1e-5)
    zq.gemv_dev(O.Q6_K, dev["g"], h2, g, ffn, hidden)
    zq.gemv_dev(O.Q6_K, dev["u"], h2, u, ffn, hidden)
    f = g / (1.0 + torch.exp(-g)) * u
    zq.gemv_dev(O.Q6_K, dev["d"], f, d, hidden, ffn)
    dd = orc.dequantize(O.Q6_K, w["d"], hidden * ffn).reshape(hidden, ffn).astype(np.float64)
    mag = np.abs(dd) @ f.abs().double().cpu().numpy() + h1.abs().double().cpu().numpy()
    err = np.abs(out.double().cpu().numpy() - (h1 + d).double().cpu().numpy())
    assert np.all(err <= 1e-4 + 1e-5 * mag)
