"""The routes of ffn_residual_fused: gate|up with SiLU * up in its store, the
residual in the down GEMV's store (fp32 and MFMA streaming kernels, with and
without SiLU * up in front) and the separate launches, at each one's edges."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
DEV = "cuda:0"


# (hidden, ffn): pair + fp32 store with 8 / 16 waves; pair + MFMA store at one
# and four row blocks per workgroup and at its most slices; gate|up on the MFMA
# kernel (Q8_0; Q4_0 as before, at the longest rows); pair + separate add (ffn not
# whole 256); SiLU * up in front (hidden past 4096) with one, two and
# four slices per row; nothing fused (hidden not whole 256)
@pytest.mark.parametrize("hidden,ffn", [(256, 256), (2304, 1024), (512, 4352), (4096, 8192), (512, 16128), (768, 16384), (512, 2880),
                                        (4352, 512), (4352, 4352), (4352, 8448), (288, 512)])
@pytest.mark.parametrize("fmt", (O.Q8_0, O.Q4_0))
def test_down_stores_the_residual_sum(zq, orc, fmt, hidden, ffn):
    """With Wo = 0 and a norm weight of 0 every product is 0 and out is x, bit
    for bit.  Otherwise the result is the chain's of separate calls: the GEMV
    sums are the same kernels', so the two differ by the SiLU's expf (2 ulp) and
    the kernels' orders of addition, both within the GEMV bar taken relative to
    the magnitudes the last projection sums."""
    aw = 256
    w = {k: orc.gen_weights(fmt, s, r, c) for k, s, r, c in
         (("o", 900, hidden, aw), ("g", 901, ffn, hidden), ("u", 902, ffn, hidden), ("d", 903, hidden, ffn))}
    dev = {}
    for k, (r, c) in {"o": (hidden, aw), "g": (ffn, hidden), "u": (ffn, hidden), "d": (hidden, ffn)}.items():
        dev[k] = torch.zeros(zq.weight_bytes(fmt, r, c), dtype=torch.uint8, device=DEV)
        dev[k][: w[k].size] = torch.from_numpy(w[k]).to(DEV)
    x, nw, a = (torch.from_numpy(orc.gen_normal(s, n)).to(DEV) for s, n in ((904, hidden), (905, hidden), (906, aw)))
    wsb = zq.ffn_residual_workspace_bytes(hidden, ffn)
    ws = torch.empty(wsb, dtype=torch.uint8, device=DEV)

    def run(att, norm, out):
        zq.ffn_residual_fused_dev(fmt, dev["o"], dev["g"], dev["u"], dev["d"], norm, x, att, out, hidden, aw, ffn,
                                  1e-5, ws, wsb)
        return out

    out = torch.full((hidden + 64,), 7.0, device=DEV)
    run(torch.zeros_like(a), torch.zeros_like(nw), out)
    assert torch.equal(out[:hidden], x) and bool((out[hidden:] == 7.0).all())

    run(a, nw, out)
    t0, h2, g, u, d = (torch.empty(n, device=DEV) for n in (hidden, hidden, ffn, ffn, hidden))
    zq.gemv_dev(fmt, dev["o"], a, t0, hidden, aw)
    h1 = t0 + x
    zq.rms_norm_dev(h1, nw, h2, 1, hidden, 1e-5)
    zq.gemv_dev(fmt, dev["g"], h2, g, ffn, hidden)
    zq.gemv_dev(fmt, dev["u"], h2, u, ffn, hidden)
    f = g / (1.0 + torch.exp(-g)) * u
    zq.gemv_dev(fmt, dev["d"], f, d, hidden, ffn)
    dd = orc.dequantize(fmt, w["d"], hidden * ffn).reshape(hidden, ffn).astype(np.float64)
    mag = np.abs(dd) @ f.abs().double().cpu().numpy() + h1.abs().double().cpu().numpy()
    got, want = out[:hidden].double().cpu().numpy(), (h1 + d).double().cpu().numpy()
    assert np.all(np.abs(got - want) <= 1e-4 + 1e-5 * mag)
    assert torch.equal(run(a, nw, x)[:hidden], out[:hidden])  # in place of x


@pytest.mark.parametrize("ffn", (4096, 4352, 14336))  # down on the fp32 and the MFMA streaming kernel
@pytest.mark.parametrize("u0", (np.inf, 3e11, np.nan))
def test_a_huge_activation_in_front_of_down(zq, orc, ffn, u0):
    """One SiLU * up is infinite, far above the others of its pair, or NaN (an
    infinite up and a gate of -inf): the outputs are infinite with the sign of the
    down weight it meets (NaN at a zero one), keep fp32's precision for the others
    where every weight it meets is 0, or are all NaN."""
    hidden, aw, r0, c0 = 512, 256, 70, 33
    w = {k: orc.gen_weights(O.Q8_0, s, r, c) for k, s, r, c in
         (("o", 910, hidden, aw), ("g", 911, ffn, hidden), ("u", 912, ffn, hidden), ("d", 913, hidden, ffn))}

    def code(k, cols, rows, col):
        """The codes of a column, writable."""
        b = w[k].reshape(-1, cols // 32, 34)
        return b[rows, col // 32, 2 + col % 32:3 + col % 32]

    # column c0 of the normalised vector is huge and reaches up's row r0 alone
    code("g", hidden, slice(None), c0)[:] = code("u", hidden, slice(None), c0)[:] = 0
    code("u", hidden, slice(r0, r0 + 1), c0)[:] = 100
    w["u"].reshape(-1, hidden // 32, 34)[r0, c0 // 32, :2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    if np.isfinite(u0):
        code("d", ffn, slice(None), r0)[:] = 0
    if np.isnan(u0):
        code("g", hidden, slice(r0, r0 + 1), c0)[:] = -100 & 255
        w["g"].reshape(-1, hidden // 32, 34)[r0, c0 // 32, :2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    x, nw, a = orc.gen_normal(914, hidden), orc.gen_normal(915, hidden), np.zeros(aw, np.float32)
    x[c0] = 1.0
    nw[c0] = u0 / 100 if np.isfinite(u0) else 3e38
    shapes = {"o": (hidden, aw), "g": (ffn, hidden), "u": (ffn, hidden), "d": (hidden, ffn)}
    dev = {k: torch.zeros(zq.weight_bytes(O.Q8_0, r, c), dtype=torch.uint8, device=DEV) for k, (r, c) in shapes.items()}
    for k in dev:
        dev[k][: w[k].size] = torch.from_numpy(w[k]).to(DEV)
    wsb = zq.ffn_residual_workspace_bytes(hidden, ffn)
    ws, out = torch.empty(wsb, dtype=torch.uint8, device=DEV), torch.empty(hidden, device=DEV)
    zq.ffn_residual_fused_dev(O.Q8_0, dev["o"], dev["g"], dev["u"], dev["d"], torch.from_numpy(nw).to(DEV),
                              torch.from_numpy(x).to(DEV), torch.from_numpy(a).to(DEV), out, hidden, aw, ffn, 1e-5, ws, wsb)
    W = {k: orc.dequantize(O.Q8_0, w[k], r * c).reshape(r, c).astype(np.float64) for k, (r, c) in shapes.items()}
    h1 = x.astype(np.float64)
    h2 = (h1 / np.sqrt((h1 * h1).mean() + 1e-5)).astype(np.float32) * nw  # fp32: up's sum overflows as there
    with np.errstate(all="ignore"):
        g, u = ((W[p] @ h2).astype(np.float32).astype(np.float64) for p in "gu")
        f = g / (1.0 + np.exp(-g)) * u
        terms = W["d"] * f
        want, mag = h1 + terms.sum(1), np.abs(h1) + np.abs(terms).sum(1)
    got = out.double().cpu().numpy()
    assert np.isfinite(np.delete(f, r0)).all() and abs(u[r0]) > 1e8 and np.isfinite(u[r0]) == np.isfinite(u0)
    if np.isnan(u0):
        assert np.isnan(f[r0]) and np.isnan(got).all()
    elif np.isinf(u0):
        assert np.array_equal(got, want, equal_nan=True) and np.isinf(got).any()
    else:  # the GEMV bar, as above
        assert np.all(np.abs(got - want) <= 1e-4 + 1e-5 * mag)


@pytest.mark.parametrize("ffn", (4352, 14336))
def test_saturated_gates_stay_on_the_digits(zq, orc, ffn):
    """Half of the gates are far below zero, so that nearly half of every pair's
    SiLU * up is next to nothing beside the rest: the down projection is the MFMA
    GEMV's as for any other x (launch_gemv's sums, bit for bit), not the fp32 form
    of values that the digits do not carry, which is several times slower."""
    hidden, aw = 512, 256
    w = {k: orc.gen_weights(O.Q8_0, s, r, c) for k, s, r, c in
         (("o", 920, hidden, aw), ("g", 921, ffn, hidden), ("u", 922, ffn, hidden), ("d", 923, hidden, ffn))}
    dev = {}
    for k, (r, c) in {"o": (hidden, aw), "g": (ffn, hidden), "u": (ffn, hidden), "d": (hidden, ffn)}.items():
        dev[k] = torch.zeros(zq.weight_bytes(O.Q8_0, r, c), dtype=torch.uint8, device=DEV)
        dev[k][: w[k].size] = torch.from_numpy(w[k]).to(DEV)
    x = torch.from_numpy(orc.gen_normal(924, hidden)).to(DEV)
    W = torch.from_numpy(orc.dequantize(O.Q8_0, w["g"], ffn * hidden).reshape(ffn, hidden))
    nw = torch.full((hidden,), float(60.0 / (W @ x.cpu()).std()), device=DEV)  # gates of +-60
    wsb = zq.ffn_residual_workspace_bytes(hidden, ffn)
    ws, out = torch.empty(wsb, dtype=torch.uint8, device=DEV), torch.empty(hidden, device=DEV)
    zq.ffn_residual_fused_dev(O.Q8_0, dev["o"], dev["g"], dev["u"], dev["d"], nw, x, torch.zeros(aw, device=DEV), out, hidden, aw,
                              ffn, 1e-5, ws, wsb)
    f = ws.view(torch.float32)[3 * hidden: 3 * hidden + ffn].clone()  # behind three hidden vectors: SiLU * up
    pairs = f.abs().reshape(-1, 64)
    far = ((pairs != 0) & (pairs < pairs.max(1, keepdim=True).values * 2.0 ** -20)).sum(1)
    assert bool((far >= 16).any())
    d = torch.empty(hidden, device=DEV)
    zq.gemv_dev(O.Q8_0, dev["d"], f, d, hidden, ffn)
    assert torch.equal(out, x + d)
