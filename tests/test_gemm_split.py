"""The fp32-activation GEMMs (zq_gemm_split.hip on split f16 activations,
zq_gemm_skinny.hip for few tokens): edges of their tiles and K splits, a
workspace for some of the tokens, rows of very different magnitude, non-finite
and extreme activations, the rounding's common part; and, on the CPU, that the
kernels neither spill nor use packed fp32 arithmetic."""
import os
import re
import subprocess

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from tests.plans import launch_split, skinny_waves, split_bytes, split_plan, takes_split
from tests.tolerance import assert_close

ALL = (O.Q8_0, O.Q4_0, O.Q6_K, O.Q4_K, O.Q5_K)


@pytest.fixture
def small(zq):
    old = zq.set_min_elements(0)  # the slot declines tiny shapes otherwise
    yield
    zq.set_min_elements(old)


# Whichever kernel the dispatch takes (mostly the few-token one: 32 or 64 tokens
# by 32 rows): one tile, one less and one more, an odd count of groups, fewer
# groups than waves, and K long enough to split.  The split kernels' own edges
# are below.
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ALL)
@pytest.mark.parametrize("m,n,blocks", [(1, 1, 8), (2, 129, 8), (127, 255, 8), (128, 256, 16), (129, 257, 24), (257, 130, 8),
                                        (70, 300, 128), (3, 33, 448), (130, 40, 264), (32, 32, 8), (33, 31, 16),
                                        (64, 65, 136), (300, 700, 256), (200, 3000, 256)])
def test_edges(zq, orc, small, fmt, m, n, blocks):
    k = 32 * blocks
    w = orc.gen_weights(fmt, 500 + n, n, k)
    X = orc.gen_normal(501 + m, m * k)
    # against the float64 product: at K = 8448 the fp32 oracle's own rounding
    # takes up to 0.96 of the bar (Q5_K), this kernel's 0.18
    assert_close(zq.gemm(fmt, w, X, m, n, k, zq.ACT_F32), orc.gemm_f64(fmt, w, X, m, n, k)[0], f"fmt={fmt} {m}x{n}x{k}")
    zq.release(w)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", (O.Q8_0, O.Q4_0))
@pytest.mark.parametrize("m", (5, 47, 700))
@pytest.mark.parametrize("blocks", (1, 2, 3, 5, 7, 31, 67))
def test_any_number_of_blocks(zq, orc, small, fmt, m, blocks):
    n, k = 270, 32 * blocks
    w = orc.gen_weights(fmt, 510 + blocks, n, k)
    X = orc.gen_normal(511, m * k)
    assert_close(zq.gemm(fmt, w, X, m, n, k, zq.ACT_F32), orc.gemm_f32(fmt, w, X, m, n, k), f"fmt={fmt} k={k}")
    zq.release(w)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,split", [(140, 700, 2048, False), (20, 70, 512, False), (140, 700, 4096, True)])
@pytest.mark.parametrize("fmt", ALL)
def test_row_magnitudes_and_non_finite(zq, orc, small, fmt, m, n, k, split):
    """Each row has its own power of two, so a row's result does not depend on
    its scale; an infinite or NaN activation stays in its row, and an infinite
    one gives what the products of the dequantised weights give."""
    assert takes_split(zq, fmt, m, n, k) == split
    w = orc.gen_weights(fmt, 520, n, k)
    X = orc.gen_normal(521, m * k).reshape(m, k)
    base = zq.gemm(fmt, w, X, m, n, k, zq.ACT_F32).reshape(m, n)
    Z = X.copy()
    for r, s in ((3, 2.0 ** -100), (4, 2.0 ** 90), (5, 0.0), (6, 2.0 ** -130)):
        Z[r] *= np.float32(s)
    Z[7, 17] = np.inf
    Z[8, 300] = -np.inf
    Z[9, 40] = np.nan
    got = zq.gemm(fmt, w, Z, m, n, k, zq.ACT_F32).reshape(m, n)
    same = [r for r in range(m) if r not in (3, 4, 5, 6, 7, 8, 9)]
    assert np.array_equal(got[same], base[same])
    assert np.array_equal(got[3], base[3] * np.float32(2.0 ** -100)) and np.array_equal(got[4], base[4] * np.float32(2.0 ** 90))
    assert np.all(got[5] == 0) and np.all(np.isfinite(got[6]))
    assert np.all(np.isnan(got[9]))
    W = orc.dequantize(fmt, w, n * k).reshape(n, k)
    with np.errstate(invalid="ignore"):
        for r, c in ((7, 17), (8, 300)):
            want = Z[r, c] * W[:, c]  # the finite terms do not matter beside it
            assert np.array_equal(got[r], want, equal_nan=True)
    zq.release(w)


# The split kernels, called directly: tiles are 128 tokens by 128 or 256 rows,
# stages 32 k with three in flight, super-blocks 256.  (tokens, rows, tile
# columns): one tile, one less and one more of each, and grids of two rounds of
# 128-column tiles, which take the 256-column form.  Q8_0 / Q4_0 take any count
# of blocks (the main loop is six stages long, and one or two are fewer than it
# has in flight); the others whole super-blocks.
def split_case(zq, orc, fmt, m, n, blocks, planes, room=None):
    """Result and launches against the float64 product (the GEMM bar; the fp32
    oracle's own rounding takes up to 0.96 of it at long K)."""
    k = 32 * blocks
    w = orc.gen_weights(fmt, 550 + n, n, k)
    X = orc.gen_normal(551 + m, m * k)
    dw = torch.full((zq.weight_bytes(fmt, n, k),), 255, dtype=torch.uint8, device="cuda:0")
    dw[: w.size] = torch.from_numpy(w).to("cuda:0")
    Y = torch.full((m * n + 64,), 7.0, device="cuda:0")
    ws_bytes = split_bytes(zq, fmt, room or m, k) + planes * m * n * 4
    ws = torch.full((ws_bytes + 256,), 255, dtype=torch.uint8, device="cuda:0")
    launches = launch_split(zq, fmt, dw, torch.from_numpy(X).to("cuda:0"), Y, ws, ws_bytes, m, n, k)
    W = orc.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64)
    want = X.reshape(m, k).astype(np.float64) @ W.T
    assert bool((Y[m * n:] == 7.0).all()) and bool((ws[ws_bytes:] == 255).all())
    assert_close(Y[: m * n].cpu().numpy(), want.reshape(-1), f"fmt={fmt} {m}x{n}x{k}")
    return launches


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ALL)
@pytest.mark.parametrize("m,n,cols", [(1, 1, 128), (127, 129, 128), (128, 128, 128), (129, 255, 128), (257, 270, 128),
                                      (255, 16639, 256), (257, 11009, 256), (129, 16641, 256), (256, 16640, 256)])
def test_split_tiles(zq, orc, fmt, m, n, cols):
    counts = (1, 2, 3, 5, 7, 31, 67) if fmt in (O.Q8_0, O.Q4_0) else (8, 16, 24, 72)
    for blocks in counts[:3] if cols == 256 else counts:
        assert split_plan(zq, fmt, m, n, 32 * blocks, 0) == (cols, 1)
        assert split_case(zq, orc, fmt, m, n, blocks, 0) == 2


# K splits: even, with a last one that is shorter, and the most
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ALL)
@pytest.mark.parametrize("m,n,blocks,planes", [(130, 40, 264, 3), (130, 1500, 128, 5), (1, 33, 448, 31)])
def test_split_k(zq, orc, fmt, m, n, blocks, planes):
    assert split_plan(zq, fmt, m, n, 32 * blocks, planes)[1] > 1
    assert split_case(zq, orc, fmt, m, n, blocks, planes) == 3


# room for the split activations of `room` tokens: the others follow, on the
# few-token kernel (one launch) or on the split one again (two)
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ALL)
@pytest.mark.parametrize("m,n,room,launches", [(300, 700, 256, 3), (129, 33, 128, 3), (500, 9000, 256, 4)])
def test_room_for_some_tokens(zq, orc, fmt, m, n, room, launches):
    assert split_case(zq, orc, fmt, m, n, 16, 0, room) == launches


def extremes(orc, fmt, w, m, n, k):
    """Activations with, in rows of their own, infinities (one, two of one sign,
    two of opposite signs, every element), a NaN beside one, magnitudes at the
    two ends of the fp32 range, and one element far above the others, where it
    meets most zero weights."""
    X = orc.gen_normal(531, m * k).reshape(m, k)
    zeros = (orc.dequantize(fmt, w, n * k).reshape(n, k) == 0).sum(0).argmax()
    X[12, zeros] = 1e8
    X[13, zeros] = -3e12
    X[14, zeros] = 1e5
    X[3, 17] = np.inf
    X[4, 40] = -np.inf
    X[5, [1, k - 1]] = np.inf
    X[6, [2, 300]] = np.inf, -np.inf
    X[7, [9, 33]] = np.inf, np.nan
    X[8] = np.where(np.arange(k) % 2, np.inf, -np.inf)
    X[9] *= np.float32(2.0 ** 120)
    X[10] *= np.float32(2.0 ** -100)
    X[11, 5] *= np.float32(2.0 ** 124)
    return X


def check_extremes(orc, fmt, w, X, got, m, n, k):
    """Against the sums of products with the dequantised weights: infinite and NaN
    where those are, with their signs, and otherwise within 8 + sqrt(k) roundings
    of the magnitudes summed (2^-24 of them each: the products', the split's and,
    as a random walk, those of k additions to a sum that one element can make
    large from the start).  Q4_K / Q5_K multiply a code and its group's offset
    apart, so there the group's largest weight counts for each."""
    W = orc.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64)
    top = np.abs(W)
    if fmt in (O.Q4_K, O.Q5_K):
        top = np.repeat(top.reshape(n, k // 32, 32).max(2), 32, axis=1)
    for r in range(min(m, 24)):
        with np.errstate(invalid="ignore", over="ignore"):
            terms = X[r].astype(np.float64) * W
            want = terms.sum(1)
        finite = np.isfinite(want)
        assert np.array_equal(got[r][~finite], want[~finite].astype(np.float32), equal_nan=True), f"row {r}"
        if finite.any():
            mag = (np.abs(X[r].astype(np.float64)) * top).sum(1)[finite]
            err = np.abs(got[r][finite].astype(np.float64) - want[finite])
            assert np.all(err <= (8 + k ** 0.5) * 2.0 ** -24 * mag), f"row {r}: {np.nanmax(err / mag) * 2.0 ** 24} roundings"


def run_dev(zq, fmt, w, X, m, n, k, ws_bytes):
    dw = torch.zeros(zq.weight_bytes(fmt, n, k), dtype=torch.uint8, device="cuda:0")
    dw[: w.size] = torch.from_numpy(w).to("cuda:0")
    Y = torch.full((m * n + 64,), 7.0, device="cuda:0")
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device="cuda:0")
    zq.gemm_dev(fmt, dw, torch.from_numpy(X).to("cuda:0"), Y, m, n, k, zq.ACT_F32, ws if ws_bytes else None, ws_bytes)
    assert bool((Y[m * n:] == 7.0).all())
    return Y[: m * n].cpu().numpy().reshape(m, n)


# one and two token tiles without a workspace; split activations with K splits
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,split", [(20, 70, 512, False), (50, 33, 768, False), (130, 1500, 4096, True)])
@pytest.mark.parametrize("fmt", ALL)
def test_extreme_activations(zq, orc, fmt, m, n, k, split):
    w = orc.gen_weights(fmt, 530, n, k)
    X = extremes(orc, fmt, w, m, n, k)
    ws_bytes = zq.gemm_workspace_bytes(fmt, m, n, k, zq.ACT_F32) if split else 0
    assert takes_split(zq, fmt, m, n, k, ws_bytes) == split
    check_extremes(orc, fmt, w, X, run_dev(zq, fmt, w, X, m, n, k, ws_bytes), m, n, k)


# The matrix cores round the sums of 16-bit products down; a kernel that let this
# add up would move every output the same way (measured: by 0.4 to 0.6 of the
# errors' spread), which a model's later layers feel more than as much noise.
# 33600 outputs or more: chance alone gives 0.01.
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,split", [(20, 1700, 4096, False), (48, 700, 4096, False), (130, 1500, 4096, True)])
@pytest.mark.parametrize("fmt", ALL)
def test_errors_have_no_common_part(zq, orc, fmt, m, n, k, split):
    w = orc.gen_weights(fmt, 540, n, k)
    X = orc.gen_normal(541, m * k).reshape(m, k)
    ws_bytes = zq.gemm_workspace_bytes(fmt, m, n, k, zq.ACT_F32) if split else 0
    assert takes_split(zq, fmt, m, n, k, ws_bytes) == split
    e = run_dev(zq, fmt, w, X, m, n, k, ws_bytes) - orc.gemm_f64(fmt, w, X.reshape(-1), m, n, k)[0].reshape(m, n)
    assert abs(e.mean()) < 0.1 * np.sqrt((e * e).mean())


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ALL)
def test_rows_marked_for_fp32(zq, orc, fmt):
    """Only rows that f16 hi + lo under one power of two do not carry are marked (the
    rows' exponents follow the split activations in the workspace): not those with
    many elements next to nothing, as SiLU leaves, or one 2^13 above the others, as
    some models' activations have."""
    m, n, k = 128, 40, 2048
    w = orc.gen_weights(fmt, 560, n, k)
    X = orc.gen_normal(561, m * k).reshape(m, k)
    X[1, 7] = np.inf
    X[2, 9] = 1e8
    X[3, [9, 700, 701]] = 1e8, -1e8, 3e7
    X[4, 9] = 1e5
    X[5, ::2] *= 1e-12
    X[6, :1900] *= 1e-12
    X[7, 9] = 8000.0
    X[8] = 0.0
    X[9, 9] = np.nan
    X[10] = np.exp2(-np.arange(k) % 60).astype(np.float32)  # evenly over 60 powers of two
    X[11, 1:] = 0.0
    marked = {1, 2, 3}
    dw = torch.zeros(zq.weight_bytes(fmt, n, k), dtype=torch.uint8, device="cuda:0")
    dw[: w.size] = torch.from_numpy(w).to("cuda:0")
    nbytes = split_bytes(zq, fmt, m, k)
    ws, Y = torch.zeros(nbytes, dtype=torch.uint8, device="cuda:0"), torch.empty(m * n, device="cuda:0")
    launch_split(zq, fmt, dw, torch.from_numpy(X).to("cuda:0"), Y, ws, nbytes, m, n, k)
    at = m * k * 4 + (m * (k // 256) * 32 if fmt in (O.Q4_K, O.Q5_K) else 0)
    ex = ws[at: at + 4 * m].view(torch.int32).cpu().numpy()
    assert set(np.flatnonzero(ex == 1 << 20)) == marked
    rows = np.array([r for r in range(m) if r not in (1, 9)])  # the two are test_extreme_activations'
    W = orc.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64)
    Xr = X[rows].astype(np.float64)
    mag = np.abs(Xr) @ np.abs(W).T + (fmt in (O.Q4_K, O.Q5_K)) * (np.abs(Xr).sum(1)[:, None] * np.abs(W).max())
    err = np.abs(Y.cpu().numpy().reshape(m, n)[rows] - Xr @ W.T)
    assert np.all(err <= (8 + k ** 0.5) * 2.0 ** -24 * mag)


# Short K and a large grid: workgroups of four and two waves, without a workspace;
# and a batch with a small matrix that takes eight, whose bits are those of single
# calls.
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,nw", [(1000, 4096, 256, 2), (130, 14300, 256, 4), (577, 4096, 1024, 4), (70, 14336, 512, 2)])
@pytest.mark.parametrize("fmt", ALL)
def test_fewer_waves(zq, orc, fmt, m, n, k, nw):
    assert skinny_waves(zq, fmt, m, n, k) == nw and skinny_waves(zq, fmt, m, 33, k) == 8
    rows = (33, n)
    ws = [orc.gen_weights(fmt, 570 + i, r, k) for i, r in enumerate(rows)]
    X = orc.gen_normal(571, m * k).reshape(m, k)
    W = orc.dequantize(fmt, ws[1], n * k).reshape(n, k).astype(np.float64)
    got = run_dev(zq, fmt, ws[1], X, m, n, k, 0)
    assert_close(got.reshape(-1), (X.astype(np.float64) @ W.T).reshape(-1), f"fmt={fmt} {m}x{n}x{k}")
    single = [run_dev(zq, fmt, w, X, m, r, k, zq.gemm_workspace_bytes(fmt, m, r, k, zq.ACT_F32)) for w, r in zip(ws, rows)]
    ds = [torch.zeros(zq.weight_bytes(fmt, r, k), dtype=torch.uint8, device="cuda:0") for r in rows]
    for d, w in zip(ds, ws):
        d[: w.size] = torch.from_numpy(w).to("cuda:0")
    Ys = [torch.empty(m * r, device="cuda:0") for r in rows]
    need = zq.gemm_batch_workspace_bytes(fmt, rows, m, k, zq.ACT_F32)
    buf = torch.empty(need + 16, dtype=torch.uint8, device="cuda:0")
    zq.gemm_batch_dev(fmt, torch.from_numpy(X).to("cuda:0"), list(zip(ds, Ys, rows)), m, k, zq.ACT_F32, buf, need)
    for Y, one in zip(Ys, single):
        assert np.array_equal(Y.cpu().numpy(), one.reshape(-1))


@pytest.mark.parametrize("src", ("zq_gemm_split.hip", "zq_gemm_skinny.hip"))
def test_generated_code(tmp_path, src):
    from zeninfer_amd.build import FLAGS, HIPCC, SRC
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path / "split.s"
    flags = [f for f in FLAGS if f not in ("-shared", "-fPIC")]
    r = subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", "-o", str(out), os.path.join(SRC, src)],
                       capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    asm = out.read_text()
    sizes = re.findall(r"^\s*\.amdhsa_private_segment_fixed_size (\d+)", asm, re.M)
    assert sizes and set(sizes) == {"0"}
    assert not re.findall(r"^\s*v_pk_(?:fma|add|mul)_f32\b", asm, re.M)
