"""The fp32-activation GEMMs (zq_gemm_split.hip on split f16 activations,
zq_gemm_skinny.hip for few tokens): edges of their tiles and K splits, rows of very different magnitude, and
non-finite activations; and, on the CPU, that its kernels neither spill nor
use packed fp32 arithmetic."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from tests.tolerance import assert_close

ALL = (O.Q8_0, O.Q4_0, O.Q6_K, O.Q4_K, O.Q5_K)


@pytest.fixture
def small(zq):
    old = zq.set_min_elements(0)  # the slot declines tiny shapes otherwise
    yield
    zq.set_min_elements(old)


# Tiles are 128 tokens by 128 or 256 rows (32 or 64 by 32 for few tokens),
# stages 32 k (three in flight), super-blocks 256: one of each, one less and one
# more, an odd count of stages, one stage, fewer groups than waves, and K long
# enough to split.
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
@pytest.mark.parametrize("m,n,k", [(140, 700, 2048), (20, 70, 512)])  # split activations; few tokens
@pytest.mark.parametrize("fmt", ALL)
def test_row_magnitudes_and_non_finite(zq, orc, small, fmt, m, n, k):
    """Each row has its own power of two, so a row's result does not depend on
    its scale; an infinite or NaN activation stays in its row, and with codes
    of one plane and no offset gives what the product of the dequantised
    weights gives."""
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
    assert not np.isfinite(got[7:9]).any()
    if fmt in (O.Q8_0, O.Q4_0):
        W = orc.dequantize(fmt, w, n * k).reshape(n, k)
        with np.errstate(invalid="ignore"):
            for r, c in ((7, 17), (8, 300)):
                want = Z[r, c] * W[:, c]  # the finite terms do not matter beside it
                assert np.array_equal(got[r], want, equal_nan=True)
    zq.release(w)


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


class SkinnyPlan(ctypes.Structure):
    _fields_ = [("ks", ctypes.c_uint32), ("us", ctypes.c_double)]


def takes_split(zq, fmt, m, n, k, ws_bytes):
    """Whether the library's planners send this call to the split kernels (else
    to the few-token kernel): the comparison launch_gemm_f32_batch makes."""
    L, z = zq.lib(), ctypes.c_size_t
    skinny, split = L._ZN2zq20plan_gemm_skinny_f32Eimmmm, L._ZN2zq13gemm_split_usEimmmPKvm
    skinny.restype, skinny.argtypes = SkinnyPlan, [ctypes.c_int, z, z, z, z]
    split.restype, split.argtypes = ctypes.c_double, [ctypes.c_int, z, z, z, ctypes.c_void_p, z]
    use = min(ws_bytes, zq.gemm_workspace_bytes(fmt, m, n, k, zq.ACT_F32))
    return skinny(fmt, m, n, k, use // (m * n * 4)).us > split(fmt, m, n, k, 256 if use else None, use)


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
