"""The matrix-core GEMM for prefill chunks (xjh_gemm) against the oracle's
matmul (src/xiaoju-pipe/core/xj_cpu.c:36-54), a float64 product of the same
dequantized weights, and the dot-product GEMV (xjh_gemv). The GEMM's
products are exact (f16 halves of the activations times small-integer
weights) and only its fp32 accumulation rounds: ~1e-7 of the float64
product; the GEMV's 21-bit activations put it ~1e-6 away."""
import ctypes as C

import numpy as np
import pytest

import oracle as orc
import xjpipe as xp
from conftest import rel_l2
from helpers import random_blocks

pytestmark = pytest.mark.gpu


def _weights(t, rows, k, seed):
    return xp.quantize(t, xp.fill_normal(rows * k, seed, 0.02).reshape(rows, k))


@pytest.mark.parametrize("t,rows,k", [
    (xp.Q4_K, 4096, 1024),     # Q4_K 4096 x 1024
    (xp.Q6_K, 3584, 1024),     # Q6_K 3584 x 1024
    (xp.Q4_K, 1000, 2560),     # rows not a multiple of 16 or 64
    (xp.Q6_K, 517, 9216),      # few rows: K split over work-groups, reduce launch
    (xp.Q4_K, 33, 256),        # one block per row
    (xp.Q4_K, 2560, 4096),     # 320 units: 160 work-groups of two (ssm_out / wo)
    (xp.Q6_K, 1024, 9216),     # 288 units: 144 work-groups of two, a row group over 18
])
@pytest.mark.parametrize("T", [1, 16, 17, 40, 64])
def test_gemm_matches_oracle_and_gemv(t, rows, k, T):
    blob = _weights(t, rows, k, 2000 + rows + k)
    xs = xp.fill_normal(T * k, 91 + T, 1.0).reshape(T, k)
    w = xp.DevWeight(t, blob, rows, k)
    got = xp.gemm(w, xs)
    want = orc.matmul(t, blob, k, rows, xs)
    assert rel_l2(got, want) < 1e-3
    wd = orc.dequant_rows(t, blob, rows, k).astype(np.float64)
    ref64 = xs.astype(np.float64) @ wd.T
    assert rel_l2(got, ref64) < 1e-6
    # the GEMV on the same inputs: both within ~1e-6 of the float64 product
    gv = np.concatenate([xp.gemv(w, xs[i:i + 5]) for i in range(0, T, 5)])
    assert rel_l2(gv, ref64) < 3e-6
    assert rel_l2(got, gv) < 3e-6
    assert np.max(np.abs(got - gv)) <= 5e-6 * np.max(np.abs(gv))


@pytest.mark.parametrize("t", [xp.Q4_K, xp.Q6_K])
def test_gemm_random_blocks_and_residual_add(t):
    """Blocks with every field random (edge fp16 scales included), and the
    residual-add form y += W x."""
    rows, k, T = 300, 1024, 37
    blob = random_blocks(t, rows, k, 5)
    w = xp.DevWeight(t, blob, rows, k)
    xs = xp.fill_normal(T * k, 8, 1.0).reshape(T, k)
    wd = orc.dequant_rows(t, blob, rows, k).astype(np.float64)
    finite = np.isfinite(wd).all(axis=1)
    ref64 = xs.astype(np.float64) @ np.where(np.isfinite(wd), wd, 0).T
    got = xp.gemm(w, xs)
    assert rel_l2(got[:, finite], ref64[:, finite]) < 1e-6
    base = xp.fill_normal(T * rows, 9, 1.0).reshape(T, rows)
    got2 = xp.gemm(w, xs, add_to=base)
    assert np.array_equal(got2[:, finite], (base + got)[:, finite])


def test_gemm_rejects_unsupported():
    blob = _weights(xp.Q4_K, 64, 256, 3)
    w = xp.DevWeight(xp.Q4_K, blob, 64, 256)
    with pytest.raises(xp.XjError):
        xp.gemm(w, np.zeros((65, 256), np.float32))
    q8 = xp.DevWeight(xp.Q8_0, _weights(xp.Q8_0, 64, 256, 4), 64, 256)
    with pytest.raises(xp.XjError):
        xp.gemm(q8, np.zeros((16, 256), np.float32))


@pytest.mark.parametrize("t,rows,k", [
    (xp.Q4_K, 18432, 256),     # more row tiles than work-groups: five per work-group, K unsplit
    (xp.Q4_K, 2560, 4096),     # two row tiles per work-group, K in three splits
    (xp.Q4_K, 1009, 2560),     # a last row tile of one row
    (xp.Q6_K, 2560, 9216),     # Q6_K, K in three splits of 48 chunks
    (xp.Q6_K, 33, 512),        # eight chunks over eight wavefronts and two splits
    (xp.Q4_K, 5, 256),         # four chunks: wavefronts without work
])
@pytest.mark.parametrize("T", [33, 48, 49, 63])
def test_narrow_gemm_edges(t, rows, k, T):
    """33 to 64 tokens: edges of the token tiles (three up to 48, else four),
    row tiles and splits of the inner elements. Activations of 22 bits, exact
    products and fp32 sums: up to 2.8e-7 of float64 measured (Q4_K), two and a
    half times that allowed; the residual-add form adds to what is there."""
    blob = _weights(t, rows, k, 3000 + rows + k)
    xs = xp.fill_normal(T * k, 191 + T, 1.0).reshape(T, k)
    w = xp.DevWeight(t, blob, rows, k)
    got = xp.gemm(w, xs)
    ref64 = xs.astype(np.float64) @ orc.dequant_rows(t, blob, rows, k).astype(np.float64).T
    assert rel_l2(got, ref64) < 7e-7
    base = xp.fill_normal(T * rows, 19, 1.0).reshape(T, rows)
    assert np.array_equal(xp.gemm(w, xs, add_to=base), base + got)


@pytest.mark.parametrize("t,rows,k,T,kind", [
    (xp.Q4_K, [2560], 4096, 128, 1),              # two slices on the narrow kernel
    (xp.Q4_K, [300, 41], 1024, 129, 1),           # ... and a slice of one token
    (xp.Q4_K, [517], 256, 1000, 2),               # the wide kernel with fewer units than work-groups, one block per row
    (xp.Q4_K, [7001], 1280, 257, 2),              # 420 units: ranges of one or two that cross row groups and token groups
    (xp.Q4_K, [2600, 1000, 16, 17], 2816, 1000, 2),   # 1320 units in ranges of five or six, four segments in shared row groups
    (xp.Q6_K, [3001], 1280, 1000, 2),             # an odd block count: d in either half of its word
    (xp.Q6_K, [2560], 9216, 300, 2),              # tiles of 36 blocks shared by ten work-groups
    (xp.Q6_K, [517, 33], 2816, 385, 2),           # a token group of one token
    (xp.Q6_K, [9000], 512, 300, 2),               # 216 units on 216 work-groups
    (xp.Q4_K, [9000], 768, 640, 2),               # 540 units of whole tiles: stored directly and shared
])
def test_piece_gemm_matches_float64(t, rows, k, T, kind):
    """The GEMM of prompt pieces against float64 products of the dequantized
    weights, and which kernel took it: ragged rows and tokens, several
    segments, ranges that cross tiles, tiles shared by several work-groups; plain,
    with an RMSNorm input, and added to what is there. Products of the 22-bit
    activations are exact and sums fp32; Q4_K subtracts the minimum terms'
    sum. Measured 2.5 to 4.0e-7 (Q4_K) and 0.9 to 1.5e-7 (Q6_K), twice the
    largest allowed."""
    bound = 8e-7 if t == xp.Q4_K else 3e-7
    ws = [xp.DevWeight(t, _weights(t, r, k, 4000 + r + k), r, k) for r in rows]
    wd = [orc.dequant_rows(t, _weights(t, r, k, 4000 + r + k), r, k).astype(np.float64) for r in rows]
    xs = xp.fill_normal(T * k, 291 + T, 1.0).reshape(T, k)
    got, kd = xp.gemm_piece(ws, xs)
    assert kd == kind
    for y, w in zip(got, wd):
        err = rel_l2(y, xs.astype(np.float64) @ w.T)
        print("piece gemm", t, rows, k, T, "error %.2e" % err)
        assert err < bound
    base = [xp.fill_normal(T * r, 29 + i, 1.0).reshape(T, r) for i, r in enumerate(rows)]
    for y, y0, b in zip(xp.gemm_piece(ws, xs, add_to=base)[0], got, base):
        assert np.array_equal(y, b + y0)
    nw = 1 + 0.1 * xp.fill_normal(k, 7, 1.0)
    x64 = xs.astype(np.float64)
    xn = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-6) * nw.astype(np.float64)
    for y, w in zip(xp.gemm_piece(ws, xs, norm_w=nw)[0], wd):
        err = rel_l2(y, xn @ w.T)
        print("  normed error %.2e" % err)
        assert err < bound
    for w in ws:
        w.free()


@pytest.mark.parametrize("t", [xp.Q4_K, xp.Q6_K])
def test_gemm_unaligned_input(t):
    """x at 4 bytes past a 16-byte boundary: 64 tokens go in launches of 32 on
    the kernel whose loads allow it, with that kernel's bits."""
    rows, k, T = 300, 512, 64
    w = xp.DevWeight(t, _weights(t, rows, k, 17), rows, k)
    xs = xp.fill_normal(T * k, 18, 1.0).reshape(T, k)
    want = np.concatenate([xp.gemm(w, xs[:32]), xp.gemm(w, xs[32:])])
    dx, dy = xp.Dev(np.concatenate([np.zeros(1, np.float32), xs.reshape(-1)])), xp.Dev(nbytes=T * rows * 4)
    err = C.create_string_buffer(512)
    assert xp.lib().xjh_gemm(t, w.ptr, rows, k, dx.ptr + 4, T, dy.ptr, 0, err, 512) == 0, err.value
    assert np.array_equal(dy.get(np.float32, (T, rows)).view(np.uint32), want.view(np.uint32))
    w.free()
