"""k_q4_gemm's tile heights (32, 64, 128 rows, chosen by the number of blocks),
its two weight fetches (whole 128-byte lines when K is a multiple of 256 and
the scales are 4-byte aligned, word by word otherwise) and its two stores
(16 bytes when every output is aligned and a multiple of 8 wide), and the
256 x 256 kernel: every output is one MFMA chain over K, so a row's bits depend
on neither the kernel nor the row count, and agree with the oracle's sums to
within one bf16 ulp on at most 1% of the outputs (fp32 order only)."""
import numpy as np
import pytest

import esdecode as E
import oracle as O
from helpers import assert_bf16_close, bf16, random_q4, rng

pytestmark = pytest.mark.gpu


def gemm(W, x, n, residual=None, shift=0):
    """es_q4_gemm of x [m, K]; shift: bf16 elements y and the residual are off 16-byte alignment."""
    m = x.shape[0]
    dx, dy = E.DeviceBuffer.from_numpy(x), E.DeviceBuffer((m * n + 8) * 2)
    dr = None
    if residual is not None:
        dr = E.DeviceBuffer.from_numpy(np.concatenate([np.zeros(shift, np.uint16), residual.ravel()]))
    E.check(E.lib().es_q4_gemm(W, dx.ptr, m, dr.ptr + 2 * shift if dr else None, dy.ptr + 2 * shift, None))
    E.synchronize()
    return dy.numpy(np.uint16)[shift:shift + m * n].reshape(m, n)


# rows that take 32-, 64- and 128-row tiles at N = 4096 (32 column blocks): up
# to 256, 512 and more; K with 1, 2, 3 and 5 steps past and without whole
# groups of four; one K in whole groups
@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 1024])
def test_rows_do_not_depend_on_the_tile_height(k):
    r = rng(8000 + k)
    n = 4096
    codes, scales, biases = random_q4(r, n, k)
    W = E.DeviceQ4(codes, scales, biases)
    x = bf16(r.normal(0, 1, (1061, k)))
    full = gemm(W.struct, x, n)
    for lo, hi in ((0, 1), (5, 36), (7, 264), (100, 133), (3, 388), (500, 1012), (0, 513)):
        print(f"case tile height k={k} rows {lo}..{hi}", flush=True)
        assert np.array_equal(gemm(W.struct, x[lo:hi], n), full[lo:hi]), (lo, hi)
    assert_bf16_close(full[:70], O.q4_gemm(codes, scales, biases, x[:70]), what=f"k={k} rows 0..69")
    assert_bf16_close(full[-9:], O.q4_gemm(codes, scales, biases, x[-9:]), what=f"k={k} last rows")


@pytest.mark.parametrize("n", [1, 7, 31, 33, 129, 1004])
@pytest.mark.parametrize("m", [1, 33, 300])
def test_ragged_columns_with_and_without_residual(m, n):
    print(f"case ragged m={m} n={n}", flush=True)
    r = rng(8100 + m + n)
    k = 512
    codes, scales, biases = random_q4(r, n, k)
    W = E.DeviceQ4(codes, scales, biases)
    x, res = bf16(r.normal(0, 1, (m, k))), bf16(r.normal(0, 1, (m, n)))
    plain = gemm(W.struct, x, n)
    assert_bf16_close(plain, O.q4_gemm(codes, scales, biases, x), what="plain")
    want = bf16(O.bf16_to_f32(res) + O.bf16_to_f32(plain))  # the residual add of the GEMM's own bits
    assert np.array_equal(gemm(W.struct, x, n, residual=res), want)


@pytest.mark.parametrize("shift", [1, 4])
def test_unaligned_outputs_and_scales(shift):
    """y and the residual `shift` elements off 16 bytes take the element
    stores; scales and biases two bytes off take the word-by-word fetch."""
    print(f"case unaligned shift={shift}", flush=True)
    r = rng(8200 + shift)
    m, n, k = 150, 264, 1024
    codes, scales, biases = random_q4(r, n, k)
    W = E.DeviceQ4(codes, scales, biases)
    x, res = bf16(r.normal(0, 1, (m, k))), bf16(r.normal(0, 1, (m, n)))
    want, want_res = gemm(W.struct, x, n), gemm(W.struct, x, n, residual=res)
    assert np.array_equal(gemm(W.struct, x, n, shift=shift), want)
    assert np.array_equal(gemm(W.struct, x, n, residual=res, shift=shift), want_res)
    off = [E.DeviceBuffer.from_numpy(np.concatenate([np.zeros(1, np.uint16), a.ravel()])) for a in (scales, biases)]
    w2 = E.Q4(W.codes.ptr, off[0].ptr + 2, off[1].ptr + 2, n, k)
    assert np.array_equal(gemm(w2, x, n), want)


# tiles of 32 rows; of 128; of 64 rows, in whole groups of steps and not; nine
# and ten row tiles of 128, so a remainder after the eight dealt to the XCDs
@pytest.mark.parametrize("m,n,k", [(1, 8, 320), (33, 24, 320), (130, 1000, 320), (300, 3584, 320), (700, 3584, 320),
                                   (203, 3584, 320), (203, 3584, 1024), (1061, 3584, 320), (1061, 3584, 1024),
                                   (1153, 1000, 1024)])
def test_swiglu_tiles(m, n, k):
    """Gate and up interleaved in a wave's 32 weight rows: two GEMMs and
    es_swiglu_rows give the same bits, at each tile height and at widths that
    are not whole blocks of 64."""
    print(f"case swiglu tiles m={m} n={n} k={k}", flush=True)
    r = rng(8300 + m + n)
    G, U = E.DeviceQ4(*random_q4(r, n, k)), E.DeviceQ4(*random_q4(r, n, k))
    x = bf16(r.normal(0, 1, (m, k)))
    dx = E.DeviceBuffer.from_numpy(x)
    dg, du = (E.DeviceBuffer.from_numpy(gemm(w.struct, x, n)) for w in (G, U))
    da, df = E.DeviceBuffer(m * n * 2), E.DeviceBuffer(m * n * 2)
    E.check(E.lib().es_swiglu_rows(dg.ptr, du.ptr, m * n, da.ptr, None))
    E.check(E.lib().es_q4_gemm_swiglu(G.struct, U.struct, dx.ptr, m, df.ptr, None))
    E.synchronize()
    assert np.array_equal(da.numpy(np.uint16), df.numpy(np.uint16))


@pytest.mark.parametrize("m,n", [(3600, 4096), (3584, 4090)])
def test_wide_kernel_gives_the_same_rows(m, n):
    """K = 2048 in 240 or 224 tiles of 256 x 256 takes the wide kernel; slices of its
    rows as smaller GEMMs do not."""
    print(f"case wide m={m} n={n}", flush=True)
    r = rng(8400 + n)
    k = 2048
    codes, scales, biases = random_q4(r, n, k)
    W = E.DeviceQ4(codes, scales, biases)
    x = bf16(r.normal(0, 1, (m, k)))
    full = gemm(W.struct, x, n)
    for lo, hi in ((0, 300), (1000, 1033), (m - 700, m)):
        assert np.array_equal(gemm(W.struct, x[lo:hi], n), full[lo:hi]), (lo, hi)
