"""The matvec of several token rows at four weight rows a pass (taken once its
waves fill the chip): widths that are not whole passes, both sides of the line
where the rule switches, K of half-wave and whole-wave rows, with and without
the residual, bit for bit the oracle's M = 1 matvec per row."""
import numpy as np
import pytest

import esdecode as E
import oracle as O
from helpers import assert_bits_equal, bf16, random_q4, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,rows", [(1024, 3584, 3), (1024, 3584, 4), (1021, 2048, 5), (1026, 3584, 32),
                                      (3584, 1024, 4), (3584, 1024, 5), (3589, 1024, 7), (516, 1024, 33),
                                      (1, 2048, 4100), (1, 2048, 6145), (1021, 2048, 7), (516, 1024, 43)])
def test_token_rows_by_four_weight_rows(n, k, rows):
    print(f"case matvec rows P n={n} k={k} rows={rows}", flush=True)
    r = rng(n + k + rows)
    codes, scales, biases = random_q4(r, n, k)
    x, res = bf16(r.normal(0, 1, (rows, k))), bf16(r.normal(0, 1, (rows, n)))
    W = E.DeviceQ4(codes, scales, biases)
    dx, dy, dh = E.DeviceBuffer.from_numpy(x), E.DeviceBuffer(rows * n * 2), E.DeviceBuffer.from_numpy(res)
    E.check(E.lib().es_q4_matvec_rows(W.struct, dx.ptr, rows, None, dy.ptr, None))
    E.check(E.lib().es_q4_matvec_rows(W.struct, dx.ptr, rows, dh.ptr, dh.ptr, None))
    E.synchronize()
    assert_bits_equal(dy.numpy(np.uint16), O.q4_matvec_rows(codes, scales, biases, x), what="rows")
    assert_bits_equal(dh.numpy(np.uint16), O.q4_matvec_rows(codes, scales, biases, x, res), what="rows + residual")
