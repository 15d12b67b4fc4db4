"""k_attn_prefill's two key halves (keys 0-15 and 16-31 of every block of 32,
one wave each, combined at the end): rows with no key in the upper half, one
key in it, and exactly whole halves, against the fp64 softmax with the bound
of the whole-kernel test (bf16 probabilities: 2^-8 of the largest V plus one
bf16 ulp); and a row's bits do not depend on the call's first row or count."""
import numpy as np
import pytest

import esdecode as E
from helpers import bf16, f32, rng
from test_gpu_prefill_rows import attention_f64

pytestmark = pytest.mark.gpu


def attend(query, kc, vc, pos0, m):
    d = [E.DeviceBuffer.from_numpy(np.ascontiguousarray(a)) for a in (query, kc, vc)]
    do = E.DeviceBuffer(m * 2048 * 2)
    E.check(E.lib().es_attn_prefill(d[0].ptr, d[1].ptr, d[2].ptr, pos0, m, kc.shape[1], do.ptr, None))
    E.synchronize()
    return do.numpy(np.uint16).reshape(m, 2048)


@pytest.mark.parametrize("pos0,m", [(0, 16), (0, 17), (15, 1), (16, 1), (31, 2), (46, 4), (63, 33), (95, 1), (200, 97)])
@pytest.mark.parametrize("spread", [1.0, 6.0])
def test_halves_against_fp64(pos0, m, spread):
    print(f"case attn halves pos0={pos0} m={m} spread={spread}", flush=True)
    r = rng(1300 + pos0 + m)
    n = pos0 + m
    query = bf16(r.normal(0, spread, (m, 2048)))
    kc, vc = bf16(r.normal(0, 1, (2, n, 256))), bf16(r.normal(0, 1, (2, n, 256)))
    got = f32(attend(query, kc, vc, pos0, m)).astype(np.float64).reshape(m, 8, 256)
    want = attention_f64(query, kc, vc, pos0, m)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(want), 1e-30))) - 7)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(f32(vc)).max() + ulp)


def test_rows_do_not_depend_on_the_call():
    r = rng(1400)
    pos0, m = 37, 150
    query = bf16(r.normal(0, 2, (m, 2048)))
    kc, vc = bf16(r.normal(0, 1, (2, pos0 + m, 256))), bf16(r.normal(0, 1, (2, pos0 + m, 256)))
    full = attend(query, kc, vc, pos0, m)
    for lo, hi in ((0, 1), (1, 34), (17, 49), (90, 150)):
        print(f"case attn rows {lo}..{hi}", flush=True)
        assert np.array_equal(attend(query[lo:hi], kc, vc, pos0 + lo, hi - lo), full[lo:hi]), (lo, hi)


@pytest.mark.parametrize("m", [1, 16, 17, 33])
def test_output_rows_at_eight_byte_alignment(m):
    """o four elements off 16-byte alignment: the same bits, nothing past the rows."""
    print(f"case attn o alignment m={m}", flush=True)
    r = rng(1500 + m)
    query, kc, vc = (bf16(r.normal(0, 1, s)) for s in ((m, 2048), (2, m, 256), (2, m, 256)))
    want = attend(query, kc, vc, 0, m)
    d = [E.DeviceBuffer.from_numpy(a) for a in (query, kc, vc)]
    do = E.DeviceBuffer.from_numpy(np.full(m * 2048 + 8, 0xA5A5, np.uint16))
    E.check(E.lib().es_attn_prefill(d[0].ptr, d[1].ptr, d[2].ptr, 0, m, m, do.ptr + 8, None))
    E.synchronize()
    got = do.numpy(np.uint16)
    assert np.array_equal(got[4:-4].reshape(m, 2048), want)
    assert np.all(got[:4] == 0xA5A5) and np.all(got[-4:] == 0xA5A5)
