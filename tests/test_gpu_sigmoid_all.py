"""sigmoid_bf over every bf16 value (NaN, infinities and denormals among them)
through the output gate (o = 1, so the result is the sigmoid itself) and
through SwiGLU (up = 1), bit for bit against the oracle."""
import numpy as np
import pytest

import esdecode as E
import oracle as O
from helpers import assert_bits_equal

pytestmark = pytest.mark.gpu


def test_every_bf16_value():
    x = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    one = np.full(65536, 0x3F80, np.uint16)
    qp = np.zeros((32, 8, 512), np.uint16)
    qp[:, :, 256:] = x.reshape(32, 8, 256)
    d = [E.DeviceBuffer.from_numpy(a) for a in (one, qp, x)]
    gated, act = E.DeviceBuffer(65536 * 2), E.DeviceBuffer(65536 * 2)
    E.check(E.lib().es_attn_gate_rows(d[0].ptr, d[1].ptr, 32, gated.ptr, None))
    E.check(E.lib().es_swiglu_rows(d[2].ptr, d[0].ptr, 65536, act.ptr, None))
    E.synchronize()
    got = gated.numpy(np.uint16).reshape(32, 2048)
    for t in range(32):
        assert_bits_equal(got[t], O.attn_gate(one[:2048], qp[t].ravel()), what=f"sigmoid of 0x{2048 * t:04x}..")
    want, got = O.swiglu(x, one), act.numpy(np.uint16)
    nan = ((want & 0x7FFF) > 0x7F80) & ((got & 0x7FFF) > 0x7F80)  # a NaN's payload is not specified
    assert_bits_equal(np.where(nan, 0, got), np.where(nan, 0, want), what="silu")


@pytest.mark.parametrize("m", [3, 191, 192, 193])
@pytest.mark.parametrize("off", [0, 1])
def test_gate_rows_aligned_and_not(off, m):
    """Pointers `off` bf16 elements past 16-byte alignment take the element
    form, aligned ones the 8-element form from 192 rows: the same bits, in place
    too."""
    r = np.random.default_rng(7)
    o = O.f32_to_bf16(r.normal(0, 1, m * 2048).astype(np.float32))
    qp = O.f32_to_bf16(r.normal(0, 2, m * 4096).astype(np.float32))
    pad = np.zeros(off, np.uint16)
    do, dq = (E.DeviceBuffer.from_numpy(np.concatenate([pad, a])) for a in (o, qp))
    E.check(E.lib().es_attn_gate_rows(do.ptr + 2 * off, dq.ptr + 2 * off, m, do.ptr + 2 * off, None))
    E.synchronize()
    got = do.numpy(np.uint16)[off:].reshape(m, 2048)
    for t in range(m):
        assert_bits_equal(got[t], O.attn_gate(o[2048 * t:2048 * t + 2048], qp[4096 * t:4096 * t + 4096]), what=f"row {t}")
