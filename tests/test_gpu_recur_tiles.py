"""The rows recurrence (k_gdn_recur_rows) at the edges of its 16-token tiles:
chunks that end one token before, at and after a tile boundary, shorter than
the staging ring of three tiles and longer, in both input forms (separate
q, k, v rows with fp32 beta; one [T, 6144] conv buffer with bf16 beta), bit
for bit against the oracle's token-by-token recurrence."""
import numpy as np
import pytest

import esdecode as E
import oracle as O
from helpers import assert_bits_equal, bf16, f32, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 95, 113])
def test_recur_rows_at_tile_edges(m):
    print(f"case recur tiles m={m}", flush=True)
    r = rng(900 + m)
    qk = r.normal(0, 1, (2, m, 16, 128))
    qk /= np.linalg.norm(qk, axis=-1, keepdims=True)
    q = bf16(qk[0] * 0.0078125).reshape(m, 2048)
    k = bf16(qk[1] * 128 ** -0.5).reshape(m, 2048)
    v = bf16(r.normal(0, 1, (m, 2048)))
    conv = np.concatenate([q, k, v], axis=1)
    g = np.exp(-r.uniform(0.01, 1.5, (m, 16))).astype(np.float32)
    beta = bf16(1 / (1 + np.exp(-r.normal(0, 1, (m, 16)))))
    state0 = r.normal(0, 0.1, (16, 128, 128)).astype(np.float32)
    want_state, want = state0.copy(), np.empty((m, 2048), np.uint16)
    for t in range(m):
        want[t] = O.gdn_recur(conv[t], g[t], beta[t], want_state)
    dg = E.DeviceBuffer.from_numpy(g)
    rows = [E.DeviceBuffer.from_numpy(a) for a in (q, k, v, f32(beta))]
    hist = [E.DeviceBuffer.from_numpy(a) for a in (conv, beta)]
    for form in ("rows", "conv"):
        ds, dy = E.DeviceBuffer.from_numpy(state0), E.DeviceBuffer(m * 2048 * 2)
        if form == "rows":
            E.check(E.lib().es_gdn_recur_rows(rows[0].ptr, rows[1].ptr, rows[2].ptr, dg.ptr, rows[3].ptr, m, ds.ptr,
                                              dy.ptr, None))
        else:
            E.check(E.lib().es_gdn_recur(hist[0].ptr, dg.ptr, hist[1].ptr, m, ds.ptr, dy.ptr, None))
        E.synchronize()
        assert_bits_equal(dy.numpy(np.uint16).reshape(m, 2048), want, what=f"{form} y")
        assert_bits_equal(ds.numpy(np.float32).reshape(16, 128, 128), want_state, what=f"{form} state")
