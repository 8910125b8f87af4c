"""GPU parity of prefill on Q6_K matrices whose scales take the whole int8 range,
against the oracle: sc (q - 32) and the fp16 constants around it must not
overflow.  Routed and shared types are opposite, so each call runs both weight
types.  The bar is the fp16 operands' 2e-3 of max|y|, as in every fp16 prefill
test."""
import numpy as np
import pytest

import roaster_amd as R
from gpu_util import SynthTable, log, prefill, rel_err

pytestmark = pytest.mark.gpu


def wide_scales(mat, rng):
    """Q6_K bytes with scales over all of int8, d reduced to keep the weights' size."""
    b = mat.reshape(-1, R.Q6K_BYTES).copy()
    b[:, 192:208] = rng.integers(0, 256, (len(b), 16), dtype=np.uint8)
    d = b[:, 208:210].copy().view(np.float16)
    b[:, 208:210] = (d / np.float16(4)).view(np.uint8)
    return b.reshape(-1)


@pytest.fixture(scope="module", params=[(256, 256, 0, 1), (768, 512, 1, 0), (2048, 512, 0, 1), (2048, 512, 1, 0)],
                ids=lambda p: "H%d-I%d-gu%d-dn%d" % p)
def table(request):
    H, I, gu, dn = request.param
    q6, sq6 = (gu, gu, dn), (1 - gu, 1 - gu, 1 - dn)
    t = SynthTable(11, n_experts=8, hidden=H, inter=I, q6=q6, sh_q6=sq6)
    rng = np.random.default_rng(5)
    for e in range(9):
        types = sq6 if e == 8 else q6
        m = [wide_scales(w, rng) if q else w for w, q in zip(t.expert(0, e), types)]
        t._experts[(0, e)] = tuple(m)
        R.check(R.lib().roaster_table_set_expert(t.t, 0, e, *(w.ctypes.data for w in m)), "set_expert")
    yield t
    t.destroy()


@pytest.mark.parametrize("T", [1, 33])
def test_wide_scales(table, T):
    H = table.desc.hidden
    X = np.stack([R.synth_normal(9, R.synth_stream(0, t, 5), H) for t in range(T)])
    Y, lg, ids, w, counts = prefill(table, X)
    assert counts.tolist() == [T] * 8
    rc, Y_ref, ids_ref, _, _ = table.oracle_layer(0).prefill(X, logits_in=lg)
    assert rc == 0 and np.array_equal(ids_ref, ids)
    err = rel_err(Y, Y_ref)
    log(f"T {T}: max|d|/max|y| = {err:.2e}")
    assert err <= 2e-3
