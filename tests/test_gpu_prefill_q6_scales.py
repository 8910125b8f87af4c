"""GPU parity of prefill on Q6_K matrices whose scales take the whole int8 range,
against the oracle: sc (q - 32) and the fp16 constants around it must not
overflow.  Routed and shared types are opposite, so each call runs both weight
types; the gate/up GEMM is the narrow one at T = 1, the wide one from T = 29 with
routed Q6_K gate matrices and from 37 with Q4_K ones (shared Q6_K).  The bar is
the fp16 operands' 2e-3 of max|y|, as in every fp16 prefill test."""
import numpy as np
import pytest

import roaster_amd as R
from gpu_util import WIDE_SCALE_TABLES, log, prefill, rel_err, wide_scale_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=WIDE_SCALE_TABLES, ids=lambda p: "H%d-I%d-gu%d-dn%d" % p)
def table(request):
    t = wide_scale_table(*request.param)
    yield t
    t.destroy()


@pytest.mark.parametrize("T", [1, 33, 37])
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
