"""GPU parity of the prefill GEMMs on narrow tiles (pf_narrow.hip) against the
oracle, where their tiles, K loops and operands can go wrong.

Eight experts, so every expert gets every token: T = 1 .. 65 covers a tile's
first and last row and one row past it (16 rows in split mode, 32 in fp16
mode; fp16 mode leaves the narrow tiles past T = 28 with Q6_K and 36 with Q4_K
gate matrices), hidden 256 / 768 / 2048 one, an odd and an even number of super-blocks,
inter 256 / 512 one and two in the down product.  Q6_K scales take the whole
int8 range: sc (q - 32) then exceeds 2048, where split mode's second weight
operand holds what fp16 rounds off.  Routed and shared types are opposite, so
each call runs both weight types.

Bars: fp16 operands 2e-3 of max|y| as every fp16 prefill test; split mode
1e-5 -- activations of 22 bits (2^-22 per product, random in sign) against
f32 sums of up to 2048 terms on both sides, about 1e-6 each, through two
products."""
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


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 65])
@pytest.mark.parametrize("prec,tol", [(R.PREC_F16, 2e-3), (R.PREC_SPLIT, 1e-5)], ids=["f16", "split"])
def test_narrow_tiles(table, T, prec, tol):
    H = table.desc.hidden
    X = np.stack([R.synth_normal(9, R.synth_stream(0, t, 5), H) for t in range(T)])
    X[T // 2] *= 2.0 ** 10                        # a row's scale is its own
    Y, lg, ids, w, counts = prefill(table, X, precision=prec)
    assert counts.tolist() == [T] * 8
    rc, Y_ref, ids_ref, _, _ = table.oracle_layer(0).prefill(X, logits_in=lg)
    assert rc == 0 and np.array_equal(ids_ref, ids)
    err = max(rel_err(Y[t], Y_ref[t]) for t in range(T))
    log(f"T {T} precision {prec}: max|d|/max|y| over rows = {err:.2e}")
    assert err <= tol
