"""GPU parity of the prefill router (pf_router_mfma_kernel) against float64,
where its blocks can go wrong: experts of 32 and of 128 (one, one short, one
past), tokens of 32 and, from 1024 tokens, of 64, K slices of one chunk, an odd
number and eight.  The router is set twice, by the synthetic fill and by
roaster_table_set_router, since each lays out the kernel's operand copy.

Bar: a logit is a sum of H products in eight slices; with u = 2^-24 each
product and each addition of a slice (H / 8) and of the slices (8) rounds once,
so |error| <= (H / 8 + 9) u sum |x w|."""
import numpy as np
import pytest

import roaster_amd as R
from gpu_util import Dev, SynthTable, prefill

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[(8, 256), (33, 768), (127, 2048), (256, 2048)], ids=lambda p: "E%d-H%d" % p)
def table(request):
    E, H = request.param
    t = SynthTable(3, n_experts=E, hidden=H, inter=256)
    yield t
    t.destroy()


def check(table, router, T):
    H = table.desc.hidden
    X = np.random.default_rng(T).standard_normal((T, H)).astype(np.float32)
    lg = prefill(table, X)[1]
    ref = X.astype(np.float64) @ router.T.astype(np.float64)
    bar = (H / 8 + 9) * 2.0 ** -24 * (np.abs(X).astype(np.float64) @ np.abs(router.T).astype(np.float64))
    assert np.all(np.abs(lg - ref) <= bar)


@pytest.mark.parametrize("T", [1, 31, 32, 33, 1023, 1024, 1025])
def test_router_logits(table, T):
    check(table, table.router(0)[0], T)


def test_router_replaced(table):
    E, H = table.desc.n_experts, table.desc.hidden
    router = np.random.default_rng(E).standard_normal((E, H)).astype(np.float32)
    old, gate_inp = (np.ascontiguousarray(a) for a in table.router(0))
    R.check(R.lib().roaster_table_set_router(table.t, 0, router.ctypes.data, gate_inp.ctypes.data), "set_router")
    check(table, router, 40)
    R.check(R.lib().roaster_table_set_router(table.t, 0, old.ctypes.data, gate_inp.ctypes.data), "set_router")
    check(table, old, 40)


@pytest.mark.parametrize("E", [256, 257])
def test_operand_copy_only_where_prefill_reads_it(E):
    """A table of more than 256 experts, which prefill refuses, carries no operand
    copy of the router; setting its router works, prefill refuses as before."""
    t = SynthTable(4, n_experts=E, hidden=256, inter=256, q6=(0, 0, 1), sh_q6=(0, 0, 1))
    try:
        mats = 256 * (2 * R.Q4K_BYTES + R.Q6K_BYTES) + 8 * 1024 * (2 * 5 + 7)      # GGML and 32-row tile layouts
        copies = 2 if E <= 256 else 1
        assert R.lib().roaster_table_bytes(t.t) == (E + 1) * mats + 4 * 256 * (E * copies + 1)
        router, gate_inp = (np.ascontiguousarray(a) for a in t.router(0))
        R.check(R.lib().roaster_table_set_router(t.t, 0, router.ctypes.data, gate_inp.ctypes.data), "set_router")
        x, y = Dev(np.zeros((1, 256), np.float32)), Dev(nbytes=1024)
        assert R.lib().roaster_moe_prefill(t.t, 0, x.p, 1, y.p, None) == (0 if E <= 256 else R.EINVAL)
        R.check(R.lib().roaster_sync(), "sync")
    finally:
        t.destroy()
