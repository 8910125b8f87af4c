"""kernel_ffn_fused over the forms its two down paths take, against the oracle:
one to nine experts, down matrices of one type (the path that issues every row
load at once, inter <= 512) and of two, inter past that path's, hidden 256; and
an earlier call's routing error, which the next call reports by returning 0,
once."""
import ctypes as C

import numpy as np
import pytest

import roaster_amd as R
from oracle import oracle as O
from gpu_util import Dev, SynthTable, alloc_w, log, rel_err

pytestmark = pytest.mark.gpu


def call(x, experts, types, I, H):
    out = np.full((len(experts), H), np.nan, np.float32)
    fx = (R.KernelFfnExpert * len(experts))()
    for f, (g, u, d), (tg, tu, td), o in zip(fx, experts, types, out):
        f.gate, f.up, f.down = alloc_w(g), alloc_w(u), alloc_w(d)
        f.gate_q6, f.up_q6, f.down_q6, f.out = tg, tu, td, o.ctypes.data
    return R.lib().kernel_ffn_fused(fx, len(experts), x.ctypes.data, I, H), out, fx


@pytest.mark.parametrize("n,H,I,types", [(1, 2048, 512, [(0, 0, 1)]), (5, 2048, 512, [(0, 0, 0)]),
                                         (9, 2048, 512, [(0, 0, 1), (1, 1, 0)]), (8, 256, 256, [(1, 0, 1)]),
                                         (9, 1024, 1024, [(0, 0, 1)])])
def test_forms(n, H, I, types):
    types = [types[k % len(types)] for k in range(n)]
    x = R.synth_normal(61, R.synth_stream(0, 0, 5), H)
    experts = [R.host_expert(61, 0, k, R.table_desc(1, 256, H, I, t, t)) for k, t in enumerate(types)]
    rc, out, fx = call(x, experts, types, I, H)
    assert rc == 1
    for k, (e, t) in enumerate(zip(experts, types)):
        ref = np.empty(H, np.float32)
        ex = O.OrcExpert(*(m.ctypes.data for m in e), *t)
        O.orc().orc_expert_decode(C.byref(ex), x.ctypes.data, I, H, ref.ctypes.data)
        err = rel_err(out[k], ref)
        assert err <= 2e-5, (k, err)


def test_reports_an_earlier_error_once():
    L = R.lib()
    H, I = 2048, 512
    t = SynthTable(62, n_experts=32)
    try:
        x = R.synth_normal(62, R.synth_stream(0, 0, 5), H)
        lg = np.full((1, 32), -np.inf, np.float32)
        lg[0, :3] = 1.0
        dx, dy, dl = Dev(x), Dev(nbytes=H * 4, shape=(1, H)), Dev(lg)
        io = R.RoasterDecodeIO(dl.p, None, None, None)
        R.check(L.roaster_moe_decode(t.t, 0, dx.p, 1, dy.p, C.byref(io)))
        e = t.expert(0, 0)
        rc, _, fx = call(x, [e], [(0, 0, 1)], I, H)
        assert rc == 0 and "finite logits" in R.last_error()
        assert L.kernel_ffn_fused(fx, 1, x.ctypes.data, I, H) == 1
        R.check(L.roaster_sync(), "sync")
    finally:
        t.destroy()
