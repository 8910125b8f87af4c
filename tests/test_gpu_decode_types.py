"""One-launch decode stacks on every matrix-type mix they are compiled for:
gate/up Q4_K or Q6_K throughout, down Q4_K or Q6_K by layer, routed and shared
down types apart, against the three-kernel path (roaster_decode_fused_layer(0))
and the oracle.

The batched kernels (2, 4 and 8 token slots, some unused) and the general
one-token kernel (mode 2) keep the three-kernel path's arithmetic: equal bit
for bit.  The folded-router kernel (one token, 256 experts, hidden 2048, inter
512) sums its logits and 1/rms in another order: ids equal, the rest within
1e-5, the bound of its Q4_K / Q6_K form.  The oracle bar is the decode tests'
1e-4."""
import ctypes as C

import numpy as np
import pytest

import roaster_amd as R
from gpu_util import SynthTable, log, rel_err
from test_gpu_decode import oracle_stack
from test_gpu_decode_layer1 import _in_mode, _near, _same, _stack

pytestmark = pytest.mark.gpu

# (routed gate/up, down, shared gate/up, down) by layer
MIXES = {"q4": [(0, 1, 0, 1), (0, 0, 0, 0), (0, 0, 0, 1), (0, 1, 0, 0)],
         "q4_q4": [(0, 0, 0, 0)] * 3,
         "q6": [(1, 1, 1, 1), (1, 0, 1, 0), (1, 1, 1, 0)]}


class LayerTable(SynthTable):
    """A SynthTable with the types of `mix` layer by layer."""

    def __init__(self, seed, mix, **kw):
        self.mix = mix
        self.seed = seed
        self.desc = R.table_desc(len(mix), **kw)
        types = (C.c_int * (6 * len(mix)))(*sum(([g, g, d, sg, sg, sd] for g, d, sg, sd in mix), []))
        self.t = R.lib().roaster_table_create_layers(C.byref(self.desc), types)
        assert self.t, R.last_error()
        R.check(R.lib().roaster_table_synth(self.t, seed, None), "table_synth")
        self._experts, self._routers = {}, {}

    def layer_desc(self, layer):
        g, d, sg, sd = self.mix[layer]
        return R.table_desc(1, self.desc.n_experts, self.desc.hidden, self.desc.inter, (g, g, d), (sg, sg, sd))

    def expert(self, layer, e):
        k = (layer, e)
        if k not in self._experts:
            self._experts[k] = R.host_expert(self.seed, layer, e, self.layer_desc(layer))
        return self._experts[k]

    def oracle_layer(self, layer, experts_needed=None):
        old = self.desc
        self.desc = self.layer_desc(layer)
        try:
            return super().oracle_layer(layer, experts_needed)
        finally:
            self.desc = old


@pytest.mark.parametrize("B", [1, 2, 3, 8])
@pytest.mark.parametrize("shape", [(256, 2048), (64, 768)], ids=lambda s: "E%d-H%d" % s)
@pytest.mark.parametrize("mix", sorted(MIXES))
def test_types(mix, shape, B):
    E, H = shape
    NL = len(MIXES[mix])
    t = LayerTable(51, MIXES[mix], n_experts=E, hidden=H, inter=512)
    try:
        name = R.lib().roaster_decode_stack_kernel(t.t, B, 0, NL).decode()
        assert name.endswith("_q6_kernel" if mix == "q6" else "_q4_kernel") or (B == 1 and E != 256), name
        h0 = np.stack([R.synth_normal(51, R.synth_stream(0, b, 5), H) for b in range(B)])
        nw = np.stack([1.0 + 0.25 * R.synth_normal(52, R.synth_stream(l, 0, 6), H) for l in range(NL)]).astype(np.float32)
        a = _stack(t, h0, NL, nw)
        three = _in_mode(0, lambda: _stack(t, h0, NL, nw))
        if B == 1:
            _same(_in_mode(2, lambda: _stack(t, h0, NL, nw)), three)
        if name.startswith("dec_stack1r"):
            _near(a, three, ref=h0)
        else:
            _same(a, three)
        h_ref, ids_ref = oracle_stack(t, h0, NL, norm_w=nw)
        assert np.array_equal(a[1], ids_ref)
        err = rel_err(a[0] - h0, h_ref - h0)
        log(f"{mix} E={E} H={H} B={B} {name}: max|d|/max|ffn| = {err:.2e}")
        assert err <= 1e-4
    finally:
        t.destroy()


@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("shape", [(256, 2048), (64, 768), (32, 512)], ids=lambda s: "E%d-H%d" % s)
@pytest.mark.parametrize("B", [2, 3, 8])
def test_inter_256_in_one_launch(shape, mix, B):
    """Inter 256 (one row per wave, one super-block per down row): bit for bit
    the three kernels' results, ids equal to the oracle's."""
    E, H = shape
    NL = len(MIXES[mix])
    t = LayerTable(61, MIXES[mix], n_experts=E, hidden=H, inter=256)
    try:
        name = R.lib().roaster_decode_stack_kernel(t.t, B, 0, NL).decode()
        assert name.endswith("_i256_q6_kernel" if mix == "q6" else "_i256_q4_kernel"), name
        h0 = np.stack([R.synth_normal(61, R.synth_stream(0, b, 5), H) for b in range(B)])
        nw = np.stack([1.0 + 0.25 * R.synth_normal(62, R.synth_stream(l, 0, 6), H) for l in range(NL)]).astype(np.float32)
        a = _stack(t, h0, NL, nw)
        _same(a, _in_mode(0, lambda: _stack(t, h0, NL, nw)))
        h_ref, ids_ref = oracle_stack(t, h0, NL, norm_w=nw)
        assert np.array_equal(a[1], ids_ref)
        assert rel_err(a[0] - h0, h_ref - h0) <= 1e-4
    finally:
        t.destroy()
