"""Measured workloads of the MoE-FFN path, through its public C entry points.

`listed()` names the workloads, `draw()` gives more of the same ranges,
`prepare()` makes what a program holds before the call (an expert table or
weights in HBM, activations), `run()` is one call, `exact()` the same result
in 64-bit torch arithmetic from the same bytes.

Weight scales are those of a quantised model's files (matrix entries of about
0.02, so that gate and up products of normalised activations are of order 1);
activations are N(0, 1), norm weights near 1, routers N(0, 0.02^2).
"""
import ctypes as C
import math

import numpy as np
import torch

import roaster_amd as R

E, TOP = 256, 8
EPS = 1e-6
# d / dmin of Q4_K and d of Q6_K blocks: |w| of about 0.02
SPEC = dict(q4k_lo=5e-5, q4k_hi=2e-4, q6k_lo=3e-5, q6k_hi=9e-5, router_sigma=0.02, gate_inp_sigma=0.02)
Q4K, Q6K = 0, 1


def listed():
    return [
        # One token through one layer, the layer's neighbours being computed elsewhere: the smallest call.
        {"name": "decode_block", "kind": "block", "tokens": 1, "hidden": 2048, "inter": 512, "gate_up": Q4K, "down": Q6K},
        # A single user's next token: every layer's MoE block, Q4_K gate/up and Q6_K down.
        {"name": "decode_stack", "kind": "stack", "tokens": 1, "layers": 40, "hidden": 2048, "inter": 512, "mix": 0},
        # Eight sequences served together, the most one call takes.
        {"name": "decode_stack_batch8", "kind": "stack", "tokens": 8, "layers": 16, "hidden": 2048, "inter": 512, "mix": 0},
        # Three sequences on a file that keeps its down matrices in Q6_K in some layers and in Q4_K in the others.
        {"name": "decode_stack_mixed", "kind": "stack", "tokens": 3, "layers": 16, "hidden": 2048, "inter": 512, "mix": 1},
        # A short prompt.
        {"name": "prefill_45", "kind": "prefill", "tokens": 45, "hidden": 2048, "inter": 512, "gate_up": Q4K, "down": Q6K,
         "precision": 0, "skew": 0.0},
        # A prompt chunk whose tokens favour a few experts.
        {"name": "prefill_512_skewed", "kind": "prefill", "tokens": 512, "hidden": 2048, "inter": 512, "gate_up": Q4K,
         "down": Q6K, "precision": 0, "skew": 0.3},
        # A long prompt on experts that are Q6_K throughout.
        {"name": "prefill_2048_q6k", "kind": "prefill", "tokens": 2048, "hidden": 2048, "inter": 512, "gate_up": Q6K,
         "down": Q6K, "precision": 0, "skew": 0.0},
        # A prompt chunk of the reference's size in the arithmetic nearest f32.
        {"name": "prefill_256_split", "kind": "prefill", "tokens": 256, "hidden": 2048, "inter": 512, "gate_up": Q4K,
         "down": Q6K, "precision": 1, "skew": 0.0},
        # The attention output projection of one token.
        {"name": "projection", "kind": "dense", "tokens": 1, "rows": 2048, "cols": 4096, "q6": Q4K},
        # The LM head for one sequence, and for five served together.
        {"name": "lm_head", "kind": "dense", "tokens": 1, "rows": 248320, "cols": 2048, "q6": Q6K},
        {"name": "lm_head_batch5", "kind": "dense", "tokens": 5, "rows": 248320, "cols": 2048, "q6": Q6K},
        # One token's nine experts from host weight memory, as the kernels.h caller's decode loop makes the call.
        {"name": "ffn_host", "kind": "ffn", "experts": 9, "hidden": 2048, "inter": 512, "gate_up": Q4K, "down": Q6K},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng):
    """Mostly the model's hidden and expert width, else another the table takes."""
    return rng.choice([(2048, 512)] * 4 + [(1024, 512), (2048, 256), (1536, 512)])


def draw(rng):
    kind = rng.choice(["block", "stack", "stack", "prefill", "prefill", "prefill", "dense", "dense", "ffn"])
    H, I = _shape(rng)
    if kind == "block":
        return {"kind": kind, "tokens": rng.choice([1, 1, rng.randint(2, 8)]), "hidden": H, "inter": I,
                "gate_up": rng.choice([Q4K, Q4K, Q6K]), "down": rng.choice([Q4K, Q6K])}
    if kind == "stack":
        B = rng.choice([1, rng.randint(2, 8)])
        return {"kind": kind, "tokens": B, "layers": rng.randint(3, 40 if B == 1 else 16), "hidden": H, "inter": I,
                "mix": rng.randint(0, 1)}
    if kind == "prefill":
        split = rng.random() < 0.25
        return {"kind": kind, "tokens": _log_int(rng, 1, 700 if split else 2048), "hidden": H, "inter": I,
                "gate_up": rng.choice([Q4K, Q4K, Q6K]), "down": rng.choice([Q4K, Q6K, Q6K]), "precision": int(split),
                "skew": rng.choice([0.0, 0.0, round(rng.uniform(0.1, 0.4), 2)])}
    if kind == "dense":
        return {"kind": kind, "tokens": rng.choice([1, rng.randint(2, 8)]), "rows": _log_int(rng, 500, 248320),
                "cols": rng.choice([512, 1024, 2048, 2048, 2560, 4096]), "q6": rng.randint(0, 1)}
    return {"kind": kind, "experts": rng.choice([8, 9, rng.randint(1, 9)]), "hidden": H, "inter": I,
            "gate_up": rng.choice([Q4K, Q6K]), "down": rng.choice([Q4K, Q6K])}


# ---- sizes -------------------------------------------------------------------
def _mat(q6, rows, cols):
    return rows * (cols // 256) * (210 if q6 else 144)


def _layer_types(case, layer):
    """(gate/up, down) types of a layer.  A mixed file keeps Q6_K down matrices in its
    first and last eighth and in every third layer between, Q4_K in the others."""
    if case["kind"] != "stack":
        return case["gate_up"], case["down"]
    if not case["mix"]:
        return Q4K, Q6K
    n = case["layers"]
    more = layer < n // 8 or layer >= 7 * n // 8 or (layer - n // 8) % 3 == 2
    return Q4K, Q6K if more else Q4K


def _layers(case):
    return case.get("layers", 1)


def work(case):
    """Each weight the tokens need read once (the experts hit being those that uniform
    routing is expected to hit), activations read and written once."""
    k = case["kind"]
    if k == "dense":
        T, r, c = case["tokens"], case["rows"], case["cols"]
        return {"bytes": _mat(case["q6"], r, c) + 4 * T * (r + c), "flops": 2.0 * T * r * c}
    H, I = case["hidden"], case["inter"]
    if k == "ffn":
        n = case["experts"]
        return {"bytes": n * (2 * _mat(case["gate_up"], I, H) + _mat(case["down"], H, I)) + 4 * H * (n + 1),
                "flops": 6.0 * n * H * I}
    T = case["tokens"]
    hit = E * (1 - (1 - TOP / E) ** T) + 1
    total = 0.0
    for l in range(_layers(case)):
        gu, dn = _layer_types(case, l)
        total += hit * (2 * _mat(gu, I, H) + _mat(dn, H, I)) + 4 * H * (E + 1)
    if k == "stack":
        total += 4 * H * _layers(case)
    total += 8 * T * H
    return {"bytes": total, "flops": _layers(case) * T * (2.0 * (E + 1) * H + 9 * 6.0 * H * I)}


def tolerance(case):
    k = case["kind"]
    if k == "prefill":
        # fp16 operands and rows (5.6e-4 from exact), or bf16 hi + lo operands (7.3e-6)
        return {"rel": 2.5e-3, "max": 5e-2} if case["precision"] == 0 else {"rel": 4e-5, "max": 2e-3}
    if k == "stack":
        # 32-bit sums, carried through the layers (up to 2.5e-5 from exact)
        return {"rel": 1e-4, "max": 1e-2}
    if k == "dense":
        # 32-bit sums, with several tokens of operands kept to 22 bits (2.3e-6)
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 4e-6, "max": 2e-4}


# ---- state -------------------------------------------------------------------
class _Table:
    """An expert table in HBM, destroyed with its last reference."""

    def __init__(self, case, seed):
        L, n = R.lib(), _layers(case)
        self.desc = R.table_desc(n, E, case["hidden"], case["inter"])
        types = (C.c_int * (6 * n))()
        for l in range(n):
            gu, dn = _layer_types(case, l)
            types[6 * l:6 * l + 6] = [gu, gu, dn, gu, gu, dn]
        self.spec = R.RoasterSynthSpec(**SPEC)
        self.p = L.roaster_table_create_layers(C.byref(self.desc), types)
        if not self.p:
            raise RuntimeError(R.last_error())
        R.check(L.roaster_table_synth(self.p, seed, C.byref(self.spec)), "table_synth")

    def __del__(self):
        if getattr(self, "p", None):
            R.lib().roaster_table_destroy(self.p)


class _State:
    pass


def _normal(seed, what, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed * 16 + what)
    return torch.randn(*shape, device="cuda", generator=g)


def _skew_bias(case, seed):
    """Logit bias skew * ln p, p proportional to rank^-1.1 over a permutation of the experts."""
    if not case["skew"]:
        return None
    p = np.empty(E)
    p[np.random.default_rng(seed).permutation(E)] = np.arange(1, E + 1, dtype=np.float64) ** -1.1
    return torch.from_numpy((case["skew"] * np.log(p / p.sum())).astype(np.float32)).cuda()


def _dense_weights(case, seed):
    """[rows][cols / 256] blocks of random quants with the scales of a model's file."""
    n = case["rows"] * (case["cols"] // 256)
    g = torch.Generator(device="cuda").manual_seed(seed * 16 + 3)
    q6 = case["q6"]
    w = torch.randint(0, 256, (n, 210 if q6 else 144), dtype=torch.uint8, device="cuda", generator=g)
    lo, hi = (SPEC["q6k_lo"], SPEC["q6k_hi"]) if q6 else (SPEC["q4k_lo"], SPEC["q4k_hi"])
    d = (torch.rand(n, 1 if q6 else 2, device="cuda", generator=g) * (hi - lo) + lo).half().view(torch.uint8)
    if q6:
        w[:, 192:208] = ((w[:, 192:208] & 63).to(torch.int16) - 32).to(torch.int8).view(torch.uint8)
        w[:, 208:210] = d
    else:
        w[:, :4] = d
    return w


def _ffn_weights(case, seed):
    H, I = case["hidden"], case["inter"]
    d = R.table_desc(1, E, H, I, (case["gate_up"], case["gate_up"], case["down"]),
                     (case["gate_up"], case["gate_up"], case["down"]))
    return [R.host_expert(seed, 0, e, d, R.RoasterSynthSpec(**SPEC)) for e in range(case["experts"])]


def prepare(case, seed):
    s = _State()
    s.kind = k = case["kind"]
    s.lib = R.lib()
    R.check(s.lib.roaster_init(), "init")
    if k == "ffn":
        s.x = _normal(seed, 1, case["hidden"]).cpu().numpy()
        s.weights = _ffn_weights(case, seed)
        s.out = np.zeros((case["experts"], case["hidden"]), np.float32)
        s.experts = (R.KernelFfnExpert * case["experts"])()
        for x, w, o in zip(s.experts, s.weights, s.out):
            at = []
            for m in w:                                    # the caller's weight memory, filled once
                granted = C.c_size_t(0)
                p = s.lib.kernel_vk_alloc_weights(m.nbytes, C.byref(granted))
                if not p:
                    raise RuntimeError(R.last_error())
                C.memmove(p, m.ctypes.data, m.nbytes)
                at.append(p)
            x.gate, x.up, x.down = at
            x.gate_q6 = x.up_q6 = case["gate_up"]
            x.down_q6 = case["down"]
            x.out = o.ctypes.data
        s.args = (s.experts, case["experts"], s.x.ctypes.data, case["inter"], case["hidden"])
        return s
    T = case["tokens"]
    if k == "dense":
        s.w = _dense_weights(case, seed)
        s.x = _normal(seed, 1, T, case["cols"])
        s.y = torch.zeros(T, case["rows"], device="cuda")
        s.args = (s.w.data_ptr(), case["q6"], s.x.data_ptr(), s.y.data_ptr(), case["rows"], case["cols"], T)
        return s
    H = case["hidden"]
    s.table = _Table(case, seed)
    s.x = _normal(seed, 1, T, H)
    s.y = torch.zeros(T, H, device="cuda")
    if k == "block":
        s.args = (s.table.p, 0, s.x.data_ptr(), T, s.y.data_ptr(), None)
    elif k == "stack":
        n = case["layers"]
        s.norm = 1 + 0.1 * _normal(seed, 2, n, H)
        s.stream = torch.cuda.ExternalStream(s.lib.roaster_stream())
        s.args = (s.table.p, s.y.data_ptr(), T, 0, n, s.norm.data_ptr(), EPS, None, None)
    else:
        s.bias = _skew_bias(case, seed)
        s.opts = R.RoasterPrefillOpts(case["precision"], None, s.bias.data_ptr() if s.bias is not None else None,
                                      None, None, None, None)
        s.args = (s.table.p, 0, s.x.data_ptr(), T, s.y.data_ptr(), C.byref(s.opts))
    return s


def run(s):
    k = s.kind
    if k == "stack":
        with torch.cuda.stream(s.stream):                  # the tokens' embeddings become the hidden state
            s.y.copy_(s.x)
        R.check(s.lib.roaster_moe_decode_stack(*s.args), "decode_stack")
    elif k == "block":
        R.check(s.lib.roaster_moe_decode(*s.args), "decode")
    elif k == "prefill":
        R.check(s.lib.roaster_moe_prefill(*s.args), "prefill")
    elif k == "dense":
        R.check(s.lib.roaster_matvec_q(*s.args), "matvec_q")
    else:
        if s.lib.kernel_ffn_fused(*s.args) != 1:
            raise RuntimeError(R.last_error())
        return s.out
    return s.y


# ---- the same in 64 bits -----------------------------------------------------
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(raw, q6, rows, cols):
    """[rows x cols] f64 of Q4_K (d, dmin, 12 scale bytes, 128 nibble bytes) or Q6_K
    (128 low-nibble bytes, 64 high-bit bytes, 16 scales, d) blocks."""
    b = raw.reshape(-1, 210 if q6 else 144)
    n = b.shape[0]
    if q6:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo, hi = ql & 15, ql >> 4                          # [half][32-run][32]
        q = torch.cat([lo, hi], dim=2).to(torch.int16)     # runs 0, 1 (low), 2, 3 (high)
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = q | (((qh >> sh) & 3).to(torch.int16) << 4)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (q.double() - 32).reshape(n, 16, 16) * sc.unsqueeze(2) * _f16(b[:, 208:210]).unsqueeze(2)
        return w.reshape(rows, cols)
    d, dmin, s = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16]
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], dim=1).double()
    m = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1).double()
    qs = b[:, 16:144].reshape(n, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], dim=2).reshape(n, 8, 32).double()
    w = q * (d * sc).unsqueeze(2) - (dmin * m).unsqueeze(2)
    return w.reshape(rows, cols)


def _expert(table, case, layer, e):
    """gate, up, down of one expert in f64, from the bytes the table holds."""
    H, I = case["hidden"], case["inter"]
    gu, dn = _layer_types(case, layer)
    at = [C.c_void_p() for _ in range(3)]
    R.check(R.lib().roaster_table_expert_ptrs(table.p, layer, e, *(C.byref(p) for p in at)), "expert_ptrs")
    out = []
    for p, q6, rows, cols in zip(at, (gu, gu, dn), (I, I, H), (H, H, I)):
        raw = np.empty(_mat(q6, rows, cols), np.uint8)
        R.check(R.lib().roaster_d2h(raw.ctypes.data, p, raw.nbytes), "d2h")
        out.append(_dequant(torch.from_numpy(raw).cuda(), q6, rows, cols))
    return out


def _ffn64(x, gate, up, down):
    g = x @ gate.T
    return (g * torch.sigmoid(g) * (x @ up.T)) @ down.T


def _moe64(table, case, seed, layer, x, bias=None):
    router, gi = (torch.from_numpy(a).cuda().double() for a in R.host_router(seed, layer, table.desc, table.spec))
    logits = x @ router.T
    if bias is not None:
        logits = logits + bias.double()
    top, ids = torch.topk(logits, TOP, dim=1)
    w = torch.softmax(top, dim=1)
    y = torch.sigmoid(x @ gi).unsqueeze(1) * _ffn64(x, *_expert(table, case, layer, E))
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        y[t] += w[t, j].unsqueeze(1) * _ffn64(x[t], *_expert(table, case, layer, e))
    return y


def exact(case, seed):
    s = prepare(case, seed)
    torch.cuda.synchronize()
    k = case["kind"]
    if k == "ffn":
        H, I = case["hidden"], case["inter"]
        x = torch.from_numpy(s.x).cuda().double().unsqueeze(0)
        out = []
        for w in s.weights:
            g, u, d = (torch.from_numpy(m).cuda() for m in w)
            out.append(_ffn64(x, _dequant(g, case["gate_up"], I, H), _dequant(u, case["gate_up"], I, H),
                              _dequant(d, case["down"], H, I)))
        return torch.cat(out).cpu().numpy()
    x = s.x.double()
    if k == "dense":
        per, c = case["cols"] // 256, case["cols"]
        return torch.cat([x @ _dequant(b, case["q6"], b.shape[0] // per, c).T for b in s.w.split(16384 * per)], dim=1)
    if k == "stack":
        h = x
        for l in range(case["layers"]):
            n = h * torch.rsqrt((h * h).mean(dim=1, keepdim=True) + EPS) * s.norm[l].double()
            h = h + _moe64(s.table, case, seed, l, n)
        return h
    return _moe64(s.table, case, seed, 0, x, getattr(s, "bias", None))
