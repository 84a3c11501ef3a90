"""The decode-path work that this library is measured on.

Six kinds of case, each one pass through public entry points of
wohper_amd.Context at the model's widths (hidden 4096, 64 heads of 448 + 64,
q_lora 1024, 8 output groups of 1024, 256 routed + 1 shared FP4 expert of
intermediate width 2048, top-6, four copies of the residual stream):

  hyper    the hyper-connection glue around one sub-block of one token
  proj     the five FP8 projections of a layer for n positions
  window   the window softmax of one position over its cached and compressed rows
  mla      one MLA attention layer for n positions
  experts  the shared and routed FP4 experts for n positions
  layer    one whole decode layer for n positions

n = 1 is a decode step, a few positions are speculative verify, tens to
hundreds a prefill chunk.  `exact` chooses the library's two numerics modes:
the default one in the reference kernel's summation order, whose results are
the same bits whatever the kernel, and the order-free one.
"""
import math

import numpy as np
import torch

import wohper_amd
from wohper_amd import model_format

HIDDEN, INTER, N_EXPERTS, TOPK = 4096, 2048, 256, 6
HEADS, NOPE, ROPE, Q_LORA, GROUPS, O_LORA = 64, 448, 64, 1024, 8, 1024
HEAD_DIM = NOPE + ROPE
EXPERT_BYTES = 3 * (INTER * HIDDEN // 2 + INTER * HIDDEN // 32)
SCALE_LO, SCALE_HI = 113, 121  # UE8M0 exponents -14 .. -6 of the FP4 groups: gate and up outputs of order one
SHARED = N_EXPERTS             # the shared expert's id in its layer
SHAPES = {"wq_a": (Q_LORA, HIDDEN), "wkv": (HEAD_DIM, HIDDEN), "wq_b": (HEADS * HEAD_DIM, Q_LORA),
          "wo_a": (GROUPS * O_LORA, HEADS * HEAD_DIM // GROUPS), "wo_b": (HIDDEN, GROUPS * O_LORA)}


def listed():
    return [
        # the glue of a decode token's sub-block: the smallest launches, in the default numerics
        dict(name="hyper_1_exact", kind="hyper", hc=4, hidden=4096, exact=True),
        # a decode token's dense weights, 107 MB
        dict(name="proj_1", kind="proj", n=1, scales="f32", exact=False),
        # an uneven handful of positions in the default numerics, scales as the checkpoints store them
        dict(name="proj_13_exact", kind="proj", n=13, scales="ue8m0", exact=True),
        # a prefill chunk of the dense weights
        dict(name="proj_192", kind="proj", n=192, scales="f32", exact=False),
        # one position deep in a long context: a full window and a thousand compressed rows
        dict(name="window_1128", kind="window", heads=64, window=128, comp=1000, pos=4003, exact=False),
        # a prefill chunk's attention in a context of about two thousand tokens
        dict(name="mla_32", kind="mla", n=32, pos=2000, comp=500, exact=False),
        # a decode token's experts
        dict(name="experts_1", kind="experts", n=1, layers=2, zipf=False, bf16=True, shared=True, exact=False),
        # a batch of tokens with skewed expert popularity
        dict(name="experts_64", kind="experts", n=64, layers=1, zipf=True, bf16=True, shared=False, exact=False),
        # a small ragged batch in the default numerics
        dict(name="experts_24_exact", kind="experts", n=24, layers=1, zipf=True, bf16=False, shared=True, exact=True),
        # a whole decode layer, order-free and in the default numerics
        dict(name="layer_1", kind="layer", n=1, pos=127, comp=0, exact=False),
        dict(name="layer_1_exact", kind="layer", n=1, pos=700, comp=175, exact=True),
        # a whole layer over a prefill chunk from the start of a prompt
        dict(name="layer_128", kind="layer", n=128, pos=0, comp=32, exact=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hyper", "proj", "proj", "window", "mla", "experts", "experts", "layer", "layer"])
    exact = rng.random() < 0.4
    if kind == "hyper":
        return dict(kind=kind, hc=rng.choice([2, 4, 4, 4]), hidden=4 * _log_int(rng, 128, 1024), exact=exact)
    if kind == "proj":
        return dict(kind=kind, n=_log_int(rng, 1, 24 if exact else 224), scales=rng.choice(["f32", "ue8m0"]),
                    exact=exact)
    if kind == "window":
        return dict(kind=kind, heads=rng.choice([16, 50, 64, 64, 128]), window=rng.choice([128, 128, rng.randint(1, 127)]),
                    comp=_log_int(rng, 16, 1900), pos=rng.randint(128, 30000), exact=exact)
    if kind == "mla":
        pos = rng.randint(0, 4000)
        return dict(kind=kind, n=_log_int(rng, 1, 12 if exact else 40), pos=pos, comp=rng.randint(0, pos // 4),
                    exact=exact)
    if kind == "experts":
        n = _log_int(rng, 1, 24 if exact else 128)
        return dict(kind=kind, n=n, layers=2 if n == 1 else 1, zipf=rng.random() < 0.5, bf16=rng.random() < 0.5,
                    shared=rng.random() < 0.7, exact=exact)
    pos = rng.randint(0, 2000)
    return dict(kind=kind, n=_log_int(rng, 1, 8 if exact else 96), pos=pos, comp=rng.randint(0, pos // 4), exact=exact)


# ------------------------------------------------------------ what a program keeps

_contexts = {}
_live_layers = set()


def _context(exact):
    """One context per numerics mode for the whole process, as a program has."""
    if exact not in _contexts:
        ctx = wohper_amd.Context(0)
        ctx.set_exact_numerics(exact)
        _contexts[exact] = ctx
    return _contexts[exact]


class _State:
    """A case's inputs and weights.  Its tensors go back to the store with it;
    its synthetic experts stay until a later state's replace them under the
    same layer id.  The id is the seed's, as the generator's bytes depend on
    it, out of sixteen so that the store stays bounded."""

    def __init__(self, case, seed):
        self.case, self.exact = case, bool(case["exact"])
        self.ctx = _context(self.exact)
        self.handles, self.layer_ids = [], []
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.seed = seed
        self.on_stream = torch.cuda.stream(torch.cuda.ExternalStream(self.ctx.stream))

    def layer_id(self, k=0):
        layer = _layer_of(self.seed, k)
        if (self.exact, layer) in _live_layers:
            raise RuntimeError("two live states use one layer id: take seeds that differ modulo 16")
        _live_layers.add((self.exact, layer))
        self.layer_ids.append(layer)
        return layer

    def __del__(self):
        try:
            _live_layers.difference_update((self.exact, k) for k in self.layer_ids)
            torch.cuda.synchronize()
            for t in self.handles:
                self.ctx.release(t)
        except Exception:  # the process's end
            pass


def _normal(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32) * scale


def _bf16_values(gen, *shape):
    return _normal(gen, *shape).bfloat16()


def _norm_weight(gen, n):
    return (1.0 + 0.1 * _normal(gen, n)).bfloat16()


def _fp8_inputs(gen, rows, cols, scales):
    """E4M3 codes uniform over the finite ones and 128 x 128 block scales
    2^U, U in [-16, -10] (whole for UE8M0, as bytes): outputs of order one."""
    c = torch.randint(0, 254, (rows, cols), generator=gen, device="cuda", dtype=torch.int16)
    codes = torch.where(c < 127, c, c + 1).to(torch.uint8)
    u = torch.rand(rows // 128, cols // 128, generator=gen, device="cuda", dtype=torch.float64) * 6.0 - 16.0
    if scales == "ue8m0":
        return codes, (torch.round(u) + 127).to(torch.uint8)
    return codes, torch.exp2(u).float()


def _store_fp8(s, codes, scales):
    fmt = wohper_amd.SCALE_UE8M0 if scales.dtype == torch.uint8 else wohper_amd.SCALE_F32
    t = s.ctx.store_fp8(codes.cpu().numpy(), *codes.shape, scales.cpu().numpy(), *scales.shape, fmt)
    s.handles.append(t)
    return t


def _routes(case, seed, layer):
    """[n, 6] expert ids and their sigmoid scores: the top 6 of N(0, 1)
    logits, or with `zipf` drawn without replacement from a popularity
    (rank + 1)^-1.1 over a seeded permutation of the experts."""
    r = np.random.default_rng([seed, layer, 11])
    n = case["n"]
    logits = r.standard_normal((n, N_EXPERTS))
    if case["zipf"]:
        pop = np.empty(N_EXPERTS)
        pop[r.permutation(N_EXPERTS)] = np.arange(1, N_EXPERTS + 1) ** -1.1
        key = np.log(pop) + r.gumbel(size=(n, N_EXPERTS))
    else:
        key = logits
    ids = np.argsort(-key, axis=1, kind="stable")[:, :TOPK]
    scores = 1.0 / (1.0 + np.exp(-np.take_along_axis(logits, ids, 1)))
    return ids.astype(np.uint32), scores.astype(np.float32)


def _layer_of(seed, k=0):
    return 1 + 2 * (seed % 16) + k


def _positions(case):
    """The positions of a chunk and how many compressed rows each sees: one
    for every four tokens before it, at most `comp`."""
    pos = list(range(case["pos"], case["pos"] + case["n"]))
    return pos, [min(case["comp"], (p + 1) // 4) for p in pos]


def _mla(s, gen):
    t = {k: _store_fp8(s, *_fp8_inputs(gen, r, c, "f32")) for k, (r, c) in SHAPES.items()}
    s.q_norm, s.kv_norm, s.sink = _norm_weight(gen, Q_LORA), _norm_weight(gen, HEAD_DIM), _normal(gen, HEADS)
    s.mla = wohper_amd.WhMlaLayer(2, HEADS, NOPE, ROPE, GROUPS, O_LORA, t["wq_a"], t["wq_b"], t["wkv"], t["wo_a"],
                                  t["wo_b"], s.q_norm.data_ptr(), s.kv_norm.data_ptr(), s.sink.data_ptr())
    s.pos, s.n_comp = _positions(s.case)
    s.cap = s.pos[-1] + 1
    s.kv = _normal(gen, s.cap, HEAD_DIM)
    s.comp = _normal(gen, max(1, s.case["comp"]), HEAD_DIM)
    s.comps = [(s.comp.data_ptr() if k else 0, k) for k in s.n_comp]


def prepare(case, seed):
    s = _State(case, seed)
    ctx, gen, kind = s.ctx, s.gen, case["kind"]
    if kind == "hyper":
        hc, hidden = case["hc"], case["hidden"]
        mix = (2 + hc) * hc
        s.x, s.fn, s.scale, s.base, s.w = _hyper_inputs(case, seed)
        s.y, s.g, s.out = (torch.empty(k, device="cuda") for k in (hidden, hidden, hc * hidden))
        s.post, s.comb = torch.empty(hc, device="cuda"), torch.empty(hc * hc, device="cuda")
    elif kind == "proj":
        n = case["n"]
        w, x = _proj_inputs(case, seed)
        s.x = x
        s.t = {k: _store_fp8(s, *v) for k, v in w.items()}
        s.y = {k: torch.empty(n, r, device="cuda") for k, (r, _) in SHAPES.items()}
        if n == 1:
            p = {k: v.data_ptr() for k, v in s.x.items()}
            y = {k: v.data_ptr() for k, v in s.y.items()}
            cols = SHAPES["wo_a"][1]
            s.descs = ctx.gemv_descs(
                [(s.t[k], 0, SHAPES[k][0], p["h"], y[k]) for k in ("wq_a", "wkv")] +
                [(s.t["wq_b"], 0, SHAPES["wq_b"][0], p["q"], y["wq_b"])] +
                [(s.t["wo_a"], g * O_LORA, (g + 1) * O_LORA, p["a"] + 4 * g * cols, y["wo_a"] + 4 * g * O_LORA)
                 for g in range(GROUPS)] + [(s.t["wo_b"], 0, HIDDEN, p["b"], y["wo_b"])])
    elif kind == "window":
        s.q, s.win, s.comp, s.sink = _window_inputs(case, seed)
        theta, yarn = wohper_amd.deepseek_rope_for_layer(2)
        s.inv = torch.from_numpy(wohper_amd.rope_inv_freqs(ROPE, theta, yarn)).cuda()
        keys = case["window"] + case["comp"]
        s.scores = torch.empty(case["heads"], keys, device="cuda")
        s.out = torch.empty(case["heads"], HEAD_DIM, device="cuda")
    elif kind == "mla":
        _mla(s, gen)
        s.hidden0 = _normal(gen, case["n"], HIDDEN)
        s.hidden = torch.empty_like(s.hidden0)
    elif kind == "experts":
        s.work, s.x = [], []
        for k in range(case["layers"]):
            layer = s.layer_id(k)
            ids, scores = _routes(case, seed, k)
            used = sorted(set(ids.reshape(-1).tolist())) + ([SHARED] if case["shared"] else [])
            for e in used:
                # the generator's stream of (0, e), whatever the store's layer id
                ctx.store_expert_synthetic(layer, e, HIDDEN, INTER, seed, SCALE_LO, SCALE_HI)
            x = _experts_x(case, seed, k)
            out = torch.empty(case["n"], HIDDEN, device="cuda")
            shared = (layer, SHARED) if case["shared"] else None
            if case["n"] == 1:
                w = scores[0] / scores[0].sum()
                routes = ctx.route_array([(layer, int(e), float(v)) for e, v in zip(ids[0], w)])
                s.work.append((layer, routes, shared, x, out))
            else:
                s.work.append((layer, (torch.from_numpy(ids.view(np.int32)).cuda(), torch.from_numpy(scores).cuda()),
                               shared, x, out))
    else:
        layer = s.layer_id()
        for e in range(N_EXPERTS + 1):
            ctx.store_expert_synthetic(layer, e, HIDDEN, INTER, seed, SCALE_LO, SCALE_HI)
        _mla(s, gen)
        gate = _normal(gen, N_EXPERTS, HIDDEN, scale=0.02).bfloat16().view(torch.int16).cpu().numpy()
        bias = _normal(gen, N_EXPERTS, scale=0.05).cpu().numpy()
        ctx.store_router(layer, model_format.build_synthetic_quant_block([
            model_format.SyntheticTensor("layers.0.ffn.gate.weight", 9, (N_EXPERTS, HIDDEN), gate.tobytes(), 11, 2404),
            model_format.SyntheticTensor("layers.0.ffn.gate.bias", 9, (N_EXPERTS,), bias.tobytes(), 12, 2405)]), HIDDEN)
        hc = 4
        mix = (2 + hc) * hc
        s.fns = [_normal(gen, mix, hc * HIDDEN, scale=(hc * HIDDEN) ** -0.5) for _ in range(2)]
        s.scales = [0.5 + torch.rand(3, generator=gen, device="cuda") for _ in range(2)]
        s.bases = [_normal(gen, mix, scale=0.5) for _ in range(2)]
        s.norms = [_norm_weight(gen, HIDDEN) for _ in range(2)]
        d = wohper_amd.WhMhcLayer()
        d.hc, d.hidden, d.sinkhorn_iters, d.hc_eps = hc, HIDDEN, 20, 1e-6
        d.hc_attn_fn, d.hc_ffn_fn = (t.data_ptr() for t in s.fns)
        d.hc_attn_scale, d.hc_ffn_scale = (t.data_ptr() for t in s.scales)
        d.hc_attn_base, d.hc_ffn_base = (t.data_ptr() for t in s.bases)
        d.attn_norm_bf16, d.ffn_norm_bf16 = (t.data_ptr() for t in s.norms)
        d.attn, d.layer_id, d.active, d.available_dev, d.n_available = s.mla, layer, TOPK, None, 0
        d.route = ctx.route_options(wohper_amd.ROUTER_SQRT_SOFTPLUS, 1.5)
        d.shared_layer, d.shared_expert = layer, SHARED
        s.layer = d
        # a residual stream a few times a sub-block's output, as it is past the first layers
        s.hidden0 = _normal(gen, case["n"], hc * HIDDEN, scale=8.0)
        s.hidden = torch.empty_like(s.hidden0)
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, case, kind = s.ctx, s.case, s.case["kind"]
    if kind == "hyper":
        hc, hidden = case["hc"], case["hidden"]
        x, y, g, post, comb = (t.data_ptr() for t in (s.x, s.y, s.g, s.post, s.comb))
        ctx.hc_pre_async(s.fn.data_ptr(), s.scale.data_ptr(), s.base.data_ptr(), hc, hidden, 20, 1e-6, x, y, post, comb)
        ctx.rms_norm_async(y, g, 1, hidden, s.w.data_ptr())
        ctx.hc_post_async(g, x, post, comb, s.out.data_ptr(), hc, hidden)
        return {"y": s.y, "post": s.post, "comb": s.comb, "norm": s.g, "out": s.out}
    if kind == "proj":
        n = case["n"]
        if n == 1:
            ctx.fp8_gemv_batch_async(s.descs)
            return s.y
        x = {k: v.data_ptr() for k, v in s.x.items()}
        y = {k: v.data_ptr() for k, v in s.y.items()}
        (ra, _), (rkv, _), (rb, _), (roa, coa) = (SHAPES[k] for k in ("wq_a", "wkv", "wq_b", "wo_a"))
        ctx.fp8_gemv_multi_pair_async(s.t["wq_a"], 0, ra, y["wq_a"], ra, s.t["wkv"], 0, rkv, y["wkv"], rkv, x["h"], n,
                                      HIDDEN)
        ctx.fp8_gemv_multi_async(s.t["wq_b"], 0, rb, x["q"], n, Q_LORA, y["wq_b"], rb)
        ctx.fp8_gemv_multi_groups_async(s.t["wo_a"], 0, roa, O_LORA, x["a"], coa, n, GROUPS * coa, y["wo_a"], roa)
        ctx.fp8_gemv_multi_async(s.t["wo_b"], 0, HIDDEN, x["b"], n, GROUPS * O_LORA, y["wo_b"], HIDDEN)
        return s.y
    if kind == "window":
        ctx.window_attention_async(s.q.data_ptr(), case["heads"], HEAD_DIM, NOPE, s.win.data_ptr(), case["window"],
                                   HEAD_DIM, s.comp.data_ptr(), case["comp"], s.sink.data_ptr(), s.inv.data_ptr(),
                                   ROPE // 2, case["pos"], s.scores.data_ptr(), s.out.data_ptr())
        return s.out
    if kind == "experts":
        outs = []
        for layer, routes, shared, x, out in s.work:
            if case["n"] == 1 and shared:
                ctx.routed_and_shared_experts_async(routes, shared, x.data_ptr(), case["bf16"], 1, out.data_ptr(),
                                                    n_routes=TOPK)
            elif case["n"] == 1:
                ctx.routed_experts_async([(r.layer_id, r.expert_id, r.route_weight) for r in routes], x.data_ptr(),
                                         case["bf16"], 1, out.data_ptr())
            else:
                ctx.moe_batch_async(layer, routes[0].data_ptr(), routes[1].data_ptr(), case["n"], TOPK, x.data_ptr(),
                                    case["bf16"], out.data_ptr(), shared)
            outs.append(out)
        return outs
    # the layers work on the hidden state in place: a pass begins with a new one
    with s.on_stream:
        s.hidden.copy_(s.hidden0)
    h, kv = s.hidden.data_ptr(), s.kv.data_ptr()
    if kind == "mla" and case["n"] == 1:
        ctx.mla_attention_decode_async(s.mla, s.pos[0], h, kv, HEAD_DIM, s.cap, *s.comps[0])
    elif kind == "mla":
        ctx.mla_attention_decode_batch_async(s.mla, s.pos, h, kv, HEAD_DIM, s.cap, s.comps)
    elif case["n"] == 1:
        ctx.deepseek_mhc_layer_async(s.layer, s.pos[0], h, kv, HEAD_DIM, s.cap, *s.comps[0])
    else:
        ctx.deepseek_mhc_layer_batch_async(s.layer, s.pos, h, kv, HEAD_DIM, s.cap, s.comps)
    return {"hidden": s.hidden, "kv": s.kv[s.pos[0]:]}


# ------------------------------------------------------------ inputs that exact() makes again

def _hyper_inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    hc, hidden = case["hc"], case["hidden"]
    mix = (2 + hc) * hc
    return (_normal(gen, hc * hidden, scale=0.5), _normal(gen, mix, hc * hidden, scale=(hc * hidden) ** -0.5),
            0.5 + torch.rand(3, generator=gen, device="cuda"), _normal(gen, mix, scale=0.5), _norm_weight(gen, hidden))


def _proj_inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n = case["n"]
    w = {k: _fp8_inputs(gen, r, c, case["scales"]) for k, (r, c) in SHAPES.items()}
    cols = {"h": HIDDEN, "q": Q_LORA, "a": GROUPS * SHAPES["wo_a"][1], "b": GROUPS * O_LORA}
    return w, {k: _normal(gen, n, c) for k, c in cols.items()}


def _window_inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return (_normal(gen, case["heads"], HEAD_DIM), _normal(gen, case["window"], HEAD_DIM),
            _normal(gen, case["comp"], HEAD_DIM), _normal(gen, case["heads"]))


def _experts_x(case, seed, layer):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 7919 * (layer + 1))
    x = _bf16_values(gen, case["n"], HIDDEN)
    return x if case["bf16"] else x.float()


def work(case):
    kind = case["kind"]
    proj = sum(r * c + (r // 128) * (c // 128) * 4 for r, c in SHAPES.values())
    if kind == "hyper":
        hcd, mix = case["hc"] * case["hidden"], (2 + case["hc"]) * case["hc"]
        return {"bytes": 4 * (hcd * (mix + 2) + 2 * case["hidden"]) + 2 * case["hidden"], "flops": 2 * hcd * (mix + 4)}
    if kind == "window":
        keys = case["window"] + case["comp"]
        return {"bytes": 4 * (keys * HEAD_DIM + 2 * case["heads"] * HEAD_DIM),
                "flops": 4 * case["heads"] * keys * HEAD_DIM}
    n = case["n"]
    dense = 2 * n * sum(r * c for r, c in SHAPES.values())
    if kind == "proj":
        ins = HIDDEN + Q_LORA + GROUPS * SHAPES["wo_a"][1] + GROUPS * O_LORA
        return {"bytes": proj + 4 * n * (ins + sum(r for r, _ in SHAPES.values())), "flops": dense}
    if kind == "experts":
        used = sum(len(set(_routes(case, 1, k)[0].reshape(-1).tolist())) + bool(case["shared"])
                   for k in range(case["layers"]))
        per = 6 * HIDDEN * INTER * (TOPK + bool(case["shared"]))
        return {"bytes": used * EXPERT_BYTES + case["layers"] * n * HIDDEN * ((2 if case["bf16"] else 4) + 4),
                "flops": case["layers"] * n * per}
    pos, comp = _positions(case)
    keys = sum(min(p + 1, 128) + k for p, k in zip(pos, comp))
    rows = min(pos[-1] + 1, 127 + n) + max(comp)
    attn = {"bytes": proj + 4 * (rows * HEAD_DIM + 2 * n * HIDDEN), "flops": dense + 4 * HEADS * HEAD_DIM * keys}
    if kind == "mla":
        return attn
    used = N_EXPERTS * (1.0 - (1.0 - TOPK / N_EXPERTS) ** n) + 1
    return {"bytes": attn["bytes"] + int(used * EXPERT_BYTES) + N_EXPERTS * HIDDEN * 2 + 4 * (2 * 24 + 2 * n) * 4 * HIDDEN,
            "flops": attn["flops"] + n * (6 * HIDDEN * INTER * (TOPK + 1) + 2 * N_EXPERTS * HIDDEN)}


def tolerance(case):
    """Exact numerics are the same bits by contract.  Order-free, each figure
    is about four times what the two numerics modes differ by (measured:
    hyper 1.6e-6, proj 2.3e-7, experts 3e-4 to 2e-3, mla 8e-4, layer 8e-3;
    the last three through values that round to the next E4M3 step); the
    window softmax has one order, and the figure is four times its distance
    from 64 bits."""
    if case["exact"]:
        return "exact"
    return {"hyper": {"rel": 6e-6}, "proj": {"rel": 1e-6}, "window": {"rel": 4e-6}, "experts": {"rel": 8e-3},
            "mla": {"rel": 1e-2}, "layer": {"rel": 3e-2}}[case["kind"]]


# ------------------------------------------------------------ the same in 64 bits

def _fp8_values(codes, scales):
    """E4M3 codes times their block scales, in 64 bits."""
    c = codes.long()
    e, m = (c >> 3) & 15, (c & 7).double()
    v = torch.where(e == 0, m * 2.0 ** -9, (1.0 + m / 8.0) * torch.exp2(e.double() - 7.0))
    v = torch.where(c >= 128, -v, v)
    sc = torch.exp2(scales.double() - 127.0) if scales.dtype == torch.uint8 else scales.double()
    return v * sc.repeat_interleave(128, 0).repeat_interleave(128, 1)


def _signed(k):
    """A 64-bit word as the signed integer of the same bits."""
    return k - (1 << 64) if k >> 63 else k


def _mix(v):
    """The splitmix64 finaliser on 64-bit words held as signed integers."""
    def shr(a, k):
        return (a >> k) & ((1 << (64 - k)) - 1)
    v = v + _signed(0x9E3779B97F4A7C15)
    v = (v ^ shr(v, 30)) * _signed(0xBF58476D1CE4E5B9)
    v = (v ^ shr(v, 27)) * _signed(0x94D049BB133111EB)
    return v ^ shr(v, 31)


def _synth_bytes(seed, stream, n):
    """n bytes of the synthetic weights' counter-based generator."""
    word = torch.arange((n + 7) // 8, device="cuda", dtype=torch.int64)
    v = _mix(seed ^ _mix(word + _signed((stream * 0x100000001B3) % (1 << 64))))
    return v.view(torch.uint8)[:n]


def _fp4_matrix(seed, layer, expert, m):
    """Matrix m (w1, w3, w2) of a synthetic expert in 64 bits: the engine's
    E2M1 table (0.125 for code 1) times the UE8M0 scale of 32 columns."""
    rows, cols = (INTER, HIDDEN) if m < 2 else (HIDDEN, INTER)
    stream = (layer << 40) ^ (expert << 8) ^ m
    b = _synth_bytes(seed, stream, rows * cols // 2)
    s = _synth_bytes(seed, stream ^ 0x5CA1E5, rows * cols // 32)
    s = SCALE_LO + s.long() % (SCALE_HI - SCALE_LO + 1)
    lut = torch.tensor([0, 0.125, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
    lut = torch.cat([lut, -lut])
    v = lut[torch.stack([b & 15, b >> 4], 1).reshape(-1).long()].reshape(rows, cols // 32, 32)
    return (v * torch.exp2(s.double() - 127.0).reshape(rows, cols // 32, 1)).reshape(rows, cols)


def _act_quant(x):
    """x rounded to E4M3 under a power-of-two scale per 64 columns, ties
    toward minus infinity as the engine's table search has them."""
    b = x.reshape(x.shape[0], -1, 64)
    amax = b.abs().amax(2, keepdim=True).clamp_min(1e-4)
    sc = torch.exp2(torch.ceil(torch.log2(amax / 448.0)))
    q = (b / sc).clamp(-448.0, 448.0)
    step = torch.exp2(torch.floor(torch.log2(q.abs().clamp_min(2.0 ** -6))) - 3.0)
    return (torch.ceil(q / step - 0.5) * step * sc).reshape(x.shape)


def _rotate(v, pos, inverse):
    """Interleaved RoPE of the last ROPE columns; the angle is the product of
    two 32-bit numbers, rounded to 32 bits, by definition of the operation."""
    theta, yarn = wohper_amd.deepseek_rope_for_layer(2)
    inv = torch.from_numpy(wohper_amd.rope_inv_freqs(ROPE, theta, yarn)).cuda()
    ang = (torch.tensor(float(pos), device="cuda") * inv).double()
    sn, cs = torch.sin(ang), torch.cos(ang)
    sn = -sn if inverse else sn
    e, o = v[:, NOPE::2].clone(), v[:, NOPE + 1::2].clone()
    v = v.clone()
    v[:, NOPE::2], v[:, NOPE + 1::2] = e * cs - o * sn, e * sn + o * cs
    return v


def _exact_hyper(case, seed):
    x, fn, scale, base, w = (t.double() for t in _hyper_inputs(case, seed))
    hc, hidden, eps = case["hc"], case["hidden"], float(np.float32(1e-6))
    mixes = (fn @ x) / torch.sqrt((x * x).mean() + eps)
    pre = torch.sigmoid(mixes[:hc] * scale[0] + base[:hc]) + eps
    post = 2.0 * torch.sigmoid(mixes[hc:2 * hc] * scale[1] + base[hc:2 * hc])
    comb = torch.softmax((mixes[2 * hc:] * scale[2] + base[2 * hc:]).reshape(hc, hc), 1) + eps
    comb = comb / (comb.sum(0, keepdim=True) + eps)
    for _ in range(19):
        comb = comb / (comb.sum(1, keepdim=True) + eps)
        comb = comb / (comb.sum(0, keepdim=True) + eps)
    xs = x.reshape(hc, hidden)
    y = pre @ xs
    g = y / torch.sqrt((y * y).mean() + eps) * w
    out = post[:, None] * g[None] + comb @ xs
    return {"y": y, "post": post, "comb": comb.reshape(-1), "norm": g, "out": out.reshape(-1)}


def _exact_proj(case, seed):
    w, x = _proj_inputs(case, seed)
    x = {k: v.double() for k, v in x.items()}
    v = {k: _fp8_values(*t) for k, t in w.items()}
    cols = SHAPES["wo_a"][1]
    y = {k: x[i] @ v[k].T for k, i in (("wq_a", "h"), ("wkv", "h"), ("wq_b", "q"), ("wo_b", "b"))}
    y["wo_a"] = torch.cat([x["a"][:, g * cols:(g + 1) * cols].contiguous() @ v["wo_a"][g * O_LORA:(g + 1) * O_LORA].T
                           for g in range(GROUPS)], 1)
    return y


def _exact_window(case, seed):
    q, win, comp, sink = (t.double() for t in _window_inputs(case, seed))
    keys = torch.cat([win, comp])
    sc = torch.cat([(q @ keys.T) * HEAD_DIM ** -0.5, sink[:, None]], 1)
    p = torch.softmax(sc, 1)[:, :-1]
    return _rotate(p @ keys, case["pos"], True)


def _exact_experts(case, seed):
    outs = []
    for k in range(case["layers"]):
        layer = _layer_of(seed, k)
        ids, scores = _routes(case, seed, k)
        ids = torch.from_numpy(ids.astype(np.int64)).cuda()
        wts = torch.from_numpy(scores).cuda().double()
        wts = wts / wts.sum(1, keepdim=True)
        x = _act_quant(_experts_x(case, seed, k).double())
        out = torch.zeros(case["n"], HIDDEN, device="cuda", dtype=torch.float64)
        for e in sorted(set(ids.reshape(-1).tolist())) + ([SHARED] if case["shared"] else []):
            if e == SHARED:
                at, w = torch.arange(case["n"], device="cuda"), torch.ones(case["n"], device="cuda", dtype=torch.float64)
            else:
                at, slot = torch.nonzero(ids == e, as_tuple=True)
                w = wts[at, slot]
            w1, w3, w2 = (_fp4_matrix(seed, layer, e, m) for m in range(3))
            g, u = (x[at] @ w1.T).clamp_max(10.0), (x[at] @ w3.T).clamp(-10.0, 10.0)
            h = _act_quant(g * torch.sigmoid(g) * u)
            out.index_add_(0, at, (h @ w2.T) * w[:, None])
        outs.append(out)
    return outs


def exact(case, seed):
    """None for an attention layer and a whole layer: they round computed
    values to E4M3 between their projections, where a last-bit difference of
    a 32-bit sum moves a value by a whole step and the later stages carry it
    on, so 64 bits give another result and not a closer one; their single
    stages are the other kinds."""
    f = {"hyper": _exact_hyper, "proj": _exact_proj, "window": _exact_window, "experts": _exact_experts}.get(case["kind"])
    return f(case, seed) if f else None
