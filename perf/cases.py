"""The work that users of this package have it do, as cases that can be timed and checked.

``listed()`` names the cases, ``draw`` gives more of the same ranges, ``prepare`` makes what a program
holds before the call, ``run`` is one pass through the public entry points, ``work`` the bytes and
flops of one pass that nothing can do without, ``tolerance`` what another correct implementation at
the same precision may differ by, and ``exact`` the same results from plain torch in 64 bits (rounded
only where the path's contract stores a tensor in its own dtype: conv outputs, gates, normalised q/k).

Kinds:
  unfused   one decode token through the separate ops a patched transformers layer calls
  decode    the graph-captured fused decode step over a stack of GDN layers
  mlp       a decode step's MLP: gate_up, SwiGLU, down, residual add + norm
  attention a decode step's GQA attention over per-slot caches
  hybrid    a whole graph-captured decode step (GDN + attention + MLP + LM head), logits out
  rule      the chunked gated delta rule, bf16 at head dim 128 (the model's shape)
  layer     the fused prefill layer between the projections, packed prompts or slot continuation
  generic   the chunked rule at other dtypes and head dims
"""
import importlib
import math

import torch

PKG = "910b_e2e_accleration_by_codex_amd"
gdn = importlib.import_module(PKG)
cb = importlib.import_module(PKG + ".cb_engine")
hybrid = importlib.import_module(PKG + ".hybrid_decode")

D, K = 128, 4
EPS = 1e-6
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
BF = torch.bfloat16


def listed():
    return [
        # one request in flight, unfused ops: the smallest call, host time and launches
        dict(name="unfused_decode_1slot", kind="unfused", slots=1, hk=16, hv=48),
        # the continuous-batching decode step, 16 slots x 48 GDN layers, graph replay
        dict(name="decode_step_48layers", kind="decode", slots=16, layers=48, hk=16, hv=32),
        # the MLP of a 27B-shaped decode layer: two weight streams and what is between them
        dict(name="mlp_decode_16", kind="mlp", slots=16, hidden=5120, mlp=17408),
        # the full-attention layer's decode attention at 27B shape, contexts of 512 to 4096
        dict(name="attention_decode_16", kind="attention", slots=16, heads=24, kv=4, hd=256, ctx_lo=512, ctx_hi=4096),
        # a whole decode step: 3 GDN layers, 1 attention layer, their MLPs and the LM head
        dict(name="hybrid_step_4layers", kind="hybrid", slots=16, hidden=5120, layers=4, mlp=17408, vocab=248320,
             ctx_lo=512, ctx_hi=4096),
        # one short prompt through the rule (353 tokens at the 27B GDN shape)
        dict(name="rule_353", kind="rule", b=1, t=353, hk=16, hv=48, decay="fast", beta="bf16", init=True),
        # the ordinary prefill chunk
        dict(name="rule_8192", kind="rule", b=1, t=8192, hk=16, hv=32, decay="fast", beta="bf16", init=True),
        # the same with long-memory heads only
        dict(name="rule_8192_slow", kind="rule", b=1, t=8192, hk=16, hv=32, decay="slow", beta="bf16", init=True),
        # the longest prompt, heads of every memory length
        dict(name="rule_32768", kind="rule", b=1, t=32768, hk=16, hv=32, decay="mixed", beta="bf16", init=True),
        # a batch of 16 fresh prompts through the fused layer
        dict(name="layer_16prompts", kind="layer", prompts=16, lo=200, hi=1500, hk=16, hv=32, cont=False),
        # one prompt's next chunk, continuing in its slot
        dict(name="layer_continue_517", kind="layer", prompts=1, lo=517, hi=517, hk=16, hv=48, cont=True),
        # the reference's CPU-runnable shape: fp32, 4 heads of 64
        dict(name="generic_fp32_512", kind="generic", dtype="fp32", b=1, t=512, hk=4, hv=4, dk=64, dv=64),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["unfused", "decode", "mlp", "attention", "hybrid", "rule", "rule", "layer", "layer", "generic"])
    hk = rng.choice([4, 8, 16])
    if kind == "unfused":
        return dict(kind=kind, slots=_log_int(rng, 1, 32), hk=hk, hv=hk * rng.choice([1, 2, 3]))
    if kind == "decode":
        hv = hk * rng.choice([1, 2, 3])
        slots = _log_int(rng, 1, 32)
        return dict(kind=kind, slots=slots, layers=_log_int(rng, 1, max(1, min(48, 48 * 16 * 32 // (slots * hv)))),
                    hk=hk, hv=hv)
    if kind == "mlp":
        return dict(kind=kind, slots=rng.randint(1, 16), hidden=128 * _log_int(rng, 4, 40), mlp=128 * _log_int(rng, 8, 136))
    if kind == "attention":
        hd, kv, slots = rng.choice([64, 128, 256]), rng.choice([1, 2, 4, 8]), _log_int(rng, 1, 32)
        hi = _log_int(rng, 64, max(64, min(16384, 16 * 4096 * 4 * 256 * 4 // (slots * kv * hd))))
        return dict(kind=kind, slots=slots, heads=kv * rng.choice([1, 2, 4, 6, 8]), kv=kv, hd=hd,
                    ctx_lo=max(1, hi // rng.choice([1, 2, 8])), ctx_hi=hi)
    if kind == "hybrid":
        hi = _log_int(rng, 64, 4096)
        return dict(kind=kind, slots=rng.randint(1, 16), hidden=128 * _log_int(rng, 8, 40), layers=rng.randint(1, 4),
                    mlp=128 * _log_int(rng, 16, 136), vocab=_log_int(rng, 1000, 248320), ctx_lo=max(1, hi // 4), ctx_hi=hi)
    if kind == "rule":
        hv = hk * rng.choice([1, 2, 3])
        b = rng.choice([1, 1, 1, 2, 3])
        return dict(kind=kind, b=b, t=_log_int(rng, 1, 32768 * 32 // (b * max(hv, 32))), hk=hk, hv=hv,
                    decay=rng.choice(["fast", "fast", "mixed", "slow"]), beta=rng.choice(["bf16", "fp32"]),
                    init=rng.random() < 0.7)
    if kind == "layer":
        prompts, hi = _log_int(rng, 1, 16), _log_int(rng, 8, 1500)
        return dict(kind=kind, prompts=prompts, lo=max(1, hi // rng.choice([1, 2, 6])), hi=hi, hk=hk,
                    hv=hk * rng.choice([1, 2, 3]), cont=rng.random() < 0.4)
    dtype = rng.choice(["fp32", "fp32", "bf16", "fp16"])
    hk = rng.choice([1, 2, 4, 8])
    return dict(kind="generic", dtype=dtype, b=rng.choice([1, 1, 2, 3]), t=_log_int(rng, 1, 2048), hk=hk,
                hv=hk * rng.choice([1, 2]), dk=rng.choice([16, 32, 64, 128]), dv=rng.choice([16, 32, 64]))


# ---- inputs ---------------------------------------------------------------------------------------
class _Rand:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda:0")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def n(self, *shape, scale=1.0, dtype=BF):
        return (torch.randn(*shape, generator=self.g, device=self.dev) * scale).to(dtype)

    def u(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device=self.dev) * (hi - lo) + lo


def _rates(r, hv, decay):
    """exp(A_log) per value head: a token's log decay is about -2.1 times it."""
    if decay == "fast":
        return torch.full((hv,), 0.1, device=r.dev)
    if decay == "slow":
        return torch.full((hv,), 0.001, device=r.dev)
    return torch.exp(r.u(hv, lo=math.log(0.003), hi=math.log(1.0)))


def _rule_inputs(case, seed):
    r = _Rand(seed)
    b, t, hk, hv = case["b"], case["t"], case["hk"], case["hv"]
    dt = DTYPES[case.get("dtype", "bf16")]
    dk, dv = case.get("dk", D), case.get("dv", D)
    x = dict(q=r.n(b, t, hk, dk, dtype=dt), k=r.n(b, t, hk, dk, dtype=dt), v=r.n(b, t, hv, dv, dtype=dt))
    x["beta"] = torch.sigmoid(r.n(b, t, hv, dtype=torch.float32)).to(DTYPES[case.get("beta", case.get("dtype", "bf16"))])
    x["g"] = -torch.nn.functional.softplus(r.n(b, t, hv, dtype=torch.float32) + 2) * _rates(r, hv, case.get("decay", "fast"))
    x["s0"] = r.n(b, hv, dk, dv, scale=0.02, dtype=torch.float32) if case.get("init", True) else None
    return x


def _gdn_params(r, hk, hv):
    c = (2 * hk + hv) * D
    return dict(cw=r.n(c, K, scale=0.5), A_log=torch.log(_rates(r, hv, "mixed")),
                dt=1.0 + r.n(hv, dtype=torch.float32, scale=0.5), nw=(1 + r.n(D, scale=0.02, dtype=torch.float32)).to(BF))


def _decode_inputs(case, seed):
    r = _Rand(seed)
    n, hk, hv, L = case["slots"], case["hk"], case["hv"], case.get("layers", 1)
    c = (2 * hk + hv) * D
    return dict(params=[_gdn_params(r, hk, hv) for _ in range(L)], mixed=r.n(L, n, c), z=r.n(L, n, hv * D),
                a=r.n(L, n, hv), b=r.n(L, n, hv), conv=r.n(L, n, c, K),
                rec=r.n(L, n, hv, D, D, scale=0.02, dtype=torch.float32))


def _lens(case):
    """The batch's prompt lengths, the same for every seed: shapes belong to the case."""
    g = torch.Generator().manual_seed(case["prompts"] * 10007 + case["hi"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["prompts"],), generator=g).tolist()


def _layer_inputs(case, seed):
    r = _Rand(seed)
    lens = _lens(case)
    hk, hv, n, t = case["hk"], case["hv"], case["prompts"], sum(lens)
    c = (2 * hk + hv) * D
    return dict(_gdn_params(r, hk, hv), lens=lens, mixed=r.n(t, c), z=r.n(t, hv * D), a=r.n(t, hv), b=r.n(t, hv),
                conv=r.n(n, c, K), rec=r.n(n, hv, D, D, scale=0.02, dtype=torch.float32))


def _mlp_inputs(case, seed):
    r = _Rand(seed)
    n, h, m = case["slots"], case["hidden"], case["mlp"]
    return dict(x=r.n(n, h), h=r.n(n, h), gate_up=r.n(2 * m, h, scale=0.02), down=r.n(h, m, scale=0.02),
                norm=r.n(h, scale=0.1))


def _inv_freq(hd, dev):
    rd = hd // 4
    return rd, 1.0 / (10000.0 ** (torch.arange(0, rd, 2, device=dev, dtype=torch.float32) / rd))


def _attn_inputs(case, seed):
    r = _Rand(seed)
    n, nh, kv, hd = case["slots"], case["heads"], case["kv"], case["hd"]
    g = torch.Generator().manual_seed(seed)
    ctx = torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (n,), generator=g)
    t = (case["ctx_hi"] + 16 + 3) // 4 * 4
    return dict(proj=r.n(n, (2 * nh + 2 * kv) * hd), pos=ctx.to(r.dev), qn=r.n(hd, scale=0.1), kn=r.n(hd, scale=0.1),
                kt=r.n(n, kv, hd, t), v=r.n(n, kv, t, hd))


def _config(case):
    return hybrid.HybridConfig(hidden=case["hidden"], layers=case["layers"], mlp=case["mlp"], vocab=case["vocab"])


def _hybrid_weights(case, seed):
    """A checkpoint of the stack: every layer's weights, the slots' states and caches, a step's input."""
    r = _Rand(seed)
    c, n = _config(case), case["slots"]
    g = torch.Generator().manual_seed(seed)
    ctx = torch.randint(case["ctx_lo"], case["ctx_hi"] + 1, (n,), generator=g)
    H, hd, kv, nh = c.hidden, c.attn_head, c.kv_heads, c.attn_heads
    t = (int(ctx.max()) + 8 + 3) // 4 * 4
    layers = []
    for i in range(c.layers):
        w = dict(full=c.is_full(i), in_norm=r.n(H, scale=0.1), post_norm=r.n(H, scale=0.1),
                 gate_up=r.n(2 * c.mlp, H, scale=0.02), down=r.n(H, c.mlp, scale=0.02))
        if w["full"]:
            w.update(qkv=r.n((2 * nh + 2 * kv) * hd, H, scale=0.02), o=r.n(H, nh * hd, scale=0.02),
                     q_norm=r.n(hd, scale=0.1), k_norm=r.n(hd, scale=0.1), kt=r.n(n, kv, hd, t), v=r.n(n, kv, t, hd))
        else:
            w.update(_gdn_params(r, c.gdn_k_heads, c.gdn_v_heads),
                     in_proj=r.n(c.conv_dim + c.gdn_v_heads * D + 2 * c.gdn_v_heads, H, scale=0.02),
                     out=r.n(H, c.gdn_v_heads * D, scale=0.02), conv=r.n(n, c.conv_dim, K),
                     rec=r.n(n, c.gdn_v_heads, D, D, scale=0.02, dtype=torch.float32))
        layers.append(w)
    return dict(cfg=c, ctx=ctx, layers=layers, final_norm=r.n(H, scale=0.1), lm_head=r.n(c.vocab, H, scale=0.02),
                inp=r.n(n, H))


# ---- prepare --------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("rule", "generic"):
        return dict(case=case, x=_rule_inputs(case, seed))
    if kind == "unfused":
        x = _decode_inputs(case, seed)
        return dict(case=case, x=x)
    if kind == "decode":
        # the engine allocates its slot buffers, captures the step once and then serves from the graph
        x = _decode_inputs(case, seed)
        conv, rec = torch.zeros_like(x["conv"]), torch.zeros_like(x["rec"])
        out = torch.zeros(case["layers"], case["slots"], case["hv"] * D, dtype=BF, device=rec.device)

        def step():
            for i, p in enumerate(x["params"]):
                gdn.gdn_decode_core(x["mixed"][i], x["z"][i], x["a"][i], x["b"][i], conv[i], p["cw"], p["A_log"],
                                    p["dt"], p["nw"], rec[i], case["hk"], case["hv"], D, out=out[i])
            return out

        graph = gdn.GDNDecodeGraph(step, device=rec.device)
        conv.copy_(x.pop("conv"))
        rec.copy_(x.pop("rec"))
        return dict(case=case, graph=graph, conv=conv, rec=rec)
    if kind == "layer":
        x = _layer_inputs(case, seed)
        lens = x["lens"]
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        # one sequence table per batch step, handed to every layer of the step
        st = dict(case=case, x=x, table=gdn.Varlen(cu, cu[-1], x["mixed"].device))
        if case["cont"]:
            # a serving batch's slot buffers: the prompts sit in every other row
            n_rows = 2 * len(lens) + 1
            st["conv"] = torch.zeros(n_rows, *x["conv"].shape[1:], dtype=BF, device=x["mixed"].device)
            st["rec"] = torch.zeros(n_rows, *x["rec"].shape[1:], device=x["mixed"].device)
            rows = [2 * i + 1 for i in range(len(lens))]
            st["conv"][rows] = x.pop("conv")
            st["rec"][rows] = x.pop("rec")
            st["rows"] = gdn.Rows(rows, len(lens), n_rows, x["mixed"].device)
        return st
    if kind == "mlp":
        x = _mlp_inputs(case, seed)
        return dict(case=case, x=x["x"], h=x["h"], norm=x["norm"], gate_up=cb.PackedWeight(x["gate_up"]),
                    down=cb.PackedWeight(x["down"]))
    if kind == "attention":
        x = _attn_inputs(case, seed)
        rd, inv = _inv_freq(case["hd"], x["proj"].device)
        return dict(case=case, x=x, rd=rd, inv=inv,
                    work=cb.attn_decode_workspace(case["slots"], case["heads"], case["hd"], x["kt"].shape[-1],
                                                  x["proj"].device))
    # hybrid: the stack with a checkpoint's weights loaded, captured once; the slots are filled after that
    w = _hybrid_weights(case, seed)
    dev = w["inp"].device
    model = hybrid.HybridDecoder(w["cfg"], case["slots"], w["ctx"], 8, dev, seed=1)
    for L, s in zip(model.layers, w["layers"]):
        for name in ("in_proj", "out", "qkv", "o", "gate_up", "down"):
            if name in s:
                setattr(L, name + "_p", cb.PackedWeight(s.pop(name)))
        L.in_norm, L.post_norm = s["in_norm"], s["post_norm"]
        if L.full:
            L.q_norm, L.k_norm = s["q_norm"], s["k_norm"]
        else:
            L.conv_w, L.A_log, L.dt_bias, L.norm_w = s["cw"], s["A_log"], s["dt"], s["nw"]
    model.final_norm = w["final_norm"]
    model.lm_head_p = cb.PackedWeight(w.pop("lm_head"))
    inp = torch.zeros_like(w["inp"])
    graph = hybrid.HybridDecodeGraph(model, inp)
    for i, (L, s) in enumerate(zip(model.layers, w["layers"])):
        if L.full:
            L.kt.copy_(s["kt"])
            L.v.copy_(s["v"])
        else:
            model.slots.conv[i].copy_(s["conv"])
            model.slots.rec[i].copy_(s["rec"])
    return dict(case=case, model=model, graph=graph, inp=inp, x=w["inp"], pos=w["ctx"].to(dev))


# ---- run ------------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("rule", "generic"):
        x = s["x"]
        return gdn.fast_chunk_gated_delta_rule_v2(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=x["s0"],
                                                  output_final_state=True, use_qk_l2norm_in_kernel=True)
    if kind == "decode":
        out = s["graph"].replay()
        return out, s["conv"], s["rec"]
    if kind == "unfused":
        x, p = s["x"], s["x"]["params"][0]
        n, hk, hv = case["slots"], case["hk"], case["hv"]
        m = gdn.causal_conv1d_update(x["mixed"][0].unsqueeze(-1), x["conv"][0], p["cw"], None, "silu").view(n, 1, -1)
        q = m[..., :hk * D].view(n, 1, hk, D)
        k = m[..., hk * D:2 * hk * D].view(n, 1, hk, D)
        v = m[..., 2 * hk * D:].view(n, 1, hv, D)
        beta, g = gdn.gdn_gating(x["a"][0], x["b"][0], p["A_log"], p["dt"])
        o, rec = gdn.recurrent_single_step(q, k, v, g.view(n, 1, hv), beta.view(n, 1, hv), x["rec"][0], True, True)
        y = gdn.gated_rmsnorm(o.reshape(-1, D), x["z"][0].view(-1, D), p["nw"], EPS)
        return y, rec, x["conv"][0]
    if kind == "layer":
        x = s["x"]
        state = dict(slots=s["rows"], conv_slots=s["conv"], rec_slots=s["rec"], continuation=True) if case["cont"] else {}
        return gdn.gdn_prefill_core(x["mixed"], x["z"], x["a"], x["b"], x["cw"], x["A_log"], x["dt"], x["nw"],
                                    case["hk"], case["hv"], D, cu_seqlens=s["table"], **state)
    if kind == "mlp":
        act = cb.swiglu(cb.decode_linear_partial(s["x"], s["gate_up"]))
        return cb.add_rms_norm(s["h"], cb.decode_linear_partial(act, s["down"]), s["norm"], EPS)
    if kind == "attention":
        x = s["x"]
        return cb.gqa_decode_attention(x["proj"], x["pos"], x["qn"], x["kn"], s["inv"], x["kt"], x["v"], case["heads"],
                                       case["kv"], case["hd"], s["rd"], EPS, work=s["work"])
    # a step of the serving loop: the slots' tokens and positions go into the graph's static buffers
    s["inp"].copy_(s["x"])
    s["model"].pos.copy_(s["pos"])
    return s["graph"].replay()


# ---- work -----------------------------------------------------------------------------------------
def _gdn_decode_bytes(n, hk, hv):
    c = (2 * hk + hv) * D
    return 2 * n * hv * D * D * 4 + 2 * n * c * K * 2 + c * K * 2 + n * c * 2 + 2 * n * hv * D * 2 + 2 * n * hv * 2


def work(case):
    kind = case["kind"]
    if kind in ("rule", "generic"):
        dt = DTYPES[case.get("dtype", "bf16")]
        es = torch.empty(0, dtype=dt).element_size()
        dk, dv, tok, hk, hv = case.get("dk", D), case.get("dv", D), case["b"] * case["t"], case["hk"], case["hv"]
        bs = torch.empty(0, dtype=DTYPES[case.get("beta", case.get("dtype", "bf16"))]).element_size()
        st = case["b"] * hv * dk * dv * 4 * (2 if case.get("init", True) else 1)
        return dict(bytes=tok * (2 * hk * dk * es + 2 * hv * dv * es + hv * (4 + bs)) + st, flops=6 * tok * hv * dk * dv)
    if kind in ("decode", "unfused"):
        L = case.get("layers", 1)
        return dict(bytes=L * _gdn_decode_bytes(case["slots"], case["hk"], case["hv"]),
                    flops=L * 6 * case["slots"] * case["hv"] * D * D)
    if kind == "layer":
        hk, hv, n = case["hk"], case["hv"], case["prompts"]
        c, t = (2 * hk + hv) * D, sum(_lens(case))
        st = n * (hv * D * D * 4 + c * K * 2) * (2 if case["cont"] else 1)
        return dict(bytes=t * (2 * c + 4 * hv * D + 4 * hv) + c * K * 2 + st, flops=t * (6 * hv * D * D + 2 * K * c))
    n = case["slots"]
    if kind == "mlp":
        w = 3 * case["hidden"] * case["mlp"]
        return dict(bytes=2 * w + 8 * n * case["hidden"], flops=2 * n * w)
    mean = (case["ctx_lo"] + case["ctx_hi"]) / 2 + 1
    if kind == "attention":
        per = case["kv"] * case["hd"]
        return dict(bytes=n * (mean * per * 4 + (3 * case["heads"] + 2 * case["kv"]) * case["hd"] * 2),
                    flops=n * mean * case["heads"] * case["hd"] * 4)
    c = _config(case)
    total = c.vocab * c.hidden * 2 + n * c.vocab * 2
    flops = 2 * n * c.vocab * c.hidden
    for i in range(c.layers):
        w = 3 * c.hidden * c.mlp
        if c.is_full(i):
            w += c.hidden * c.attn_head * (3 * c.attn_heads + 2 * c.kv_heads)
            total += n * mean * c.kv_heads * c.attn_head * 4
            flops += n * mean * c.attn_heads * c.attn_head * 4
        else:
            w += c.hidden * (c.conv_dim + 2 * c.gdn_v_heads * D + 2 * c.gdn_v_heads)
            total += _gdn_decode_bytes(n, c.gdn_k_heads, c.gdn_v_heads)
            flops += 6 * n * c.gdn_v_heads * D * D
        total += 2 * w
        flops += 2 * n * w
    return dict(bytes=total, flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind == "generic":
        return {"rel": {"fp32": 1e-5, "fp16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
    if kind == "hybrid":
        return {"rel": 3e-2}
    return {"rel": 1e-2}


# ---- 64 bits --------------------------------------------------------------------------------------
def _r(x, dtype=BF):
    """Rounded once to the dtype the path's contract stores, back in 64 bits."""
    return x.to(dtype).double()


def _l2norm64(x):
    dt, x = x.dtype, x.double()
    s = _r(_r(x * x, dt).sum(-1, keepdim=True), dt)
    return _r(x * _r(torch.rsqrt(_r(s + 1e-6, dt)), dt), dt)


def _rule64(q, k, v, g, beta, s0):
    """Token recurrence: q, k [B, T, Hk, dk] (normalised), v [B, T, Hv, dv], g, beta [B, T, Hv], all 64 bits."""
    B, T, Hk, dk = q.shape
    Hv, dv = v.shape[2:]
    ex = lambda x: x.repeat_interleave(Hv // Hk, 2).permute(1, 0, 2, 3).reshape(T, B * Hv, 1, dk)  # noqa: E731
    q, k = ex(q) / math.sqrt(dk), ex(k)
    v = v.permute(1, 0, 2, 3).reshape(T, B * Hv, 1, dv)
    gam = g.permute(1, 0, 2).reshape(T, B * Hv, 1, 1).exp()
    bet = beta.permute(1, 0, 2).reshape(T, B * Hv, 1, 1)
    S = torch.zeros(B * Hv, dk, dv, dtype=torch.float64, device=q.device) if s0 is None \
        else s0.double().reshape(B * Hv, dk, dv).clone()
    out = torch.empty(T, B * Hv, 1, dv, dtype=torch.float64, device=q.device)
    for t in range(T):
        S.mul_(gam[t])
        d = (v[t] - torch.bmm(k[t], S)) * bet[t]
        S.baddbmm_(k[t].transpose(1, 2).contiguous(), d)
        torch.bmm(q[t], S, out=out[t])
    return out.view(T, B, Hv, dv).permute(1, 0, 2, 3), S.view(B, Hv, dk, dv)


def _gated_norm64(o, z, w):
    """bf16 rule output, normalised, weighted, times silu(gate)."""
    o, z = _r(o), z.double()
    x = _r(o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS))
    return _r(w.double() * x) * torch.nn.functional.silu(z)


def _silu64(x):
    return _r(torch.nn.functional.silu(_r(x)))


def _conv64(x, hist, w, decode):
    """x [n, T, C], hist [n, C, K] (the previous K inputs) -> conv + SiLU [n, T, C], the last K inputs.
    At decode the conv is bf16 products summed, so each product is rounded."""
    full = torch.cat([hist.transpose(1, 2).double(), x.double()], 1)
    T = x.shape[1]
    taps = [full[:, j + 1:j + 1 + T] * w[:, j].double() for j in range(K)]
    y = sum(_r(p) if decode else p for p in taps)
    return _silu64(y), full[:, -K:].transpose(1, 2)


def _gates64(a, b, A_log, dt):
    return -A_log.double().exp() * torch.nn.functional.softplus(a.double() + dt.double()), _r(torch.sigmoid(b.double()))


def _gdn64(mixed, z, a, b, conv, rec, p, hk, hv):
    """The decode GDN layer core on [n, 1, ...] inputs."""
    n, T = mixed.shape[:2]
    m, conv = _conv64(mixed, conv, p["cw"], True)
    g, beta = _gates64(a, b, p["A_log"], p["dt"])
    q = _l2norm64(m[..., :hk * D].to(BF).view(n, T, hk, D))
    k = _l2norm64(m[..., hk * D:2 * hk * D].to(BF).view(n, T, hk, D))
    o, rec = _rule64(q, k, m[..., 2 * hk * D:].view(n, T, hv, D), g, beta, rec)
    return _gated_norm64(o, z.reshape(n, T, hv, D), p["nw"]).reshape(n, T, hv * D), conv, rec


def _attn64(proj, pos, qn, kn, inv, rd, kt, vc, nh, kv, hd):
    n = proj.shape[0]
    x = proj.double()
    qg = x[:, :2 * nh * hd].view(n, nh, 2, hd)
    k, v = x[:, 2 * nh * hd:(2 * nh + kv) * hd].view(n, kv, hd), x[:, (2 * nh + kv) * hd:].view(n, kv, hd)
    norm = lambda y, w: _r(y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * (1 + w.double()))  # noqa: E731
    ang = (pos.float()[:, None] * inv).double()[:, None]  # the angle is a 32-bit product, as rotary tables hold it
    c, s = torch.cat([ang.cos()] * 2, -1), torch.cat([ang.sin()] * 2, -1)

    def rope(y):
        a, b = y[..., :rd // 2], y[..., rd // 2:rd]
        return torch.cat([_r(y[..., :rd] * c + torch.cat([-b, a], -1) * s), y[..., rd:]], -1)

    q, k = rope(norm(qg[:, :, 0], qn)), rope(norm(k, kn))
    out = torch.empty(n, nh, hd, dtype=torch.float64, device=x.device)
    for i, p in enumerate(pos.tolist()):
        ks = torch.cat([kt[i, :, :, :p].double(), k[i].unsqueeze(-1)], -1)
        vs = torch.cat([vc[i, :, :p].double(), v[i].unsqueeze(1)], 1)
        sc = torch.matmul(q[i].view(kv, nh // kv, hd), ks) / math.sqrt(hd)
        out[i] = torch.matmul(torch.softmax(sc, -1), vs).view(nh, hd)
    return (_r(out) * _r(torch.sigmoid(qg[:, :, 1]))).reshape(n, nh * hd)


def _mm64(x, w):
    """x [n, K] times a bf16 weight [N, K], in pieces of rows."""
    return torch.cat([torch.matmul(x.double(), p.double().t()) for p in w.split(1 << 15)], -1)


def _add_norm64(h, delta, w):
    h = h.double() if delta is None else _r(h.double() + _r(delta))
    return h, h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * (1 + w.double())


def _mlp64(x, gate_up, down):
    gu = _r(_mm64(x, gate_up))
    m = gu.shape[-1] // 2
    return _mm64(_r(_silu64(gu[:, :m]) * gu[:, m:]), down)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rule", "generic"):
        x = _rule_inputs(case, seed)
        return _rule64(_l2norm64(x["q"]), _l2norm64(x["k"]), x["v"].double(), x["g"].double(), x["beta"].double(), x["s0"])
    if kind in ("decode", "unfused"):
        x = _decode_inputs(case, seed)
        got = [_gdn64(x["mixed"][i].unsqueeze(1), x["z"][i].unsqueeze(1), x["a"][i].unsqueeze(1), x["b"][i].unsqueeze(1),
                      x["conv"][i], x["rec"][i], p, case["hk"], case["hv"]) for i, p in enumerate(x["params"])]
        out, conv, rec = (torch.stack([g[j] for g in got]) for j in range(3))
        if kind == "unfused":
            return out.view(-1, D), rec[0].contiguous(), conv[0]
        return out.squeeze(2), conv, rec
    if kind == "layer":
        x = _layer_inputs(case, seed)
        outs, t0 = [], 0
        n, longest = len(x["lens"]), max(x["lens"])
        p = {name: x[name] for name in ("cw", "A_log", "dt", "nw")}
        # prompts side by side, padded at the end: a padded token neither decays nor writes
        c, hk, hv = x["mixed"].shape[1], case["hk"], case["hv"]
        m = torch.zeros(n, longest, c, dtype=torch.float64, device=x["a"].device)
        g = torch.zeros(n, longest, hv, dtype=torch.float64, device=x["a"].device)
        beta = torch.zeros_like(g)
        convs = []
        for i, L in enumerate(x["lens"]):
            sl = slice(t0, t0 + L)
            hist = x["conv"][i:i + 1] if case["cont"] else torch.zeros_like(x["conv"][:1])
            mi, cs = _conv64(x["mixed"][sl].unsqueeze(0), hist, p["cw"], False)
            m[i, :L] = mi[0]
            convs.append(cs[0])
            g[i, :L], beta[i, :L] = _gates64(x["a"][sl], x["b"][sl], p["A_log"], p["dt"])
            t0 += L
        q = _l2norm64(m[..., :hk * D].to(BF).view(n, longest, hk, D))
        k = _l2norm64(m[..., hk * D:2 * hk * D].to(BF).view(n, longest, hk, D))
        o, rec = _rule64(q, k, m[..., 2 * hk * D:].view(n, longest, hv, D), g, beta,
                         x["rec"] if case["cont"] else None)
        o = torch.cat([o[i, :L] for i, L in enumerate(x["lens"])])
        out = _gated_norm64(o, x["z"].view(-1, hv, D), p["nw"]).reshape(-1, hv * D)
        conv = torch.stack(convs)
        if not case["cont"]:
            return out, conv, rec
        rows = [2 * i + 1 for i in range(n)]
        conv_s = torch.zeros(2 * n + 1, *conv.shape[1:], dtype=torch.float64, device=conv.device)
        rec_s = torch.zeros(2 * n + 1, *rec.shape[1:], dtype=torch.float64, device=conv.device)
        conv_s[rows], rec_s[rows] = conv, rec
        return out, conv_s, rec_s
    if kind == "mlp":
        x = _mlp_inputs(case, seed)
        return _add_norm64(x["h"], _mlp64(x["x"], x["gate_up"], x["down"]), x["norm"])
    if kind == "attention":
        x = _attn_inputs(case, seed)
        rd, inv = _inv_freq(case["hd"], x["proj"].device)
        return _attn64(x["proj"], x["pos"], x["qn"], x["kn"], inv, rd, x["kt"], x["v"], case["heads"], case["kv"], case["hd"])
    w = _hybrid_weights(case, seed)
    c = w["cfg"]
    pos = w["ctx"].to(w["inp"].device)
    rd, inv = _inv_freq(c.attn_head, pos.device)
    h, x = w["inp"], None
    h, x = _add_norm64(h, None, w["layers"][0]["in_norm"])
    for i, s in enumerate(w["layers"]):
        if s["full"]:
            o = _attn64(_r(_mm64(_r(x), s["qkv"])), pos, s["q_norm"], s["k_norm"], inv, rd, s["kt"], s["v"],
                        c.attn_heads, c.kv_heads, c.attn_head)
            mix = _mm64(_r(o), s["o"])
        else:
            pr = _r(_mm64(_r(x), s["in_proj"])).unsqueeze(1)
            C, hv = c.conv_dim, c.gdn_v_heads
            core, _, _ = _gdn64(pr[..., :C], pr[..., C:C + hv * D], pr[..., C + hv * D + hv:],
                                pr[..., C + hv * D:C + hv * D + hv], s["conv"], s["rec"], s, c.gdn_k_heads, hv)
            mix = _mm64(_r(core[:, 0]), s["out"])
        h, x = _add_norm64(h, mix, s["post_norm"])
        last = i + 1 == len(w["layers"])
        h, x = _add_norm64(h, _mlp64(_r(x), s["gate_up"], s["down"]),
                           w["final_norm"] if last else w["layers"][i + 1]["in_norm"])
    return _mm64(_r(x), w["lm_head"])
