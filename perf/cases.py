"""Workloads for timing the MI355X Qwen3.5-0.8B library through its public
entry points (qw.py over the C ABI, engine.py for whole-model calls).

Shapes are the model's: hidden 1024, MLP 3584, 16 Gated-DeltaNet heads of
128 x 128, 8 query / 2 KV heads of 256, vocabulary 248320, 24 layers of which
every fourth is full attention.  Kinds of cases:

  stack    consecutive MLP blocks at decode sizes (qw_mlp_stack)
  block    one period of the decoder (three Gated-DeltaNet layers and one
           full-attention layer, MLPs included) for one new token of each of
           B sequences, captured once and replayed, as a decode loop does
  attn     the gated full-attention core between its projections: decode
           (one token per sequence, the model's six layers in a graph) or
           prefill (T tokens per sequence, one call)
  gdn      the Gated-DeltaNet core between its projections, T prompt tokens
  mlp      a prefill MLP layer: RMSNorm, gate/up, SiLU*mul, down, residual
  head     the tied lm_head with greedy argmax
  model    whole-model prefill of prompts, then the last token's logits
"""
import importlib.util
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _module(name, file):
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(ROOT, "qwen3.5_0.8b_deploy_amd", file))
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        sys.modules[name] = mod
    return sys.modules[name]


qw = _module("qw_perf", "qw.py")
em = _module("qw_perf_engine", "engine.py")

H, I, V, EPS = em.H, em.I, em.V_DEFAULT, 1e-6
NH, KD, VD, CK, CD, LIN_IN = em.LNH, em.KD, em.VD, em.CK, em.CD, em.LIN_IN
FNH, NKV, HD, FULL_IN = em.FNH, em.FNKV, em.HD, em.FULL_IN
ROT, THETA = 64, 1.0e7
LAYERS = 24
STD = 0.64  # of a projection's output: sqrt(1024) * 0.02

ACT = {"bf16": torch.bfloat16, "int8": torch.float16, "f32": torch.float32}
FMT = {"bf16": qw.WFMT_BF16, "int8": qw.WFMT_INT8, "f32": qw.WFMT_F32}
WBYTES = {"bf16": 2, "int8": 1, "f32": 4}


def listed():
    return [
        # the smallest call of a decode loop: one token through the model's 24 MLPs
        {"name": "stack-bf16-1", "kind": "stack", "fmt": "bf16", "tokens": 1, "layers": 24},
        # INT8 serving of a medium batch, 24 MLPs of FP16 activations
        {"name": "stack-int8-40", "kind": "stack", "fmt": "int8", "tokens": 40, "layers": 24},
        # interactive decode of one sequence: launches and latency
        {"name": "block-1", "kind": "block", "fmt": "bf16", "batch": 1, "context": 1000},
        # batched decode, ragged contexts up to 4096 tokens
        {"name": "block-32", "kind": "block", "fmt": "bf16", "batch": 32, "context": 4096},
        # long-context decode of one sequence: the six layers' KV caches are the traffic
        {"name": "attn-decode-32k", "kind": "attn", "kv": "int8", "batch": 1, "tokens": 1, "context": 32000},
        # a long prompt from position 0
        {"name": "attn-prefill-4096", "kind": "attn", "kv": "int8", "batch": 1, "tokens": 4096, "context": 0},
        # the exact FP32 cache, two prompts continued in chunks from ragged positions
        {"name": "attn-chunk-f32", "kind": "attn", "kv": "f32", "batch": 2, "tokens": 600, "context": 1000},
        # the recurrent layers' share of a usual prompt
        {"name": "gdn-1000", "kind": "gdn", "batch": 1, "tokens": 1000},
        # an INT8 prompt of ordinary length
        {"name": "mlp-int8-1000", "kind": "mlp", "fmt": "int8", "tokens": 1000},
        # a large batch of prompts
        {"name": "mlp-bf16-16384", "kind": "mlp", "fmt": "bf16", "tokens": 16384},
        # the head of a batched decode step
        {"name": "head-bf16-48", "kind": "head", "fmt": "bf16", "tokens": 48},
        # time to the first token of one prompt
        {"name": "model-777", "kind": "model", "batch": 1, "tokens": 777},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["stack", "block", "attn-decode", "attn-prefill", "attn-prefill", "gdn", "gdn", "mlp", "mlp",
                       "head", "model"])
    if kind == "stack":
        return {"kind": kind, "fmt": rng.choice(["bf16", "int8"]), "tokens": _log(rng, 1, 256),
                "layers": rng.choice([6, 12, 24])}
    if kind == "block":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "fmt": "bf16", "batch": batch, "context": _log(rng, 64, min(32768, 262144 // batch))}
    if kind == "attn-decode":
        batch = _log(rng, 1, 64)
        return {"kind": "attn", "kv": rng.choice(["int8", "int8", "f32"]), "batch": batch, "tokens": 1,
                "context": _log(rng, 64, min(32768, 131072 // batch))}
    if kind == "attn-prefill":
        kv = rng.choice(["int8", "int8", "f32"])
        batch = rng.choice([1, 1, 2, 3, 8])
        most = (4096 if kv == "int8" else 1024) // batch
        return {"kind": "attn", "kv": kv, "batch": batch, "tokens": _log(rng, 16, most),
                "context": rng.choice([0, 0, _log(rng, 64, 4096)])}
    if kind == "gdn":
        batch = rng.choice([1, 1, 2, 5, 16])
        return {"kind": kind, "batch": batch, "tokens": _log(rng, 24, 8192 // batch)}
    if kind == "mlp":
        fmt = rng.choice(["bf16", "bf16", "int8", "int8", "f32"])
        return {"kind": kind, "fmt": fmt, "tokens": _log(rng, 24, 512 if fmt == "f32" else 16384)}
    if kind == "head":
        return {"kind": kind, "fmt": rng.choice(["bf16", "int8"]), "tokens": _log(rng, 1, 256)}
    batch = rng.choice([1, 1, 2])
    return {"kind": kind, "batch": batch, "tokens": _log(rng, 32, 777 // batch)}


# --------------------------------------------------------------------------
# inputs, from the seed alone


class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        x = torch.randn(*shape, generator=self.g, device="cuda", dtype=dtype)
        return x.mul_(std)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)

    def integers(self, lo, hi, *shape, dtype=torch.int32):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)

    def matrix(self, n, k, fmt):
        """W[n][k] of std 0.02: (tensor, None), or (INT8 codes, row scales)."""
        w = self.normal(n, k, std=0.02, dtype=torch.float32 if fmt == "f32" else torch.bfloat16)
        if fmt != "int8":
            return w, None
        s = w.abs().amax(dim=1).float() / 127.0
        return torch.round(w.float() / s[:, None]).clamp_(-127, 127).to(torch.int8), s

    def codes(self, *shape):
        """INT8 cache codes of normal values quantized by their head's maximum."""
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float16).mul_(42.0).round_().clamp_(
            -127, 127).to(torch.int8)


def _mlp_inputs(r, fmt):
    return {"gate": r.matrix(I, H, fmt), "up": r.matrix(I, H, fmt), "down": r.matrix(H, I, fmt),
            "post_norm": r.normal(H, std=0.1)}


def _gdn_inputs(r, batch):
    return {"conv": r.normal(CD, CK, std=0.5), "A_log": r.normal(NH, std=0.5), "dt_bias": r.normal(NH, std=0.5),
            "norm_w": 1.0 + r.normal(VD, std=0.1), "cs": r.normal(batch, CD, CK - 1, std=STD),
            "rs": r.normal(batch, NH, KD * VD, std=0.1)}


def _attn_inputs(r, batch, capacity, kv):
    shape = (batch, capacity, NKV, HD)
    if kv == "int8":
        cache = (r.codes(*shape), r.codes(*shape), r.uniform(*shape[:3], lo=0.02, hi=0.028),
                 r.uniform(*shape[:3], lo=0.012, hi=0.018))
    else:
        cache = (r.normal(*shape), r.normal(*shape, std=STD), torch.zeros(shape[:3], device="cuda"),
                 torch.zeros(shape[:3], device="cuda"))
    return {"q_norm": r.normal(HD, std=0.1), "k_norm": r.normal(HD, std=0.1), "cache": cache}


def _positions(r, batch, context):
    """Ragged starts: one sequence at the full context, the others from an eighth of it."""
    pos = r.integers(context // 8, context + 1, batch)
    pos[0] = context
    return pos


def _inputs(case, seed):
    r = _Rand(seed)
    kind = case["kind"]
    if kind == "stack":
        return {"mlps": [_mlp_inputs(r, case["fmt"]) for _ in range(case["layers"])],
                "x": r.normal(case["tokens"], H).to(ACT[case["fmt"]])}
    if kind == "mlp":
        return {"mlp": _mlp_inputs(r, case["fmt"]), "x": r.normal(case["tokens"], H)}
    if kind == "head":
        return {"E": r.matrix(V, H, case["fmt"]), "h": r.normal(case["tokens"], H).to(ACT[case["fmt"]])}
    if kind == "gdn":
        return {"core": _gdn_inputs(r, case["batch"]),
                "rows": r.normal(case["batch"] * case["tokens"], LIN_IN, std=STD)}
    if kind == "attn":
        B, T = case["batch"], case["tokens"]
        n = LAYERS // 4 if T == 1 else 1
        return {"cores": [_attn_inputs(r, B, case["context"] + T, case["kv"]) for _ in range(n)],
                "pos": _positions(r, B, case["context"]),
                "rows": [r.normal(B * T, FULL_IN, std=STD) for _ in range(n)]}
    if kind == "block":
        B, fmt, layers = case["batch"], case["fmt"], []
        for i in range(4):
            L = {"in_norm": r.normal(H, std=0.1), "mlp": _mlp_inputs(r, fmt), "out": r.matrix(H, NH * VD, fmt)}
            if em.is_linear_layer(i):
                L["in"] = [r.matrix(n, H, fmt) for n in (CD, NH * VD, NH, NH)]
                L["core"] = _gdn_inputs(r, B)
            else:
                L["in"] = [r.matrix(n, H, fmt) for n in (2 * FNH * HD, NKV * HD, NKV * HD)]
                L["core"] = _attn_inputs(r, B, case["context"] + 1, "int8")
            layers.append(L)
        return {"layers": layers, "table": r.normal(4096, H, dtype=torch.bfloat16), "ids": r.integers(0, 4096, B),
                "pos": _positions(r, B, case["context"])}
    layers = []  # the whole model, as the engine takes it
    for i in range(LAYERS):
        m = lambda n, k, std=0.02: r.normal(n, k, std=std, dtype=torch.bfloat16).float()  # noqa: E731
        res = 0.02 / math.sqrt(2 * LAYERS)  # the projections onto the residual stream, scaled with depth
        L = {"in_norm": r.normal(H, std=0.1), "post_norm": r.normal(H, std=0.1), "gate": m(I, H), "up": m(I, H),
             "down": m(H, I, res)}
        if em.is_linear_layer(i):
            L.update(qkv=m(CD, H), a=m(NH, H), b=m(NH, H), z=m(NH * VD, H), conv=r.normal(CD, CK, std=0.5),
                     out=m(H, NH * VD, res), A_log=r.normal(NH, std=0.5), dt_bias=r.normal(NH, std=0.5),
                     norm_w=1.0 + r.normal(VD, std=0.1))
        else:
            L.update(q=m(2 * FNH * HD, H), k=m(NKV * HD, H), v=m(NKV * HD, H), q_norm=r.normal(HD, std=0.1),
                     k_norm=r.normal(HD, std=0.1), o=m(H, FNH * HD, res))
        layers.append(L)
    return {"layers": layers, "final_norm": r.normal(H, std=0.1),
            # large against what a layer adds, as in a trained model: otherwise 16-bit
            # rounding differences of the first layers grow tenfold on the way up
            "embed": r.normal(V, H, std=0.25, dtype=torch.bfloat16),
            "ids": r.integers(0, V, case["batch"], case["tokens"])}


# --------------------------------------------------------------------------
# what a program holds before the call


def _pack_mlp(ctx, m, fmt):
    (g, gs), (u, us), (d, ds) = m["gate"], m["up"], m["down"]
    return qw.Weight.pack_glu_device(ctx, g, u, FMT[fmt], gs, us), qw.Weight.pack_device(ctx, d, FMT[fmt], scales=ds)


def _gdn_core(ctx, c, rows, out, tokens):
    z = CD + NH * VD
    args = (ctx, c["conv"], c["A_log"], c["dt_bias"], c["norm_w"], rows[:, :CD], rows[:, CD:z], rows[:, z:z + NH],
            rows[:, z + NH:], c["cs"], c["rs"], out, NH)
    if tokens == 1:
        qw.gdn_decode(*args)
    else:
        qw.gdn_prefill(*args, tokens)


def _attn_core(ctx, c, pos, rows, out, tokens):
    q = 2 * FNH * HD
    qw.attn_forward(ctx, c["q_norm"], c["k_norm"], c["cache"], pos, rows, rows[:, HD:], rows[:, q:],
                    rows[:, q + NKV * HD:], out, tokens=tokens, q_head_stride=2 * HD, max_len=c["cache"][0].shape[1])


def _decode_block(s):
    """The engine's decode step over four layers, on the FP32 residual stream."""
    ctx, x, xh, core, pos = s["ctx"], s["x"], s["xh"], s["out"], s["pos"]
    many = x.shape[0] > em.NORM_FIRST_MIN_BATCH  # the engine's own rule
    qw.embedding_gather(ctx, s["table"], s["ids"], x)
    for L in s["layers"]:
        row = s["row_lin"] if "cs" in L["core"] else s["row_full"]
        if many:
            qw.rmsnorm(ctx, x, L["in_norm"], xh)
            qw.linear(ctx, L["w_in"], xh, row)
        else:
            qw.linear(ctx, L["w_in"], x, row, gamma=L["in_norm"])
        if "cs" in L["core"]:
            _gdn_core(ctx, L["core"], row, core, 1)
        else:
            _attn_core(ctx, L["core"], pos, row, core, 1)
        if many:
            qw.linear(ctx, L["w_out"], core, x, residual=x)
            qw.rmsnorm(ctx, x, L["post_norm"], xh)
            qw.mlp_fused(ctx, L["gu"], L["dn"], xh, x, residual=x)
        else:
            qw.layer_tail(ctx, L["w_out"], core, L["gu"], L["dn"], x, gamma=L["post_norm"])


def _capture(ctx, body):
    """Capture body's calls, as a decode loop does before its first token."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        g = qw.Graph(ctx, stream)
        with g:
            body()
    return g


def prepare(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    rows = case.get("batch", 1) * case.get("tokens", 1)
    ctx = qw.Context(0, qw.lib().qw_workspace_query(rows, LIN_IN, 4096) if rows > 4096 else 0)
    s = {"case": case, "ctx": ctx}
    if kind == "stack":
        packed = [_pack_mlp(ctx, m, case["fmt"]) for m in inp["mlps"]]
        s.update(gu=[p[0] for p in packed], dn=[p[1] for p in packed], gammas=[m["post_norm"] for m in inp["mlps"]],
                 x=inp["x"], y=torch.empty_like(inp["x"]))
    elif kind == "mlp":
        s["gu"], s["dn"] = _pack_mlp(ctx, inp["mlp"], case["fmt"])
        s.update(post_norm=inp["mlp"]["post_norm"], x=inp["x"], xn=torch.empty_like(inp["x"], dtype=ACT[case["fmt"]]),
                 y=torch.empty_like(inp["x"]))
    elif kind == "head":
        s.update(E=qw.Weight.pack_device(ctx, inp["E"][0], FMT[case["fmt"]], scales=inp["E"][1]), h=inp["h"],
                 ids=torch.empty(rows, dtype=torch.int32, device="cuda"), top=torch.empty(rows, device="cuda"))
    elif kind == "gdn":
        s.update(inp, out=torch.empty(rows, NH * VD, device="cuda", dtype=torch.bfloat16))
    elif kind == "attn":
        dt = torch.bfloat16 if case["kv"] == "int8" else torch.float32
        s.update(inp, outs=[torch.empty(rows, FNH * HD, device="cuda", dtype=dt) for _ in inp["cores"]])
        if case["tokens"] == 1:
            s["graph"] = _capture(ctx, lambda: [_attn_core(ctx, c, s["pos"], r, o, 1)
                                                for c, r, o in zip(s["cores"], s["rows"], s["outs"])])
    elif kind == "block":
        s.update(layers=[], table=inp["table"], ids=inp["ids"], pos=inp["pos"], x=torch.empty(rows, H, device="cuda"),
                 xh=torch.empty(rows, H, device="cuda", dtype=torch.bfloat16),
                 row_lin=torch.empty(rows, LIN_IN, device="cuda"), row_full=torch.empty(rows, FULL_IN, device="cuda"),
                 out=torch.empty(rows, NH * VD, device="cuda", dtype=torch.bfloat16))
        for L in inp["layers"]:
            gu, dn = _pack_mlp(ctx, L["mlp"], case["fmt"])
            s["layers"].append({"in_norm": L["in_norm"], "post_norm": L["mlp"]["post_norm"], "core": L["core"],
                                "w_in": qw.Weight.pack_concat_device(ctx, [w for w, _ in L["in"]], FMT[case["fmt"]]),
                                "w_out": qw.Weight.pack_device(ctx, L["out"][0], FMT[case["fmt"]]), "gu": gu, "dn": dn})
        s["graph"] = _capture(ctx, lambda: _decode_block(s))
    else:
        s.update(ids=inp["ids"], logits=torch.empty(case["batch"], V, device="cuda"),
                 eng=em.DecodeEngine(qw, ctx, inp["layers"], inp["final_norm"], inp["embed"], case["batch"],
                                     case["tokens"] + 64))
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "stack":
        qw.mlp_stack(ctx, s["gu"], s["dn"], s["x"], s["y"], gammas=s["gammas"])
        return s["y"]
    if kind == "mlp":
        qw.rmsnorm(ctx, s["x"], s["post_norm"], s["xn"])
        qw.mlp_fused(ctx, s["gu"], s["dn"], s["xn"], s["y"], residual=s["x"])
        return s["y"]
    if kind == "head":
        qw.lmhead_argmax(ctx, s["E"], s["h"], s["ids"], s["top"])
        return s["ids"], s["top"]
    if kind == "gdn":
        _gdn_core(ctx, s["core"], s["rows"], s["out"], case["tokens"])
        return s["out"], s["core"]["cs"], s["core"]["rs"]
    if kind == "attn":
        if case["tokens"] == 1:
            s["graph"].launch(torch.cuda.current_stream())
        else:
            _attn_core(ctx, s["cores"][0], s["pos"], s["rows"][0], s["outs"][0], case["tokens"])
        return s["outs"], [c["cache"] for c in s["cores"]]
    if kind == "block":
        s["graph"].launch(torch.cuda.current_stream())
        cores = [L["core"] for L in s["layers"]]
        return s["x"], [(c["cs"], c["rs"]) if "cs" in c else c["cache"][2:] for c in cores]
    eng = s["eng"]
    eng.reset([0] * case["batch"])
    eng.prefill(s["ids"], check=False)
    qw.linear(ctx, eng.E, eng.xn, s["logits"])
    return s["logits"], [(P["cs"], P["rs"]) if P["linear"] else P["cache"][2:] for P in eng.layers]


# --------------------------------------------------------------------------
# what a pass cannot do without


def _attn_work(B, T, ctx_sum, kv):
    """ctx_sum: keys that the first tokens of the sequences find, over the sequences."""
    code = (HD + 4) if kv == "int8" else 4 * HD
    keys = ctx_sum + B * T
    out = 2 if kv == "int8" else 4
    pairs = T * ctx_sum + B * T * (T + 1) / 2
    return (2 * NKV * keys * code + B * T * (FULL_IN * 4 + 2 * NKV * code + FNH * HD * out), 4 * FNH * HD * pairs)


def _gdn_work(B, T):
    state = B * (NH * KD * VD + CD * (CK - 1)) * 4
    return 2 * state + B * T * (LIN_IN * 4 + NH * VD * 2), B * T * NH * (6 * KD * VD + 3 * 2 * CK * KD)


def _mlp_work(M, fmt, act):
    return 3 * H * I * WBYTES[fmt] + M * H * 2 * act, 6 * M * H * I


def work(case):
    kind = case["kind"]
    B, T = case.get("batch", 1), case.get("tokens", 1)
    mean = B * case.get("context", 0) * 9 / 16  # _positions: a uniform eighth to all
    if kind == "stack":
        b, f = _mlp_work(T, case["fmt"], 2)
        return {"bytes": case["layers"] * (b - T * H * 4) + T * H * 4, "flops": case["layers"] * f}
    if kind == "mlp":
        b, f = _mlp_work(T, case["fmt"], 4)
        return {"bytes": b, "flops": f}
    if kind == "head":
        return {"bytes": V * H * WBYTES[case["fmt"]] + T * H * 2, "flops": 2 * T * V * H}
    if kind == "gdn":
        b, f = _gdn_work(B, T)
        return {"bytes": b, "flops": f}
    if kind == "attn":
        b, f = _attn_work(B, T, mean if B > 1 else case["context"], case["kv"])
        n = LAYERS // 4 if T == 1 else 1
        return {"bytes": n * b, "flops": n * f}
    proj = (LIN_IN + NH * VD) * H, (FULL_IN + FNH * HD) * H
    if kind == "block":
        periods, ctx_sum, head = 1, mean if B > 1 else case["context"], 0
    else:
        periods, ctx_sum, head = LAYERS // 4, 0, V * H
    weights = 3 * proj[0] + proj[1] + 4 * 3 * H * I
    state = 3 * 2 * B * (NH * KD * VD + CD * (CK - 1)) * 4
    kv = 2 * NKV * (ctx_sum + B * T) * (HD + 4)
    _, fg = _gdn_work(B, T)
    _, fa = _attn_work(B, T, ctx_sum, "int8")
    return {"bytes": periods * (2 * weights + state + kv) + 2 * head + B * T * H * 4,
            "flops": periods * (2 * B * T * weights + 3 * fg + fa) + 2 * B * head}


def tolerance(case):
    """About four times the largest difference seen between two orders of
    summation of the same path (other token groups, key splits, chunk lengths,
    routes); where the route has no other order, about four times its distance
    from the 64-bit result."""
    kind = case["kind"]
    if kind == "stack":  # 16-bit roundings of the hidden state after every block
        return {"rel": 3e-2, "max": 0.12} if case["fmt"] == "bf16" else {"rel": 8e-3, "max": 0.06}
    if kind == "block":
        return {"rel": 4e-3, "max": 0.06}
    if kind == "model":  # 16-bit roundings that travel through 24 layers
        return {"rel": 2.6e-2, "max": 0.5}
    if kind == "mlp":
        return {"rel": {"f32": 4e-6, "int8": 4e-4, "bf16": 3e-3}[case["fmt"]]}
    if kind == "head":
        return {"rel": 1e-6, "differ": 0.0}
    if kind == "gdn":
        return {"rel": 1e-4, "max": 0.03}
    if case["kv"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 4e-3, "max": 0.03, "differ": 1e-5}


# --------------------------------------------------------------------------
# the same in 64 bits


def _w64(w):
    q, s = w
    return q.double() if s is None else q.double() * s.double()[:, None]


def _norm64(x, gamma):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + gamma.double())


def _silu64(x):
    return x * torch.sigmoid(x)


def _mlp64(m, x):
    n = _norm64(x, m["post_norm"])
    return x + (_silu64(n @ _w64(m["gate"]).T) * (n @ _w64(m["up"]).T)) @ _w64(m["down"]).T


def _gdn64(c, rows, B, T):
    """(out, conv state, recurrent state) of T tokens of each of B sequences."""
    rows = rows.double().view(B, T, -1)
    raw, z = rows[..., :CD], rows[..., CD:CD + NH * VD].reshape(B, T, NH, VD)
    a, b = rows[..., CD + NH * VD:CD + NH * VD + NH], rows[..., CD + NH * VD + NH:LIN_IN]
    cs, S = c["cs"].double(), c["rs"].double().view(B, NH, KD, VD).clone()
    hist = torch.cat([cs.flip(2).transpose(1, 2), raw], dim=1)  # oldest first
    w = c["conv"].double()
    mixed = raw * w[:, CK - 1]
    for j in range(CK - 1):  # state j is the input j + 1 tokens ago
        mixed = mixed + hist[:, CK - 2 - j:CK - 2 - j + T] * w[:, j]
    mixed = _silu64(mixed)
    q, k, v = (t.view(B, T, NH, KD) for t in mixed.split(NH * KD, dim=2))
    q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + EPS) / math.sqrt(KD)
    k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + EPS)
    beta = torch.sigmoid(b)
    decay = torch.exp(-torch.exp(c["A_log"].double()) * torch.nn.functional.softplus(a + c["dt_bias"].double()))
    out = torch.empty(B, T, NH, VD, device=rows.device, dtype=torch.float64)
    for t in range(T):
        S.mul_(decay[:, t, :, None, None])
        d = (v[:, t] - (S * k[:, t, :, :, None]).sum(2)) * beta[:, t, :, None]
        S.add_(k[:, t, :, :, None] * d[:, :, None, :])
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    out = out / torch.sqrt(out.square().mean(-1, keepdim=True) + EPS) * c["norm_w"].double() * _silu64(z)
    cs = hist[:, -(CK - 1):].flip(1).transpose(1, 2).contiguous()
    return out.reshape(B * T, NH * VD), cs, S.view(B, NH, KD * VD)


def _rope64(x, pos):
    ang = pos.double()[:, None] / THETA ** (torch.arange(0, ROT, 2, device=x.device).double() / ROT)
    co, si = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    x0, x1 = x[..., 0:ROT:2].clone(), x[..., 1:ROT:2].clone()
    x[..., 0:ROT:2], x[..., 1:ROT:2] = x0 * co - x1 * si, x0 * si + x1 * co
    return x


def _attn64(c, pos, rows, B, T):
    """(out, cache after the call) of T tokens of each of B sequences."""
    kc, vc, ks, vs = c["cache"]
    int8 = kc.dtype == torch.int8
    rows = rows.double().view(B, T, -1)
    nq = 2 * FNH * HD
    qg = rows[..., :nq].reshape(B, T, FNH, 2, HD)
    new_k, new_v = (rows[..., nq + i * NKV * HD:nq + (i + 1) * NKV * HD].reshape(B, T, NKV, HD) for i in (0, 1))
    kc, vc, ks, vs = kc.clone(), vc.clone(), ks.double(), vs.double()
    out = torch.empty(B, T, FNH, HD, device=rows.device, dtype=torch.float64)
    for b in range(B):
        p0 = int(pos[b])
        at = torch.arange(p0, p0 + T, device=rows.device)
        q = _rope64(_norm64(qg[b, :, :, 0], c["q_norm"]), at)
        k = _rope64(_norm64(new_k[b], c["k_norm"]), at)
        for dst, sc, x in ((kc, ks, k), (vc, vs, new_v[b])):
            if int8:
                m = x.abs().amax(-1) / 127.0
                m = torch.where(m > 1e-8, m, torch.ones_like(m))
                sc[b, p0:p0 + T] = m
                y = x / m[..., None]
                dst[b, p0:p0 + T] = (torch.sign(y) * torch.floor(y.abs() + 0.5)).clamp(-127, 127).to(torch.int8)
            else:
                dst[b, p0:p0 + T] = x.float()
        K, Vv = kc[b, :p0 + T].double(), vc[b, :p0 + T].double()
        if int8:
            K, Vv = K * ks[b, :p0 + T, :, None], Vv * vs[b, :p0 + T, :, None]
        mask = torch.arange(p0 + T, device=rows.device)[None, :] > at[:, None]
        for h in range(FNH):
            g = h // (FNH // NKV)
            sc = (q[:, h] @ K[:, g].T / math.sqrt(HD)).masked_fill_(mask, -math.inf)
            out[b, :, h] = torch.softmax(sc, -1) @ Vv[:, g]
    out = out * torch.sigmoid(qg[:, :, :, 1])
    return out.reshape(B * T, FNH * HD), ([kc, vc] if int8 else [kc.double(), vc.double()]) + [ks, vs]


def _layers64(layers, x, pos, B, T):
    states = []
    for L in layers:
        rows = _norm64(x, L["in_norm"]) @ torch.cat([_w64(w) for w in L["in"]]).T
        if "cs" in L["core"]:
            y, cs, rs = _gdn64(L["core"], rows, B, T)
            states.append((cs, rs))
        else:
            y, cache = _attn64(L["core"], pos, rows, B, T)
            states.append(cache[2:])
        x = _mlp64(L["mlp"], x + y @ _w64(L["out"]).T)
    return x, states


def exact(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    B, T = case.get("batch", 1), case.get("tokens", 1)
    if kind == "stack":
        x = inp["x"].double()
        for m in inp["mlps"]:
            x = _mlp64(m, x)
        return x
    if kind == "mlp":
        return _mlp64(inp["mlp"], inp["x"].double())
    if kind == "head":
        w, h = _w64(inp["E"]), inp["h"].double()
        best = [(h[i:i + 32] @ w.T).max(dim=1) for i in range(0, T, 32)]
        return torch.cat([m.indices for m in best]).int(), torch.cat([m.values for m in best])
    if kind == "gdn":
        return _gdn64(inp["core"], inp["rows"], B, T)
    if kind == "attn":
        done = [_attn64(c, inp["pos"], r, B, T) for c, r in zip(inp["cores"], inp["rows"])]
        codes = case["kv"] == "int8"  # bytes that follow from 32-bit roundings have no such value
        return [o for o, _ in done], [(None, None, *c[2:]) if codes else tuple(c) for _, c in done]
    if kind == "block":
        return _layers64(inp["layers"], inp["table"].double()[inp["ids"].long()], inp["pos"], B, 1)
    layers = []
    for i, L in enumerate(inp["layers"]):
        plain = lambda *names: [(L[n], None) for n in names]  # noqa: E731
        mlp = {"gate": (L["gate"], None), "up": (L["up"], None), "down": (L["down"], None), "post_norm": L["post_norm"]}
        if em.is_linear_layer(i):
            core = {n: L[n] for n in ("conv", "A_log", "dt_bias", "norm_w")}
            core.update(cs=torch.zeros(B, CD, CK - 1, device="cuda"), rs=torch.zeros(B, NH, KD * VD, device="cuda"))
            ins, out = plain("qkv", "z", "a", "b"), (L["out"], None)
        else:
            core = {"q_norm": L["q_norm"], "k_norm": L["k_norm"], "cache": qw.kv_cache(B, T + 64, NKV, HD)}
            ins, out = plain("q", "k", "v"), (L["o"], None)
        layers.append({"in_norm": L["in_norm"], "in": ins, "core": core, "out": out, "mlp": mlp})
    pos = torch.zeros(B, dtype=torch.int32, device="cuda")
    x, states = _layers64(layers, inp["embed"].double()[inp["ids"].long().reshape(-1)], pos, B, T)
    last = _norm64(x.view(B, T, H)[:, -1], inp["final_norm"])
    return last @ inp["embed"].double().T, states
