"""The calls whose speed matters to a user of this framework, with their inputs, their exact results and how far a
correct implementation may be from them.

Ten kinds of call, each through a public entry point: the single-stream stage (``FastVerifyStage.decode`` and
``tree_decode``), the ragged stage step (``RaggedStage.forward``), the two MoE blocks (MXFP4 through ``ops``, FP8
through ``Fp8MoeStage``), attention over decode / verify rows and over a prefill chunk, the projections, the lm_head
and the sampler.  Shapes are the framework's own: GPT-OSS-120B layers (``GptOssShape``) and the DeepSeek-V3-shaped
FP8 layer (``DsV3Shape``); a vocabulary of 201,088 tokens.

Weights, KV and activations are random: E2M1 codes uniform, E8M0 scale bytes 119..123 (110..114 in the down
projections, so that a block's output stays below its residual, as a trained one's does), dense weights N(0, 0.02), KV
and hidden rows N(0, 1) in bf16.  Every tensor comes from the case's seed alone."""
import math
import random

import torch

from flyai_amd import ops
from flyai_amd.rope import YarnRotary
from flyai_amd.runtime import FastVerifyStage, Fp8MoeStage, KVWorkspace, RaggedStage
from flyai_amd.stage_parts import FinalNorm
from flyai_amd.weights import DsV3Shape, Fp8MoeLayerWeights, GptOssShape, LayerWeights

DEV = "cuda"
BF16, F64 = torch.bfloat16, torch.float64
SH = GptOssShape()
DS = DsV3Shape()
VOCAB = 201088
LAYERS = 4            # of a stage case: sliding, full, sliding, full
LINEAR_LAYERS = 4     # of a projection case: together with the other states', more than the caches hold
HQ, HKV, D = SH.n_q_heads, SH.n_kv_heads, SH.head_dim
NQ, NKV = HQ * D, HKV * D
FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


# ---- the cases ----------------------------------------------------------------------------------------

def listed():
    return [
        # one user, one token: the interactive decode step, where launches and latency count
        {"name": "stream_1_token", "kind": "stream", "tokens": 1, "kv": 1500},
        # speculative decoding of one user: three drafted chains of six tokens, verified as a tree
        {"name": "tree_18_nodes", "kind": "tree", "width": 3, "depth": 6, "kv": 3001},
        # continuous batching: 24 decode rows and 8 four-token verify rows (the benchmark's batch)
        {"name": "batch_32_decode", "kind": "batch", "decode": 24, "verify": 8, "chunk": 0, "prior": 0, "kv_hi": 8192},
        # a prompt's 2048-token chunk beside 48 decode rows (the benchmark's prefill batch)
        {"name": "batch_chunk_2048", "kind": "batch", "decode": 48, "verify": 0, "chunk": 2048, "prior": 4096, "kv_hi": 8192},
        # one MoE block for a few streams (the benchmark's small block)
        {"name": "moe_12_tokens", "kind": "moe", "tokens": 12, "hot": False},
        # one MoE block for a short prompt chunk beside decode rows: about ten rows an expert
        {"name": "moe_333_tokens", "kind": "moe", "tokens": 333, "hot": False},
        # one FP8 MoE layer over 64 ragged streams (the benchmark's FP8 batch)
        {"name": "fp8_moe_155_tokens", "kind": "fp8", "tokens": 155},
        # decode attention of a full layer, long contexts, verify rows among them
        {"name": "attn_16_long", "kind": "attn", "seqs": 16, "verify": 5, "kv_hi": 32768, "window": 0},
        # prefill attention of a full layer: a short prompt's chunk that is no multiple of the tiles
        {"name": "prefill_attn_1000", "kind": "prefill", "chunk": 1000, "prior": 3000, "window": 0},
        # the projections of a layer at a batch between decode and prefill
        {"name": "linear_137_rows", "kind": "linear", "rows": 137},
        # the tail of a decode step: final norm, logits and greedy token of 24 streams
        {"name": "head_24_rows", "kind": "head", "rows": 24},
        # sampled decoding: nucleus sampling of 8 streams, each with a drafted token to check
        {"name": "sample_8_rows", "kind": "sample", "rows": 8, "temp": 0.8, "top_k": 0, "top_p": 0.95},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("stream", "tree", "batch", "batch", "moe", "moe", "fp8", "attn", "prefill", "linear", "head", "sample"))
    if kind == "stream":
        return {"kind": kind, "tokens": rng.randint(1, 8), "kv": _log_int(rng, 16, 8000)}
    if kind == "tree":
        return {"kind": kind, "width": rng.randint(1, 4), "depth": rng.randint(2, 8), "kv": _log_int(rng, 64, 8000)}
    if kind == "batch":
        chunk = rng.choice((0, _log_int(rng, 33, 2000)))
        return {"kind": kind, "decode": _log_int(rng, 1, 48), "verify": rng.randint(0, 8), "chunk": chunk,
                "prior": rng.randint(0, 4096) if chunk else 0, "kv_hi": _log_int(rng, 512, 8192)}
    if kind == "moe":
        return {"kind": kind, "tokens": _log_int(rng, 1, 2100), "hot": rng.random() < 0.3}
    if kind == "fp8":
        return {"kind": kind, "tokens": _log_int(rng, 1, 400)}
    if kind == "attn":
        return {"kind": kind, "seqs": _log_int(rng, 1, 96), "verify": rng.randint(1, 8),
                "kv_hi": _log_int(rng, 1000, 32768), "window": rng.choice((0, 0, SH.window))}
    if kind == "prefill":
        return {"kind": kind, "chunk": _log_int(rng, 32, 2048), "prior": rng.randint(0, 6000),
                "window": rng.choice((0, 0, SH.window))}
    if kind == "linear":
        return {"kind": kind, "rows": _log_int(rng, 1, 2100)}
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 1, 64)}
    return {"kind": kind, "rows": _log_int(rng, 1, 64), "temp": round(rng.uniform(0.5, 1.2), 2),
            "top_k": rng.choice((0, 0, 50, 200)), "top_p": rng.choice((1.0, 0.9, 0.95))}


# ---- inputs -------------------------------------------------------------------------------------------

def _gen(seed, *salt):
    h = int(seed)
    for s in salt:
        h = (h * 1000003 + int(s) + 17) % (1 << 61)
    g = torch.Generator(device=DEV)
    g.manual_seed(h)
    return g


def _randn(g, *shape, std=1.0):
    return (torch.randn(*shape, device=DEV, generator=g) * std).to(BF16)


def _experts(g):
    E, H, I = SH.n_experts, SH.hidden, SH.intermediate
    u8 = dict(dtype=torch.uint8, device=DEV, generator=g)
    return dict(
        w13_blocks=torch.randint(0, 256, (E, 2 * I, H // 32, 16), **u8),
        w13_scales=torch.randint(119, 124, (E, 2 * I, H // 32), **u8),
        b13=torch.randn(E, 2 * I, device=DEV, generator=g) * 0.02,
        w2_blocks=torch.randint(0, 256, (E, H, I // 32, 16), **u8),
        w2_scales=torch.randint(110, 115, (E, H, I // 32), **u8),
        b2=torch.randn(E, H, device=DEV, generator=g) * 0.02)


def _layer(seed, i):
    """The tensors of stage layer i."""
    g = _gen(seed, 1, i)
    H = SH.hidden
    return dict(
        ln1=1.0 + 0.05 * torch.randn(H, device=DEV, generator=g), ln2=1.0 + 0.05 * torch.randn(H, device=DEV, generator=g),
        wqkv=_randn(g, SH.qkv_width, H, std=0.02), bqkv=_randn(g, SH.qkv_width, std=0.02),
        wo=_randn(g, H, NQ, std=0.02), bo=_randn(g, H, std=0.02), sinks=_randn(g, HQ).float(),
        router_w=_randn(g, SH.n_experts, H, std=0.02), router_b=_randn(g, SH.n_experts, std=0.02),
        sliding=i % 2 == 0, **_experts(g))


def _rope_inv_freq():
    return 150000.0 ** (-torch.arange(0, D, 2, dtype=torch.float32) / D)


def _kv(seed, layer, caps):
    """Dense keys and values of every slot of one layer: lists of bf16 [Hkv, cap, 64]."""
    g = _gen(seed, 2, layer)
    k, v = _randn(g, sum(caps) * HKV, D), _randn(g, sum(caps) * HKV, D)
    sizes = [HKV * c for c in caps]
    return ([t.view(HKV, -1, D) for t in k.split(sizes)], [t.view(HKV, -1, D) for t in v.split(sizes)])


def _fill(kv, seed):
    for l in range(kv.n_layers):
        for s, (k, v) in enumerate(zip(*_kv(seed, l, kv.caps))):
            kv.set_dense(l, s, k, v)


def _cap(n):
    return max(64, (n + 63) // 64 * 64)


def _log_lengths(rng, n, lo, hi):
    got = [math.log(lo) + (math.log(hi) - math.log(lo)) * (i + rng.random()) / n for i in range(n)]
    rng.shuffle(got)
    return got


def _lens(case, seed):
    """(q_lens, starts) of a stage or attention case; KV lengths vary with the seed, their sum hardly."""
    rng = random.Random(int(seed) * 31 + 5)

    def lengths(n, lo, hi):  # one in each of n equal parts of the range
        got = [int(lo + (hi - lo) * (i + rng.random()) / n) for i in range(n)]
        rng.shuffle(got)
        return got

    k = case["kind"]
    if k == "stream":
        return [case["tokens"]], [case["kv"]]
    if k == "tree":
        return [case["width"] * case["depth"]], [case["kv"]]
    if k == "prefill":
        return [case["chunk"]], [case["prior"]]
    if k == "attn":
        q = [1 if i % 2 == 0 else case["verify"] for i in range(case["seqs"])]
        return q, [int(math.exp(v)) for v in _log_lengths(rng, case["seqs"], 128, case["kv_hi"] - 8)]
    q = [1] * case["decode"] + [4] * case["verify"]
    st = lengths(len(q), min(512, case["kv_hi"] // 2), case["kv_hi"]) if q else []
    return ([case["chunk"]] + q, [case["prior"]] + st) if case["chunk"] else (q, st)


def _caps(case, need):
    """The slots' capacities: the longest context of the case's kind of row, whatever the seed drew."""
    if case["kind"] != "batch":
        return [_cap(n) for n in need]
    rest = [_cap(case["kv_hi"] + 4)] * (case["decode"] + case["verify"])
    return [_cap(need[0])] + rest if case["chunk"] else rest


def _tree(case):
    """width chains of depth nodes, level by level."""
    par, dep = [], []
    for d in range(case["depth"]):
        for w in range(case["width"]):
            par.append(-1 if d == 0 else (d - 1) * case["width"] + w)
            dep.append(d)
    return par, dep


def _hidden(seed, rows, width):
    return _randn(_gen(seed, 3), rows, width)


def _moe_inputs(case, seed):
    g = _gen(seed, 4)
    w = _experts(g)
    rw, rb = _randn(g, SH.n_experts, SH.hidden, std=0.02), _randn(g, SH.n_experts, std=0.02)
    if case["hot"]:  # a tenth of the experts take about half of the tokens
        rb[torch.randperm(SH.n_experts, device=DEV, generator=g)[:SH.n_experts // 10]] += 1.2
    x, res = _randn(g, case["tokens"], SH.hidden), _randn(g, case["tokens"], SH.hidden)
    return w, rw, rb, x, res


def _fp8_inputs(case, seed):
    """e4m3 weights [257 experts (the last one shared), N, K] with one E8M0 scale per 128x128 block."""
    g = _gen(seed, 5)
    E, H, I = DS.n_experts + 1, DS.hidden, DS.intermediate

    def weight(n, k):
        w = torch.empty(E, n, k, dtype=torch.uint8, device=DEV)
        for e in range(0, E, 32):  # N(0, 100): what a 128x128 block of normal weights looks like after scaling
            m = min(32, E - e)
            w[e:e + m] = (torch.randn(m, n, k, device=DEV, dtype=BF16, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        s = torch.randint(114, 116, (E, n // 128, k // 128), dtype=torch.uint8, device=DEV, generator=g)  # 2^-13, 2^-12
        return w, s

    w1, w3, w2 = weight(I, H), weight(I, H), weight(H, I)
    rank = torch.randperm(DS.n_experts, generator=g, device=DEV).float() + 1.0
    return dict(w1=w1, w3=w3, w2=w2, ln=1.0 + 0.05 * torch.randn(H, device=DEV, generator=g),
                router_w=_randn(g, DS.n_experts, H, std=0.02), e_bias=1.6 * rank.pow(-DS.zipf_s),
                h=_randn(g, case["tokens"], H))


def _head_inputs(case, seed):
    g = _gen(seed, 6)
    # a trained head's logits are a few units wide: weights N(0, 0.02) under a final norm of about 3
    return (_randn(g, VOCAB, SH.hidden, std=0.02), 3.0 + 0.2 * torch.randn(SH.hidden, device=DEV, generator=g),
            _randn(g, case["rows"], SH.hidden))


def _sample_inputs(case, seed):
    """Logits with a normal body and a few dozen likely tokens a row; the drafted token is one of the likely ones."""
    g = _gen(seed, 7)
    R = case["rows"]
    x = torch.randn(R, VOCAB, device=DEV, generator=g) * 2.0
    span = VOCAB // 40  # the likely tokens: one in each fortieth of the vocabulary
    top = torch.arange(40, device=DEV) * span + torch.randint(0, span, (R, 40), device=DEV, generator=g)
    likely = 16.0 - 10.0 * torch.rand(R, 40, device=DEV, generator=g)
    x.scatter_(1, top, likely)
    top = top.gather(1, likely.argsort(1, descending=True))
    pick = torch.randint(0, 6, (R, 1), device=DEV, generator=g)
    return (x.to(BF16), top.gather(1, pick)[:, 0].to(torch.int32).contiguous(),
            torch.rand(R, dtype=F64, device=DEV, generator=g))


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case}
    if k in ("stream", "tree", "batch"):
        q, st = _lens(case, seed)
        need = [a + b for a, b in zip(q, st)]
        layers = [LayerWeights(**_layer(seed, i)).repack() for i in range(LAYERS)]
        rot = YarnRotary.from_inv_freq(_rope_inv_freq(), 1.0, _cap(max(need)) + 64, DEV)
        s["h"] = _hidden(seed, sum(q), SH.hidden)
        if k == "batch":
            kv = KVWorkspace(LAYERS, len(q), max(need), HKV, D, DEV, caps=_caps(case, need))
            s["stage"] = RaggedStage(SH, layers, rot, kv, max(64, sum(q)), len(q), device=DEV)
            s["q"], s["st"] = q, st
        else:
            s["stage"] = FastVerifyStage({"layers": layers, "rotary": rot, "shape": SH}, need[0], DEV, max_tokens=64)
            s["h"] = s["h"][None]
            kv = s["stage"].cache
            s["tree"] = _tree(case) if k == "tree" else None
        s["kv"] = kv
        _fill(kv, seed)
    elif k == "moe":
        w, s["rw"], s["rb"], s["x"], s["res"] = _moe_inputs(case, seed)
        s["w13"], s["w2"] = ops.mxfp4_repack(w["w13_blocks"], w["w13_scales"]), ops.mxfp4_repack(w["w2_blocks"], w["w2_scales"])
        s["b13"], s["b2"] = w["b13"], w["b2"]
    elif k == "fp8":
        w = _fp8_inputs(case, seed)
        s["h"] = w["h"]
        s["stage"] = Fp8MoeStage(DS, [Fp8MoeLayerWeights(
            ln=w["ln"], router_w=w["router_w"], e_bias=w["e_bias"],
            w13_packed=ops.fp8_repack(*w["w1"], *w["w3"]), w2_packed=ops.fp8_repack(*w["w2"]))])
    elif k in ("attn", "prefill"):
        q, st = _lens(case, seed)
        s["kv"] = kv = KVWorkspace(1, len(q), max(a + b for a, b in zip(q, st)), HKV, D, DEV, caps=[a + b for a, b in zip(q, st)])
        _fill(kv, seed)
        s["q"] = _hidden(seed, sum(q), NQ).view(-1, HQ, D)
        s["sinks"] = _randn(_gen(seed, 8), HQ).float()
        s["base"] = torch.tensor([kv.base(i) for i in range(len(q))], dtype=torch.int64, device=DEV)
        s["cap"] = torch.tensor(kv.caps, dtype=torch.int32, device=DEV)
        if k == "attn":
            items, groups, s["n_small"] = ops.attn_plan(q, st, HKV, case["window"], 1024)
            s["items"], s["groups"] = items.to(DEV), groups.to(DEV)
        else:
            _, _, _, pit = ops.attn_plan_prefill(q, st, HKV, case["window"], 1024, 32)
            s["items"], s["out"] = pit.to(DEV), torch.empty_like(s["q"])
    elif k == "linear":
        g = _gen(seed, 9)
        s["x"], s["a"], s["res"] = _randn(g, case["rows"], SH.hidden), _randn(g, case["rows"], NQ), _randn(g, case["rows"], SH.hidden)
        s["w"] = [(_randn(g, SH.qkv_width, SH.hidden, std=0.02), _randn(g, SH.qkv_width, std=0.02),
                   _randn(g, SH.hidden, NQ, std=0.02), _randn(g, SH.hidden, std=0.02)) for _ in range(LINEAR_LAYERS)]
    elif k == "head":
        w, n, s["h"] = _head_inputs(case, seed)
        s["norm"], s["w"] = FinalNorm(n, SH.rms_eps), ops.bf16_tile_repack(w)
    else:
        s["x"], s["draft"], s["u"] = _sample_inputs(case, seed)
    return s


# ---- the calls ----------------------------------------------------------------------------------------

def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "stream":
        return {"h": s["stage"].decode(s["h"], c["kv"]), "k": s["kv"].k, "v": s["kv"].v}
    if k == "tree":
        return {"h": s["stage"].tree_decode(s["h"], c["kv"], *s["tree"]), "k": s["kv"].k, "v": s["kv"].v}
    if k == "batch":
        h = s["stage"].forward(s["h"].clone(), s["q"], s["st"], list(range(len(s["q"]))))
        return {"h": h, "k": s["kv"].k, "v": s["kv"].v}
    if k == "moe":
        E, H, I = SH.n_experts, SH.hidden, SH.intermediate
        ids, wts, _, off, perm, inv = ops.moe_route_permute(s["x"], s["rw"], s["rb"], SH.top_k)
        h = ops.moe_gate_up(s["x"], perm, off, SH.top_k, s["w13"], s["b13"], E, I)
        y = ops.moe_down(h, off, s["w2"], s["b2"], E, H)
        return {"out": ops.moe_combine(y, inv, wts, residual=s["res"]), "ids": ids, "weights": wts}
    if k == "fp8":
        return s["stage"].forward(s["h"].clone())
    if k == "attn":
        return ops.attn_ragged(s["q"], s["kv"].k[0], s["kv"].v[0], s["base"], s["cap"], s["sinks"], c["window"], s["items"],
                               s["groups"], s["n_small"], HKV)
    if k == "prefill":
        return ops.attn_prefill(s["q"], s["kv"].k[0], s["kv"].v[0], s["base"], s["cap"], s["sinks"], c["window"], s["items"],
                                HKV, s["out"])
    if k == "linear":
        return [(ops.linear(s["x"], wqkv, bqkv), ops.linear(s["a"], wo, bo, residual=s["res"].clone()))
                for wqkv, bqkv, wo, bo in s["w"]]
    if k == "head":
        ids, logits = ops.lm_head_argmax(s["norm"](s["h"]), s["w"], VOCAB, want_logits=True)
        return {"ids": ids, "logits": logits}
    return ops.sample_rows(s["x"], c["temp"], c["top_k"], c["top_p"], draft=s["draft"], u=s["u"], want_p_draft=True, want_draw=True)


# ---- what a call cannot do without ----------------------------------------------------------------------

def _touched(experts, k, tokens, hot=False):
    if hot:  # half of the assignments on a tenth of the experts
        a, b = experts // 10, experts - experts // 10
        return a * (1 - (1 - min(1.0, 0.5 * k / a)) ** tokens) + b * (1 - (1 - 0.5 * k / b) ** tokens)
    return experts * (1 - (1 - k / experts) ** tokens)


def _moe_work(T, hot=False):
    E, H, I, k = SH.n_experts, SH.hidden, SH.intermediate, SH.top_k
    per = 3 * I * H * 17 // 32 + 4 * (2 * I + H)  # codes, scales, biases
    return _touched(E, k, T, hot) * per + E * H * 2 + 3 * T * H * 2 + T * k * 8, 2.0 * T * k * 3 * I * H + 2.0 * T * E * H


def _attn_work(q, st, window):
    bts = fl = 0
    for n, s in zip(q, st):
        lo = max(0, s - window + 1) if window else 0
        bts += (s + n - lo) * NKV * 4 + 2 * n * NQ * 2
        seen = sum(min(s + i + 1, window) if window else s + i + 1 for i in (0, n - 1)) / 2 * n
        fl += 4 * seen * NQ
    return bts, fl


def work(case):
    k = case["kind"]
    if k in ("stream", "tree", "batch"):
        q, st = _lens(case, 0)
        T, H = sum(q), SH.hidden
        b, f = _moe_work(T)
        proj = (SH.qkv_width + NQ) * H
        b, f = b + proj * 2 + T * NKV * 4, f + 2.0 * T * proj
        b, f = b * LAYERS, f * LAYERS
        for i in range(LAYERS):
            ab, af = _attn_work(q, st, SH.window if i % 2 == 0 else 0)
            b, f = b + ab - 4 * T * NQ, f + af  # the queries and the output stay inside the layer
    elif k == "moe":
        b, f = _moe_work(case["tokens"], case["hot"])
    elif k == "fp8":
        T, H, I, E, n = case["tokens"], DS.hidden, DS.intermediate, DS.n_experts, DS.top_k
        groups = min(E, n * T, _touched(E, n, T) * 0.84) + 1  # the Zipf-shaped selection leaves some out
        b, f = groups * 3 * I * H * (1 + 1 / 16384) + E * H * 2 + 2 * T * H * 2, 2.0 * T * ((n + 1) * 3 * I * H + E * H)
    elif k in ("attn", "prefill"):
        b, f = _attn_work(*_lens(case, 0), case["window"])
    elif k == "linear":
        R, H = case["rows"], SH.hidden
        proj = (SH.qkv_width + NQ) * H
        b, f = LINEAR_LAYERS * (proj * 2 + R * (H + SH.qkv_width + NQ + 2 * H) * 2), LINEAR_LAYERS * 2.0 * R * proj
    elif k == "head":
        b, f = VOCAB * SH.hidden * 2 + case["rows"] * (SH.hidden + VOCAB) * 2, 2.0 * case["rows"] * VOCAB * SH.hidden
    else:
        b, f = case["rows"] * VOCAB * 2, case["rows"] * VOCAB * 4.0
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    k = case["kind"]
    if k == "sample":
        return "exact"  # the draw and its probabilities are defined by integer weights, whatever the order of the sums
    if k in ("stream", "tree", "batch"):
        # four layers: a changed rounding moves some tokens' fourth expert
        return {"rel": 0.03, "max": 0.9}
    if k == "moe":
        return {"rel": 0.01, "max": 0.1, "differ": 0.005}
    if k == "fp8":
        return {"rel": 0.02, "max": 0.3}
    if k in ("attn", "prefill"):
        return {"rel": 0.01, "max": 0.1}
    if k == "linear":
        return {"rel": 0.008, "max": 0.05}
    return {"rel": 0.01, "max": 0.05, "differ": 0.01}  # head: near-ties may pick the other token


# ---- the same results in 64 bits --------------------------------------------------------------------------

def _norm64(x, w, eps):
    x = x.to(F64)
    return w.to(F64) * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _mx64(blocks, scales):
    """[N, G, 16] code bytes and [N, G] E8M0 bytes -> [N, 32 G]."""
    lut = torch.tensor(FP4, dtype=F64, device=DEV)
    b = blocks.long()
    v = torch.stack((lut[b & 15], lut[b >> 4]), -1).flatten(-2)
    return (v * torch.exp2(scales.to(F64) - 127.0)[..., None]).flatten(-2)


def _moe64(x, rw, rb, w):
    """(sum of the weighted experts, ids, weights).  The router's logits are bf16 by definition."""
    lg = (x @ rw.to(F64).T + rb.to(F64)).to(torch.float32).to(BF16).to(F64)
    ids = torch.sort(-lg, dim=1, stable=True).indices[:, :SH.top_k].sort(1).values
    wts = torch.softmax(lg.gather(1, ids), 1)
    out = torch.zeros_like(x)
    for e in range(SH.n_experts):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if not tok.numel():
            continue
        gu = x[tok] @ _mx64(w["w13_blocks"][e], w["w13_scales"][e]).T + w["b13"][e].to(F64)
        g, u = gu[:, 0::2].clamp(max=7.0), gu[:, 1::2].clamp(-7.0, 7.0)
        y = ((u + 1) * g * torch.sigmoid(1.702 * g)) @ _mx64(w["w2_blocks"][e], w["w2_scales"][e]).T + w["b2"][e].to(F64)
        out[tok] += wts[tok, slot][:, None] * y
    return out, ids.to(torch.int32), wts


def _attn64(q, keys, values, q_lens, starts, sinks, window, seen=None):
    """q [T, Hq, 64]; keys / values: a list of [Hkv, n, 64] a sequence.  seen: a [T, n] mask in place of the causal one."""
    out, t = torch.empty_like(q), 0
    for b, (n, st) in enumerate(zip(q_lens, starts)):
        lo = max(0, st - window + 1) if window else 0
        hi = st + n
        pos, key = torch.arange(st, hi, device=DEV)[:, None], torch.arange(lo, hi, device=DEV)[None]
        ok = seen[:, lo:hi] if seen is not None else (key <= pos) & ((key > pos - window) if window else True)
        for h in range(HKV):
            qh = q[t:t + n, 8 * h:8 * h + 8].reshape(n * 8, D)
            s = (qh @ keys[b][h, lo:hi].to(F64).T * D ** -0.5).view(n, 8, -1).masked_fill(~ok[:, None], -math.inf)
            sk = sinks[8 * h:8 * h + 8].to(F64)[None, :, None].expand(n, 8, 1)
            p = torch.softmax(torch.cat((s, sk), -1), -1)[..., :-1].reshape(n * 8, -1)
            out[t:t + n, 8 * h:8 * h + 8] = (p @ values[b][h, lo:hi].to(F64)).view(n, 8, D)
        t += n
    return out


def _stage64(case, seed):
    q, st = _lens(case, seed)
    T = sum(q)
    h = _hidden(seed, T, SH.hidden).to(F64)
    tree = _tree(case) if case["kind"] == "tree" else None
    slot = torch.cat([torch.arange(s, s + n, device=DEV) for n, s in zip(q, st)])
    pos = torch.tensor(tree[1], device=DEV) + st[0] if tree else slot
    ang = pos.cpu().float()[:, None] * _rope_inv_freq()[None]
    cos, sin = (f(ang).to(BF16).to(DEV).to(F64)[:, None] for f in (torch.cos, torch.sin))

    def rope(x):
        a, b = x.chunk(2, -1)
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    for i in range(LAYERS):
        w = _layer(seed, i)
        window = SH.window if w["sliding"] else 0
        qkv = _norm64(h, w["ln1"], SH.rms_eps) @ w["wqkv"].to(F64).T + w["bqkv"].to(F64)
        qr, kr = rope(qkv[:, :NQ].reshape(T, HQ, D)), rope(qkv[:, NQ:NQ + NKV].reshape(T, HKV, D))
        vr = qkv[:, NQ + NKV:].reshape(T, HKV, D)
        keys, vals, t = [], [], 0
        for b, (k, v) in enumerate(zip(*_kv(seed, i, _caps(case, [a + c for a, c in zip(q, st)])))):
            k, v = k.to(F64), v.to(F64)
            k[:, st[b]:st[b] + q[b]], v[:, st[b]:st[b] + q[b]] = kr[t:t + q[b]].transpose(0, 1), vr[t:t + q[b]].transpose(0, 1)
            keys.append(k)
            vals.append(v)
            t += q[b]
        seen, low = None, window
        if tree:  # a node sees the committed keys, itself and its ancestors; the window is one of depths
            seen = torch.zeros(T, st[0] + T, dtype=torch.bool, device=DEV)
            for n in range(T):
                seen[n, max(0, st[0] + tree[1][n] - window + 1) if window else 0:st[0]] = True
                a = n
                while a >= 0 and (not window or tree[1][n] - tree[1][a] < window):
                    seen[n, st[0] + a] = True
                    a = tree[0][a]
            low = 0
        o = _attn64(qr, keys, vals, q, st, w["sinks"], low, seen)
        h = h + o.reshape(T, NQ) @ w["wo"].to(F64).T + w["bo"].to(F64)
        h = h + _moe64(_norm64(h, w["ln2"], SH.rms_eps), w["router_w"], w["router_b"], w)[0]
    return h


def _fp8_64(case, seed):
    w = _fp8_inputs(case, seed)
    x = _norm64(w["h"], w["ln"], DS.rms_eps)
    E, n = DS.n_experts, DS.top_k
    p = torch.sigmoid(x @ w["router_w"].to(F64).T)
    choice = (p + w["e_bias"].to(F64)).view(-1, DS.n_group, E // DS.n_group)
    best = choice.topk(2, -1).values.sum(-1).topk(DS.topk_group, -1).indices
    keep = torch.zeros_like(choice[..., 0], dtype=torch.bool).scatter_(1, best, True)
    ids = choice.masked_fill(~keep[..., None], -math.inf).flatten(1).topk(n, -1).indices
    wts = p.gather(1, ids)
    wts = wts / wts.sum(1, keepdim=True) * DS.route_scale

    def dense(name, e):
        b, s = w[name]
        s = torch.exp2(s[e].to(F64) - 127.0)
        return b[e].view(torch.float8_e4m3fn).to(F64) * s.repeat_interleave(128, 0).repeat_interleave(128, 1)

    def expert(e, rows):
        g = rows @ dense("w1", e).T
        return (g * torch.sigmoid(g) * (rows @ dense("w3", e).T)) @ dense("w2", e).T

    out = w["h"].to(F64) + expert(E, x)
    for e in range(E):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel():
            out[tok] += wts[tok, slot][:, None] * expert(e, x[tok])
    return out


def _sample64(case, seed):
    x, draft, _ = _sample_inputs(case, seed)
    z = x.to(F64) / float(torch.tensor(case["temp"], dtype=torch.float32))
    if 0 < case["top_k"] < VOCAB:
        z = z.masked_fill(z < z.topk(case["top_k"], 1).values[:, -1:], -math.inf)
    p = torch.softmax(z, 1)
    if 0 < case["top_p"] < 1:  # a token stays while the mass before it, likeliest first, is at most top_p
        v, order = torch.sort(p, dim=1, descending=True, stable=True)
        keep = (v.cumsum(1) - v) <= float(torch.tensor(case["top_p"], dtype=torch.float32))
        p = p * torch.zeros_like(p).scatter_(1, order, keep.to(F64))
    p = p / p.sum(1, keepdim=True)
    return p.gather(1, draft.long()[:, None])[:, 0]


def exact(case, seed):
    k = case["kind"]
    if k in ("stream", "tree", "batch"):  # the pools hold the state's own, mostly unwritten, KV
        h = _stage64(case, seed)
        return {"h": h if k == "batch" else h[None], "k": None, "v": None}
    if k == "moe":
        w, rw, rb, x, res = _moe_inputs(case, seed)
        out, ids, wts = _moe64(x.to(F64), rw, rb, w)
        return {"out": out + res.to(F64), "ids": ids, "weights": wts}
    if k == "fp8":
        return _fp8_64(case, seed)
    if k in ("attn", "prefill"):
        q, st = _lens(case, seed)
        keys, vals = _kv(seed, 0, [_cap(a + b) for a, b in zip(q, st)])
        qq = _hidden(seed, sum(q), NQ).view(-1, HQ, D).to(F64)
        return _attn64(qq, keys, vals, q, st, _randn(_gen(seed, 8), HQ).float(), case["window"])
    if k == "linear":
        g = _gen(seed, 9)
        x, a, res = (_randn(g, case["rows"], n).to(F64) for n in (SH.hidden, NQ, SH.hidden))
        out = []
        for _ in range(LINEAR_LAYERS):
            wqkv, bqkv, wo, bo = (_randn(g, *s, std=0.02).to(F64) for s in ((SH.qkv_width, SH.hidden), (SH.qkv_width,), (SH.hidden, NQ), (SH.hidden,)))
            out.append((x @ wqkv.T + bqkv, res + a @ wo.T + bo))
        return out
    if k == "head":
        w, n, h = _head_inputs(case, seed)
        x = _norm64(h, n, SH.rms_eps)
        return {"ids": None, "logits": torch.cat([x @ part.to(F64).T for part in w.split(16384)], 1)}
    return {"p_draft": _sample64(case, seed), "draw": None}
