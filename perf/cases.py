"""Timed cases of the prefill path: its blocks and layers through the public ops, over the range of calls a server
makes.  A prefill call packs any number of new tokens up to a chunk of 16384 rows: the few tokens of a
conversation's next turn or of a long prompt's last chunk, an ordinary prompt of some hundred to some thousand
tokens, a full chunk.  Every case is one stage of a layer for such a call:

    proj     the fp8 projections `fp8.a` (q_a / kv_a / index key) and `fp8.b` (q_b / index query)
    out      the attention output: activation quant and the fp8 o projection
    mlp      the dense layers' MLP: gate_up GEMM, SiLU-mul-quant, down GEMM
    heads    the absorbed-MLA head-batched bf16 GEMMs W_UK and W_UV
    rows     the row kernels: residual add + RMSNorm + quant, MLA prep into the paged caches, q post
    indexer  one sub-chunk (at most 1024 rows) against its context: key gather, MQA logits, top 2048, stream rows
    moe      the whole MoE block: router, routing tables, gather, experts, shared expert, combine

Inputs come from plain torch (activations N(0, 1) with 1% outlier columns, weights N(0, 0.02), UE8M0 blocks of 128);
weights are laid out once, as at load time.
"""
import functools
import math

import torch

from kern_glm53_amd import moe as kgmoe
from kern_glm53_amd import ops

H, QL, KVL, ROPE, NOPE, VD, HEADS, IH, ID = 6144, 2048, 512, 64, 192, 256, 64, 32, 128
NA, NB, MLA = QL + KVL + ROPE + ID, HEADS * (NOPE + ROPE) + IH * ID, KVL + ROPE
EXPERTS, TOPK, INTER, DENSE = 256, 8, 2048, 12288
CHUNK, SUB, PAGE = 16384, 1024, 64 * 132
PROJ = {"a": (NA, H), "b": (NB, QL)}


def listed():
    return [
        # the smallest call: a handful of new tokens through the latent projection, bound by launch and latency
        {"name": "proj_a_7", "kind": "proj", "op": "a", "rows": 7},
        # a short prompt, not a multiple of any tile
        {"name": "proj_b_150", "kind": "proj", "op": "b", "rows": 150},
        # an ordinary prompt through quant and the K = 16384 projection
        {"name": "out_1000", "kind": "out", "rows": 1000},
        # a full chunk through it: the largest dense product
        {"name": "out_16384", "kind": "out", "rows": 16384},
        # a first dense layer's MLP for a short prompt
        {"name": "mlp_420", "kind": "mlp", "rows": 420},
        # the head-batched products of an ordinary prompt
        {"name": "heads_640", "kind": "heads", "rows": 640},
        # the row kernels of a longer one, three sequences packed
        {"name": "rows_2050", "kind": "rows", "rows": 2050, "seqs": 3},
        # a conversation's next turn: few rows against long contexts, two sequences packed
        {"name": "indexer_40", "kind": "indexer", "rows": 40, "context": 24000, "seqs": 2},
        # a whole sub-chunk at the end of a long document
        {"name": "indexer_1024", "kind": "indexer", "rows": 1024, "context": 65536, "seqs": 1},
        # the MoE block of a next turn, of an ordinary prompt and of a full chunk
        {"name": "moe_24", "kind": "moe", "rows": 24},
        {"name": "moe_1500", "kind": "moe", "rows": 1500},
        {"name": "moe_16384", "kind": "moe", "rows": 16384},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "out", "mlp", "heads", "rows", "indexer", "indexer", "moe", "moe"])
    c = {"kind": kind}
    if kind == "proj":
        c["op"] = rng.choice(sorted(PROJ))
    if kind == "indexer":
        c["seqs"] = rng.choice([1, 1, 2, 3])
        c["rows"] = _log_int(rng, c["seqs"], SUB)
        c["context"] = _log_int(rng, max(512, c["rows"]), 65536)        # tokens of each sequence
        return c
    c["rows"] = _log_int(rng, 1, 8192 if kind == "mlp" else CHUNK)
    if kind == "rows":
        c["seqs"] = rng.randint(1, min(4, c["rows"]))
    return c


# ------------------------------------------------------------------ operands in plain torch

def _dev():
    return torch.device("cuda")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)
    return g


def _up(x, m):
    return -(-x // m) * m


def _activations(rows, cols, g, outlier=10.0):
    x = torch.randn(rows, cols, generator=g, device=_dev())
    x[:, torch.randperm(cols, generator=g, device=_dev())[: cols // 100]] *= outlier
    return x.bfloat16()


def _exponent(amax, eps):
    """The UE8M0 byte of a block: 127 + ceil(log2(max(amax, eps) / 448))."""
    m, e = torch.frexp(amax.double().clamp_min(eps) / 448.0)
    return e.int() + 127 - (m == 0.5).int()


def _codes(x, e):
    """e4m3 codes of x / 2^(e - 127), saturating."""
    return torch.ldexp(x, 127 - e).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)


def _pack(e, rows):
    """Exponents [rows][K / 128] -> words [ceil(K / 512)][rows], byte kb & 3 of word kb >> 2, as bytes."""
    kb = e.shape[1]
    out = torch.zeros(_up(kb, 4) // 4, rows, 4, dtype=torch.uint8, device=e.device)
    for b in range(kb):
        out[b >> 2, : e.shape[0], b & 3] = e[:, b].to(torch.uint8)
    return out.view(-1)


def _quant_rows(x, rows, eps=1e-10):
    """(codes, scale words for `rows` rows) of x [r][K] per 128 columns."""
    f = x.float().view(x.shape[0], -1, 128)
    e = _exponent(f.abs().amax(2), eps)
    return _codes(f, e[:, :, None]).view(x.shape), _pack(e, rows)


def _weights(n, k, g, std=0.02):
    """(codes [n][k], scale words [k / 512][n]) of an N(0, std) matrix in 128 x 128 blocks."""
    nb = _up(n, 128)
    w = torch.randn(nb, k, generator=g, device=_dev()).mul_(std).view(nb // 128, 128, k // 128, 128)
    e = _exponent(w.abs().amax((1, 3)), 1e-4)
    q = _codes(w, e[:, None, :, None]).view(nb, k)[:n].contiguous()
    return q, _pack(e.repeat_interleave(128, 0)[:n], n)


def _unpack(words, rows, k):
    """Scale words -> 2^(e - 127), f64 [rows][k / 128]."""
    b = words.view(-1, rows, 4).permute(1, 0, 2).reshape(rows, -1)[:, : k // 128]
    return torch.ldexp(torch.ones_like(b, dtype=torch.float64), b.int() - 127)


def _f64(codes, words, rows, k):
    """The matrix that codes [.][k] and scale words for `rows` rows hold, in f64."""
    n = codes.shape[0]
    v = codes.view(torch.float8_e4m3fn).double().view(n, k // 128, 128)
    return (v * _unpack(words, rows, k)[:n, :, None]).view(n, k)


def _fp8_round(x):
    """x (f64 [r][K]) through bf16 and the per-128 UE8M0 e4m3 quant, back in f64."""
    f = x.bfloat16().float().view(x.shape[0], -1, 128)
    e = _exponent(f.abs().amax(2), 1e-10)[:, :, None]
    c = _codes(f, e).view(torch.float8_e4m3fn).double()
    return torch.ldexp(c, e - 127).view(x.shape)


def _silu_mul(gu):
    """SiLU(gate) * up of f64 [r][2 I] whose halves are stored in bf16."""
    gu = gu.bfloat16().double()
    g, u = gu.chunk(2, 1)
    return g * torch.sigmoid(g) * u


def _mm_rows(x, w, step=2048):
    return torch.cat([x[i: i + step] @ w.t() for i in range(0, x.shape[0], step)])


def _rope_table(n):
    inv = 8e6 ** (-torch.arange(32, device=_dev(), dtype=torch.float64) / 32)
    ang = torch.arange(n, device=_dev(), dtype=torch.float64)[:, None] * inv
    return torch.cat([ang.cos(), ang.sin()], 1).bfloat16().contiguous()


def _split(total, parts):
    return [total // parts + (i < total % parts) for i in range(parts)]


def _empty(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype, device=_dev())


def _bias(rank):
    """The router's correction bias by popularity rank: it leaves the largest expert five times the mean's rows and
    the smallest half of it (at a full chunk, about 2600 and 215 of a mean of 512)."""
    return -0.03 * torch.log1p(rank.float())


# ------------------------------------------------------------------ preparation

def prepare(case, seed):
    g, t = _gen(seed), case["rows"]
    s = {"kind": case["kind"], "rows": t}
    return {"proj": _prepare_proj, "out": _prepare_out, "mlp": _prepare_mlp, "heads": _prepare_heads,
            "rows": _prepare_rows, "indexer": _prepare_indexer, "moe": _prepare_moe}[case["kind"]](case, s, t, g)


def _prepare_proj(case, s, t, g):
    n, k = PROJ[case["op"]]
    s["n"], s["k"] = n, k
    s["a"], s["sfa"] = _quant_rows(_activations(t, k, g), t)
    s["w"], s["sfb"] = _weights(n, k, g)
    s["c"] = _empty(t, n)
    return s


def _prepare_out(case, s, t, g):
    k = HEADS * VD
    s["x"] = _activations(t, k, g)
    s["w"], s["sfb"] = _weights(H, k, g)
    s["q"], s["sf"] = _empty(t, k, dtype=torch.uint8), _empty(ops.sf_words(k) * t * 4, dtype=torch.uint8)
    s["c"] = _empty(t, H)
    return s


def _prepare_mlp(case, s, t, g):
    s["a"], s["sfa"] = _quant_rows(_activations(t, H, g), t)
    s["wgu"], s["sfgu"] = _weights(2 * DENSE, H, g)
    s["wdn"], s["sfdn"] = _weights(H, DENSE, g)
    s["gu"] = _empty(t, 2 * DENSE)
    s["q"], s["sf"] = _empty(t, DENSE, dtype=torch.uint8), _empty(ops.sf_words(DENSE) * t * 4, dtype=torch.uint8)
    s["c"] = _empty(t, H)
    return s


def _prepare_heads(case, s, t, g):
    bf = lambda std, *shape: (torch.randn(*shape, generator=g, device=_dev()) * std).bfloat16()
    s["qb"] = bf(1.0, t, NB)
    s["wuk"], s["kvb"] = bf(0.05, HEADS, KVL, NOPE), bf(0.05, HEADS * (NOPE + VD), KVL)
    s["qmla"], s["o"], s["ov"] = _empty(t, HEADS, MLA), bf(0.5, t, HEADS, KVL), _empty(t, HEADS, VD)
    return s


def _prepare_rows(case, s, t, g):
    bf = lambda *shape: torch.randn(*shape, generator=g, device=_dev()).bfloat16()
    s["h"], s["res0"], s["res"] = _activations(t, H, g), bf(t, H), _empty(t, H)
    s["gamma"] = (1 + 0.1 * torch.randn(H, generator=g, device=_dev())).bfloat16()
    s["xn"], s["xq"] = _empty(t, H), _empty(t, H, dtype=torch.uint8)
    s["xsf"] = _empty(ops.sf_words(H) * t * 4, dtype=torch.uint8)
    lens, before = _split(t, case["seqs"]), 1000
    s["ctx"] = _up(max(lens) + before, 64)
    s["slots"] = s["ctx"] * case["seqs"]
    s["rope"] = _rope_table(s["ctx"])
    # every sequence continues after 1000 cached tokens; its pages are scattered over the cache
    pages = torch.randperm(s["slots"] // 64, generator=g, device=_dev()).view(case["seqs"], -1)
    pos = [torch.arange(before, before + n, device=_dev()) for n in lens]
    s["pos"] = torch.cat(pos).int()
    s["slot"] = torch.cat([pages[i][p // 64] * 64 + p % 64 for i, p in enumerate(pos)])
    s["x"], s["qb"], s["iw"] = bf(t, NA), bf(t, NB), bf(t, IH)
    s["g_q"], s["g_kv"], s["ik_w"], s["ik_b"] = bf(QL), bf(KVL), bf(ID), bf(ID)
    s["kv"], s["idx"] = _empty(s["slots"], 656, dtype=torch.uint8), _empty(s["slots"] // 64 * PAGE, dtype=torch.uint8)
    s["qq"], s["qsf"] = _empty(t, QL, dtype=torch.uint8), _empty(ops.sf_words(QL) * t * 4, dtype=torch.uint8)
    s["qmla"], s["iq"] = _empty(t, HEADS, MLA), _empty(t, IH, ID, dtype=torch.uint8)
    s["wout"] = _empty(t, IH, dtype=torch.float32)
    return s


def _index_rows(case):
    """Per row of the call: the start of its sequence in the key stream and the keys it sees."""
    ks, klen = [], []
    for i, n in enumerate(_split(case["rows"], case["seqs"])):
        ks += [i * case["context"]] * n
        klen += range(case["context"] - n + 1, case["context"] + 1)
    return ks, klen


def _prepare_indexer(case, s, t, g):
    ctx, seqs = case["context"], case["seqs"]
    s["ctx"], s["seqs"], s["keys"], s["stride"] = ctx, seqs, ctx * seqs, _up(ctx, 256)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=_dev())
    ks, klen = _index_rows(case)
    s["ks"], s["klen"], s["zero"] = i32(ks), i32(klen), _empty(t, dtype=torch.int32)
    s["ke"] = s["ks"] + s["klen"]
    e4 = lambda x: x.clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    s["iq"] = e4(torch.randn(t, IH, ID, generator=g, device=_dev()) * 100)
    s["w"] = torch.randn(t, IH, generator=g, device=_dev()) * (0.01 / 64)
    # the paged index cache: 64 rows of 128 codes, then their 64 scales; a sequence's pages are scattered
    n_pages = seqs * (_up(ctx, 64) // 64)
    idx = _empty(n_pages, PAGE, dtype=torch.uint8)
    idx[:, : 64 * ID] = e4(torch.randn(n_pages, 64 * ID, generator=g, device=_dev()) * 100)
    scale = torch.exp2(torch.randint(-9, -6, (n_pages, 64), generator=g, device=_dev()).float())
    idx[:, 64 * ID:] = scale.view(torch.uint8)
    s["idx"] = idx.view(-1)
    s["table"] = torch.randperm(n_pages, generator=g, device=_dev()).int().view(seqs, -1).contiguous()
    s["seq_lens"] = i32([ctx] * seqs)
    s["kg"], s["ksf"] = _empty(ctx * seqs, ID, dtype=torch.uint8), _empty(ctx * seqs, dtype=torch.float32)
    s["logits"] = _empty(t, s["stride"], dtype=torch.float32)
    s["ind"], s["tlen"] = _empty(t, 2048, dtype=torch.int32), _empty(t, dtype=torch.int32)
    return s


def _prepare_moe(case, s, t, g):
    rows = _up(t, 128)
    s["buf"] = kgmoe.MoEBuffers(_up(t, 16), rows, _dev())
    s["xn"] = _empty(rows, H)
    s["xn"][:t] = _activations(t, H, g)
    s["xq"], s["xsf"] = _quant_rows(s["xn"], rows)

    def experts(n, k):
        """All experts' weights in fragment order, and their scale words."""
        wf = torch.empty(EXPERTS * n, k, dtype=torch.uint8, device=_dev())
        sf = []
        for e in range(EXPERTS):
            w, f = _weights(n, k, g)
            ops.fp8_weight_frag(w, wf[e * n:], n, k)
            sf.append(f)
        return wf, torch.cat(sf)

    w13f, sf13 = experts(2 * INTER, H)
    w2f, sf2 = experts(H, INTER)
    sgu, sfsgu = _weights(2 * INTER, H, g)
    sdn, sfsdn = _weights(H, INTER, g)
    w_r = (torch.randn(EXPERTS, H, generator=g, device=_dev()) * 0.009).bfloat16()      # logits near N(0, 1)
    rank = torch.randperm(EXPERTS, generator=g, device=_dev())
    s["w"] = kgmoe.MoEWeights(w_r, _bias(rank), torch.tensor([2.5], dtype=torch.bfloat16, device=_dev()),
                              None, sf13, None, sf2, sgu, sfsgu, sdn, sfsdn, w13f=w13f, w2f=w2f)
    s["h"] = _empty(rows, H)
    return s


# ------------------------------------------------------------------ one pass

def run(state):
    s, t = state, state["rows"]
    if s["kind"] == "proj":
        ops.fp8_gemm(s["a"], s["w"], s["sfa"], s["sfb"], s["c"], t, n=s["n"], k=s["k"], rows=t, lda=s["k"],
                     ldc=s["n"], sfa_rows=t)
        return s["c"]
    if s["kind"] == "out":
        k = HEADS * VD
        ops.quant(s["x"], k, s["q"], s["sf"], t, k, t)
        ops.fp8_gemm(s["q"], s["w"], s["sf"], s["sfb"], s["c"], t, n=H, k=k, rows=t, lda=k, ldc=H, sfa_rows=t)
        return {"c": s["c"], "q": s["q"], "sf": s["sf"]}
    if s["kind"] == "mlp":
        ops.fp8_gemm(s["a"], s["wgu"], s["sfa"], s["sfgu"], s["gu"], t, n=2 * DENSE, k=H, rows=t, lda=H,
                     ldc=2 * DENSE, sfa_rows=t)
        ops.silu_mul_quant(s["gu"], DENSE, s["q"], s["sf"], t, None, t)
        ops.fp8_gemm(s["q"], s["wdn"], s["sf"], s["sfdn"], s["c"], t, n=H, k=DENSE, rows=t, lda=DENSE, ldc=H,
                     sfa_rows=t)
        return {"gu": s["gu"], "c": s["c"]}
    if s["kind"] == "heads":
        ops.bf16_batched(s["qb"], s["wuk"], s["qmla"], t, n=KVL, k=NOPE, rows=t,
                         a_strides=(NB * 2, (NOPE + ROPE) * 2), b_strides=(NOPE * 2, KVL * NOPE * 2),
                         d_strides=(HEADS * MLA * 2, MLA * 2))
        ops.bf16_batched(s["o"], s["kvb"][NOPE:], s["ov"], t, n=VD, k=KVL, rows=t,
                         a_strides=(HEADS * KVL * 2, KVL * 2), b_strides=(KVL * 2, (NOPE + VD) * KVL * 2),
                         d_strides=(HEADS * VD * 2, VD * 2))
        return {"qmla": s["qmla"], "ov": s["ov"]}
    if s["kind"] == "rows":
        s["res"].copy_(s["res0"])                      # the residual stream as the previous layer left it
        ops.add_rms_quant(s["h"], s["res"], s["gamma"], s["xn"], s["xq"], s["xsf"], t, t)
        ops.mla_prep(s["x"], NA, s["g_q"], s["g_kv"], s["rope"], s["pos"], s["slot"], s["kv"], s["idx"], s["ik_w"],
                     s["ik_b"], s["qq"], s["qsf"], t, t, fp8=True, num_slots=s["slots"], rope_rows=s["ctx"])
        ops.q_post(s["qb"], NB, s["rope"], s["pos"], s["qmla"], s["iq"], s["iw"], s["wout"], 1, t,
                   rope_rows=s["ctx"])
        return {k: s[k] for k in ("res", "xn", "xq", "xsf", "kv", "idx", "qq", "qsf", "qmla", "iq", "wout")}
    if s["kind"] == "indexer":
        ops.idx_gather(s["idx"], s["table"], s["table"].shape[1], s["seq_lens"], s["seqs"], s["kg"], s["ksf"],
                       blocks=-(-s["ctx"] * s["seqs"] // 64) + s["seqs"])
        ops.mqa_logits(s["iq"], s["kg"], s["ksf"], s["w"], s["ks"], s["ke"], s["logits"], t, s["keys"], s["stride"])
        ops.topk_prefill(s["logits"], s["zero"], s["klen"], s["ind"], t, s["stride"])
        ops.topk_stream(s["ind"], s["ks"], s["klen"], s["tlen"], t)
        return {"logits": s["logits"], "ind": s["ind"], "tlen": s["tlen"]}
    kgmoe.moe_block(s["xn"], s["xq"], s["xsf"], s["w"], s["buf"], s["h"], t)
    b = s["buf"]
    return {"h": s["h"], "rl": b.rl[:t], "ids": b.ids[:t], "wts": b.wts[:t]}


# ------------------------------------------------------------------ what a pass cannot do without

def _gemm_work(m, n, k):
    return n * k + n * k // 16384 * 4 + m * k + m * k // 128 + 2 * m * n, 2 * m * n * k


@functools.lru_cache(None)
def _popularity():
    """Share of the tokens that each expert takes in the MoE cases (router logits N(0, 1) and their bias)."""
    z = torch.randn(4096, EXPERTS, generator=torch.Generator().manual_seed(1))
    ids = (torch.sigmoid(z) + _bias(torch.arange(EXPERTS))).topk(TOPK, 1).indices
    return torch.bincount(ids.flatten(), minlength=EXPERTS).double() / 4096


def _expected_experts(t):
    """Experts that t tokens reach."""
    return float((1 - (1 - _popularity()) ** t).sum())


def work(case):
    t, kind = case["rows"], case["kind"]
    if kind == "proj":
        b, f = _gemm_work(t, *PROJ[case["op"]])
    elif kind == "out":
        b, f = _gemm_work(t, H, HEADS * VD)
        b += 2 * t * HEADS * VD
    elif kind == "mlp":
        b1, f1 = _gemm_work(t, 2 * DENSE, H)
        b2, f2 = _gemm_work(t, H, DENSE)
        b, f = b1 + b2, f1 + f2
    elif kind == "heads":
        b = 2 * HEADS * (t * (NOPE + KVL + KVL + VD) + KVL * NOPE + VD * KVL)
        f = 2 * t * HEADS * (KVL * NOPE + VD * KVL)
    elif kind == "rows":
        add = 2 * 2 * H + 2 * 2 * H + H + H // 128
        prep = 2 * NA + 128 + QL + QL // 128 + 656 + 132
        post = HEADS * ROPE * 2 * 2 + IH * ID * 3 + IH * 6 + 128
        b, f = t * (add + prep + post), 0
    elif kind == "indexer":
        total = sum(_index_rows(case)[1])
        b = case["context"] * case["seqs"] * 132 + t * (IH * ID + IH * 4 + 8) + 4 * total + 4 * t * 2048
        f = 2 * IH * ID * total
    else:
        live = _expected_experts(t)
        wide = EXPERTS * H * 2 + (live + 1) * (2 * INTER * H + H * INTER) * (1 + 4 / 16384)
        b, f = wide + t * (2 * H + H + H // 128 + 2 * H), 2 * t * (TOPK + 1) * 3 * INTER * H + 2 * t * EXPERTS * H
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # four times the distance of the results from 64-bit sums: bf16 outputs 1.7e-3, the logits (f32 sums of fp8
    # products, whose matrix instruction keeps 13 bits below its largest product) 1.6e-5, the MoE block and the dense
    # MLP, which pass an e4m3 quant between two products, 2.5e-3 to 2.9e-3
    kind = case["kind"]
    if kind == "indexer":
        return {"rel": 6e-5, "max": 6e-3, "differ": 0.01}
    if kind in ("moe", "mlp"):
        return {"rel": 1e-2, "max": 0.5, "differ": 0.01}
    return {"rel": 7e-3, "max": 0.1, "differ": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits

def exact(case, seed):
    s, t, kind = prepare(case, seed), case["rows"], case["kind"]
    if kind == "proj":
        return _mm_rows(_f64(s["a"], s["sfa"], t, s["k"]), _f64(s["w"], s["sfb"], s["n"], s["k"]))
    if kind == "out":
        k = HEADS * VD
        q, sf = _quant_rows(s["x"], t)
        w = _f64(s["w"], s["sfb"], H, k)
        sc = _unpack(sf, t, k)
        rows = [((q[i: i + 1024].view(torch.float8_e4m3fn).double().view(-1, k // 128, 128)
                  * sc[i: i + 1024, :, None]).view(-1, k)) @ w.t() for i in range(0, t, 1024)]
        return {"c": torch.cat(rows), "q": None, "sf": None}
    if kind == "mlp":
        gu = _mm_rows(_f64(s["a"], s["sfa"], t, H), _f64(s["wgu"], s["sfgu"], 2 * DENSE, H))
        c = _mm_rows(_fp8_round(_silu_mul(gu)), _f64(s["wdn"], s["sfdn"], H, DENSE))
        return {"gu": gu, "c": c}
    if kind == "heads":
        q = s["qb"].view(t, -1)[:, : HEADS * (NOPE + ROPE)].view(t, HEADS, NOPE + ROPE)
        kvb = s["kvb"].view(HEADS, NOPE + VD, KVL)
        qmla = torch.zeros(t, HEADS, MLA, dtype=torch.float64, device=_dev())
        ov = torch.empty(t, HEADS, VD, dtype=torch.float64, device=_dev())
        for h in range(HEADS):
            qmla[:, h, :KVL] = q[:, h, :NOPE].double() @ s["wuk"][h].double().t()
            ov[:, h] = s["o"][:, h].double() @ kvb[h, NOPE:].double().t()
        return {"qmla": qmla, "ov": ov}
    if kind == "rows":
        return _exact_rows(s, t)
    if kind == "indexer":
        return _exact_indexer(case, s, t)
    return _exact_moe(s, t)


def _rope(x, cs):
    """Interleaved pairs of the last dimension (64) rotated by cos | sin rows cs [T][1][64]."""
    x1, x2, c, sn = x[..., 0::2], x[..., 1::2], cs[..., :32], cs[..., 32:]
    return torch.stack([x1 * c - x2 * sn, x2 * c + x1 * sn], -1).flatten(-2)


def _exact_rows(s, t):
    res = s["res0"].double() + s["h"].double()
    r = res.bfloat16().double()
    xn = (r / (r.square().mean(1, keepdim=True) + 1e-5).sqrt()).bfloat16().double() * s["gamma"].double()
    cs = s["rope"][s["pos"].long()].double()[:, None, :]
    qmla = torch.zeros(t, HEADS, MLA, dtype=torch.float64, device=_dev())
    qb = s["qb"].double()
    qmla[:, :, KVL:] = _rope(qb[:, : HEADS * 256].view(t, HEADS, 256)[:, :, NOPE:], cs)
    iq = qb[:, HEADS * 256:].view(t, IH, ID)
    iq = torch.cat([_rope(iq[:, :, :64], cs), iq[:, :, 64:]], 2)
    e = _exponent(iq.float().abs().amax(2), 1e-4)
    wout = torch.ldexp(s["iw"].double(), e - 127) * (128 ** -0.5) * (32 ** -0.5)
    out = dict.fromkeys(("res", "xn", "xq", "xsf", "kv", "idx", "qq", "qsf", "qmla", "iq", "wout"))
    out.update(res=res, xn=xn, qmla=qmla, wout=wout)
    return out


def _exact_indexer(case, s, t):
    ctx, seqs = case["context"], case["seqs"]
    pages = s["idx"].view(-1, PAGE)
    out = torch.zeros(t, s["stride"], dtype=torch.float64, device=_dev())
    ks, klen = _index_rows(case)
    row = 0
    for i, n in enumerate(_split(t, seqs)):
        pg = pages[s["table"][i].long()]
        k = pg[:, : 64 * ID].reshape(-1, ID)[:ctx].contiguous().view(torch.float8_e4m3fn).double()
        sc = pg[:, 64 * ID:].contiguous().view(torch.float32).reshape(-1)[:ctx].double()
        for r in range(row, row + n, 16):
            m = min(16, row + n - r)
            q = s["iq"][r: r + m].view(torch.float8_e4m3fn).double().view(-1, ID)
            d = (q @ k.t() * sc).relu_().view(m, IH, ctx) * s["w"][r: r + m].double()[:, :, None]
            out[r: r + m, :ctx] = d.sum(1)
            for j in range(m):
                out[r + j, klen[r + j]:] = 0
        row += n
    return {"logits": out, "ind": None, "tlen": None}


def _frag_f64(wf, e, sf, n, k):
    """Expert e's fragment-order weights in f64: blocks of 32 rows x 64 K bytes, byte h*1024 + l*16 + x of block
    (T, b) is row 32T + (l & 31), column 64b + 32(l >> 5) + 16h + x."""
    b = wf[e * n: (e + 1) * n].view(n // 32, k // 64, 2, 2, 32, 16)      # [T][b][h][l >> 5][l & 31][x]
    codes = b.permute(0, 4, 1, 3, 2, 5).reshape(n, k)
    words = sf.view(EXPERTS, -1)[e]
    return _f64(codes, words, n, k)


def _exact_moe(s, t):
    w = s["w"]
    rl = s["xn"][:t].double() @ w.w_r.double().t()
    sig = torch.sigmoid(rl)
    ids = (sig + w.bias.double()).topk(TOPK, 1).indices
    wts = sig.gather(1, ids)
    wts = wts / wts.sum(1, keepdim=True) * w.rs.double()
    rows = s["xq"].shape[0]
    sc = _unpack(s["xsf"], rows, H)

    def act(i):
        return (s["xq"][i].view(torch.float8_e4m3fn).double().view(-1, H // 128, 128) * sc[i][:, :, None]).view(-1, H)

    h = torch.zeros(rows, H, dtype=torch.float64, device=_dev())
    wgu, wdn = _f64(w.w_sgu, w.sf_sgu, 2 * INTER, H), _f64(w.w_sdn, w.sf_sdn, H, INTER)
    for i in range(0, t, 2048):
        at = torch.arange(i, min(t, i + 2048), device=_dev())
        h[at] = (_fp8_round(_silu_mul(act(at) @ wgu.t())) @ wdn.t()).bfloat16().double()
    for e in range(EXPERTS):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        if not tok.numel():
            continue
        wgu, wdn = _frag_f64(w.w13f, e, w.sf13, 2 * INTER, H), _frag_f64(w.w2f, e, w.sf2, H, INTER)
        y = (_fp8_round(_silu_mul(act(tok) @ wgu.t())) @ wdn.t()).bfloat16().double()
        h[tok] += wts[tok, slot][:, None] * y
    return {"h": h, "rl": rl, "ids": None, "wts": None}
