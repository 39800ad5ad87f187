"""What this framework is measured on: the pieces of a speculative-decoding verify step, from one
request's nine rows to a batch at the step's limit of 256 rows, through the public entry points.

A case is a dict of plain values with a "kind":

  linear   one GGUF projection of a block (ops.gemm_kquant_a)
  step     a whole captured verify step of a few layers (VerifyModel), returning its logits
  moe      the MoE block on normalised rows (ops.inference_moe)
  attn     the attention block: QK norm, RoPE, cache write, paged attention, O projection
  head     the LM head of a GGUF checkpoint (ops.inference_head)
  lists    acceptance with sampling parameters: top-k/top-p lists, then rejection sampling
  accept   DFlash proposal and acceptance over the whole vocabulary (verify.Acceptance)
  markov   the DSpark Markov head's proposal (draft_heads.MarkovHead)

Shapes are those of the dense 8B and the MoE 35B-A3B configurations of snowllm_amd/verify.py.
"""
import math

import torch

from snowllm_amd import layers, ops
from snowllm_amd.draft_heads import MarkovHead
from snowllm_amd.verify import Acceptance, LayerWeights, VerifyConfig, VerifyModel

Q4_K, Q5_K, Q6_K, Q8_0, F16, BF16 = 4, 5, 6, 8, 16, 17
FORMATS = (Q4_K, Q5_K, Q6_K, Q8_0)
BLOCK_BYTES = {Q4_K: 144, Q5_K: 176, Q6_K: 210, Q8_0: 272}   # per 256 weights
VOCAB = 151936
EPS = 1e-6
# (N, K) of the projections: the 35B-A3B shape's QKV and O, the 8B shape's QKV, O, gate/up and down
PROJECTIONS = ((5120, 2048), (2048, 4096), (6144, 4096), (4096, 4096), (14336, 4096), (4096, 14336))
# per-layer shapes: hidden, heads, kv heads, head size, rotated pairs, RoPE base
DENSE = dict(hidden=4096, heads=32, kv_heads=8, head_dim=128, rot_half=64, rope_theta=1e6)
MOE = dict(hidden=2048, heads=16, kv_heads=2, head_dim=256, rot_half=32, rope_theta=1e7)
FFN, EXPERTS, EXPERT_FFN, TOPK = 14336, 256, 512, 8
# five chains of drafts that branch at the last accepted token
TREE = (-1, 0, 1, 2, 3, 4, 0, 6, 7, 8, 9)


def listed():
    return [
        # one request's block (8 drafts) through one projection: the latency of a single launch
        dict(name="linear_9", kind="linear", fmt=Q4_K, rows=9, n=14336, k=4096),
        # fourteen requests verified together, the widest contraction of the 8B shape
        dict(name="linear_126", kind="linear", fmt=Q4_K, rows=126, n=4096, k=14336),
        # the single-user decode step: one request of 9 rows, 8K context, MoE
        dict(name="step_moe_9", kind="step", moe=True, layers=2, requests=1, block=9, context=8192),
        # a serving batch on the dense model: twelve requests of 9 rows, mixed contexts
        dict(name="step_dense_108", kind="step", moe=False, layers=2, requests=12, block=9,
             context=2048),
        # the MoE block of a batch, in the mix of a Q4_K_M file (down projections in Q6_K)
        dict(name="moe_60", kind="moe", gu=Q4_K, dn=Q6_K, rows=60),
        # long context, one tree of 11 rows, 8-bit attention weights
        dict(name="attn_220k_tree", kind="attn", moe=True, fmt=Q8_0, requests=1, block=11,
             context=220000, tree=True, spread=0.0),
        # a batch with contexts of mixed lengths, 128-wide heads
        dict(name="attn_batch_8", kind="attn", moe=False, fmt=Q4_K, requests=8, block=9,
             context=6000, tree=False, spread=0.9),
        # the LM head of a Q4_K_M / Q6_K file over five requests
        dict(name="head_q6k_45", kind="head", fmt=Q6_K, rows=45),
        # chat sampling parameters (top-k 20, top-p 0.95) for a batch of four
        dict(name="lists_topk_36", kind="lists", requests=4, block=9, vocab=VOCAB, top_k=20,
             top_p=0.95),
        # nucleus sampling with top-k unset: candidate lists as wide as the vocabulary
        dict(name="lists_topp_9", kind="lists", requests=1, block=9, vocab=VOCAB, top_k=0,
             top_p=0.9),
        # DFlash: the selector's proposal, then acceptance at temperature 1, whole vocabulary
        dict(name="accept_9", kind="accept", requests=1, block=9, vocab=VOCAB),
        # DSpark: four requests' proposals of 8 drafts with confidences
        dict(name="markov_4", kind="markov", requests=4, block=8, vocab=VOCAB, rank=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "step", "moe", "attn", "head", "lists", "accept",
                       "markov"))
    block = rng.randint(1, 16)
    if kind == "linear":
        n, k = rng.choice(PROJECTIONS)
        return dict(kind=kind, fmt=rng.choice(FORMATS), rows=_log_int(rng, 1, 256), n=n, k=k)
    if kind == "step":
        moe = rng.random() < 0.5
        requests = _log_int(rng, 1, (64 if moe else 108) // block or 1)
        return dict(kind=kind, moe=moe, layers=rng.randint(1, 2), requests=requests, block=block,
                    context=_log_int(rng, 100, 2048))
    if kind == "moe":
        gu, dn = rng.choice(((Q4_K, Q4_K), (Q4_K, Q6_K), (Q5_K, Q6_K), (Q6_K, Q6_K)))
        return dict(kind=kind, gu=gu, dn=dn, rows=_log_int(rng, 1, 64))
    if kind == "attn":
        moe = rng.random() < 0.5
        block = rng.randint(1, 16 if moe else 32)
        tokens = _log_int(rng, 100, 220000)
        return dict(kind=kind, moe=moe, fmt=rng.choice((Q4_K, Q8_0)),
                    requests=_log_int(rng, 1, max(1, min(32, 110000 // tokens))), block=block,
                    context=tokens, tree=False, spread=rng.choice((0.0, 0.5, 0.9)))
    if kind == "head":
        return dict(kind=kind, fmt=rng.choice((Q4_K, Q6_K, Q8_0, BF16)), rows=_log_int(rng, 1, 64))
    vocab = rng.choice((32000, 50257, VOCAB, 248320))
    if kind == "lists":
        top_k = rng.choice((0, 1, _log_int(rng, 2, 100), _log_int(rng, 100, 1024)))
        return dict(kind=kind, requests=rng.randint(1, 3 if top_k == 0 else 6),
                    block=rng.randint(1, 9), vocab=vocab, top_k=top_k,
                    top_p=rng.choice((0.8, 0.9, 0.95, 1.0)) if top_k else rng.choice((0.8, 0.95)))
    if kind == "accept":
        return dict(kind=kind, requests=_log_int(rng, 1, 8), block=rng.randint(2, 16), vocab=vocab)
    return dict(kind=kind, requests=_log_int(rng, 1, 8), block=rng.randint(1, 8), vocab=vocab,
                rank=rng.choice((64, 128, 256)))


# ------------------------------------------------------------------------------------------
# seeded inputs
# ------------------------------------------------------------------------------------------
def _gen(seed, part=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + part)


def _rand(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _gamma(g, n):
    return (1.0 + 0.02 * _rand(g, n)).bfloat16()


def _blocks(fmt, n, k, g):
    """GGUF blocks of a random [n, k] weight: zero-mean values of standard deviation about
    k ** -0.5, as blocks quantised from a trained matrix hold them."""
    nb, std = n * k // 256, k ** -0.5
    raw = torch.randint(0, 256, (nb, BLOCK_BYTES[fmt]), dtype=torch.uint8, device="cuda",
                        generator=g)
    spread = 1.0 + 0.2 * _rand(g, nb)
    if fmt in (Q4_K, Q5_K):
        # 6-bit scales and mins of eight sub-blocks; the min offsets half the quants' range
        half_range, rms_q = (7.5, 4.61) if fmt == Q4_K else (15.5, 9.23)
        step = 8 if fmt == Q4_K else 16
        d = (spread * (std / (36.5 * rms_q))).abs()
        raw[:, 0:4] = torch.stack([d, step * d], 1).half().view(torch.uint8).view(nb, 4)
        sc = torch.randint(0, 64, (nb, 8), dtype=torch.int32, device="cuda", generator=g)
        mn = torch.round(sc.float() * (half_range / step)).int()
        lo = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        mid = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
        hi = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
        raw[:, 4:16] = torch.cat([lo, mid, hi], 1).to(torch.uint8)
    elif fmt == Q6_K:
        sc = torch.randint(-64, 65, (nb, 16), dtype=torch.int8, device="cuda", generator=g)
        raw[:, 192:208] = sc.view(torch.uint8)
        d = (spread * (std / (37.2 * 18.5))).abs()
        raw[:, 208:210] = d.half().view(torch.uint8).view(nb, 2)
    else:
        d = ((1.0 + 0.2 * _rand(g, nb * 8)) * (std / 73.9)).abs().half().view(torch.uint8)
        raw.view(nb * 8, 34)[:, 0:2] = d.view(nb * 8, 2)
    return raw.view(-1)


def _decode(fmt, raw, n, k):
    """The [n, k] values of GGUF blocks, in 64 bits."""
    b = raw.view(-1, BLOCK_BYTES[fmt])
    half = lambda x: x.contiguous().view(torch.float16).double()  # noqa: E731
    if fmt in (Q4_K, Q5_K):
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:144] if fmt == Q4_K else b[:, 48:176]
        qs = qs.view(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32).int()
        if fmt == Q5_K:
            shift = torch.arange(8, device=b.device).view(1, 8, 1)
            q = q | (((b[:, 16:48].int().view(-1, 1, 32) >> shift) & 1) << 4)
        d, dmin = half(b[:, 0:2]).view(-1, 1, 1), half(b[:, 2:4]).view(-1, 1, 1)
        w = d * sc.double().unsqueeze(2) * q.double() - dmin * mn.double().unsqueeze(2)
    elif fmt == Q6_K:
        ql, qh = b[:, 0:128].int().view(-1, 2, 64), b[:, 128:192].int().view(-1, 2, 32)
        runs = [(ql[:, :, 0:32] & 15) | ((qh & 3) << 4),
                (ql[:, :, 32:64] & 15) | (((qh >> 2) & 3) << 4),
                (ql[:, :, 0:32] >> 4) | (((qh >> 4) & 3) << 4),
                (ql[:, :, 32:64] >> 4) | (((qh >> 6) & 3) << 4)]
        q = torch.stack(runs, 2).view(-1, 16, 16) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().unsqueeze(2)
        w = half(b[:, 208:210]).view(-1, 1, 1) * sc * q.double()
    else:
        b = raw.view(-1, 34)
        w = half(b[:, 0:2]).view(-1, 1) * b[:, 2:].contiguous().view(torch.int8).double()
    return w.reshape(n, k)


def _pack(fmt, raw, n, k, count=1):
    if count > 1:
        return ops.kquant_shuffle_stack(fmt, raw, count, n, k)
    return ops.gemm_kquant_shuffle_b(fmt, raw, n, k)


def _pages(g, requests, pages, spare=8):
    perm = torch.randperm(requests * pages + spare, device="cuda", generator=g)
    return perm[:requests * pages].int().view(requests, pages).contiguous()


def _pools(g, blocks, kv_heads, d):
    k = torch.empty(blocks, kv_heads, d // 16, 16, 16, dtype=torch.bfloat16, device="cuda")
    v = torch.empty(blocks, kv_heads, 4, d, 4, dtype=torch.bfloat16, device="cuda")
    return k.normal_(generator=g), v.normal_(generator=g)


def _contexts(case, seed):
    """The requests' context lengths: the longest is the case's, the others spread below it."""
    g = torch.Generator().manual_seed(int(seed) + 77)
    spread = case.get("spread", 0.9)
    u = torch.rand(case["requests"], generator=g) * spread
    u[0] = 0.0
    return [max(1, int(case["context"] * (1.0 - float(x)))) for x in u]


def _masks(case):
    """Ancestor masks of the block's rows (bit j: row j is visible)."""
    if case.get("tree"):
        out = []
        for i, p in enumerate(TREE):
            out.append((1 << i) | (out[p] if p >= 0 else 0))
        return out
    return [(2 << t) - 1 for t in range(case["block"])]


def _depths(case):
    if not case.get("tree"):
        return list(range(case["block"]))
    out = []
    for p in TREE:
        out.append(0 if p < 0 else out[p] + 1)
    return out


# ------------------------------------------------------------------------------------------
# linear, head, moe
# ------------------------------------------------------------------------------------------
def _linear_inputs(case, seed):
    g = _gen(seed)
    raw = _blocks(case["fmt"], case["n"], case["k"], g)
    return raw, _rand(g, case["rows"], case["k"]).bfloat16()


def _prepare_linear(case, seed):
    raw, x = _linear_inputs(case, seed)
    m, n, k = case["rows"], case["n"], case["k"]
    quant, meta = _pack(case["fmt"], raw, n, k)
    ws = torch.empty(ops.gemm_kquant_a_ws_bytes(m, k), dtype=torch.uint8, device="cuda")
    out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    return dict(kind="linear", args=(case["fmt"], x, quant, meta, out, m, n, k, ws), out=out)


def _run_linear(s):
    ops.gemm_kquant_a(*s["args"])
    return s["out"]


def _exact_linear(case, seed):
    raw, x = _linear_inputs(case, seed)
    return x.double() @ _decode(case["fmt"], raw, case["n"], case["k"]).T


def _head_inputs(case, seed):
    g = _gen(seed)
    h = MOE["hidden"]
    if case["fmt"] == BF16:
        w = (_rand(g, VOCAB, h) * h ** -0.5).bfloat16()
    else:
        w = _blocks(case["fmt"], VOCAB, h, g)
    return w, _rand(g, case["rows"], h).bfloat16()


def _prepare_head(case, seed):
    w, x = _head_inputs(case, seed)
    ops.select_geometry(0)
    if case["fmt"] == BF16:
        w = ops.lm_head_shuffle_weight(w)
    else:
        w = ops.KQuantProjWeight(*_pack(case["fmt"], w, VOCAB, MOE["hidden"]), case["fmt"])
    scratch = torch.empty(ops.lm_head_scratch_bytes(case["rows"]), dtype=torch.uint8,
                          device="cuda")
    out = torch.empty(case["rows"], VOCAB, device="cuda")
    return dict(kind="head", args=(x, w, out, scratch), out=out)


def _run_head(s):
    ops.inference_head(*s["args"])
    return s["out"]


def _exact_head(case, seed):
    w, x = _head_inputs(case, seed)
    out = []
    for r0 in range(0, VOCAB, 16384):   # in slices: the whole head in 64 bits is large
        r1 = min(VOCAB, r0 + 16384)
        if case["fmt"] == BF16:
            part = w[r0:r1].double()
        else:
            row = MOE["hidden"] // 256 * BLOCK_BYTES[case["fmt"]]
            part = _decode(case["fmt"], w[r0 * row:r1 * row], r1 - r0, MOE["hidden"])
        out.append(x.double() @ part.T)
    return torch.cat(out, 1)


def _experts(g, gu, dn):
    """GGUF blocks of one MoE layer: (expert gate/up stack, expert down stack, shared gate/up,
    shared down) and the router [E + 1, H] with logits of standard deviation about 2.5."""
    h, f = MOE["hidden"], EXPERT_FFN
    raws = (_blocks(gu, EXPERTS * 2 * f, h, g), _blocks(dn, EXPERTS * h, f, g),
            _blocks(gu, 2 * f, h, g), _blocks(dn, h, f, g))
    return raws, (_rand(g, EXPERTS + 1, h) * (2.5 * h ** -0.5)).bfloat16()


def _pack_experts(raws, gu, dn):
    h, f = MOE["hidden"], EXPERT_FFN
    return (_pack(gu, raws[0], 2 * f, h, EXPERTS), _pack(dn, raws[1], h, f, EXPERTS),
            _pack(gu, raws[2], 2 * f, h), _pack(dn, raws[3], h, f))


def _moe_inputs(case, seed):
    g = _gen(seed)
    raws, router = _experts(g, case["gu"], case["dn"])
    return raws, router, _rand(g, case["rows"], MOE["hidden"]).bfloat16()


def _prepare_moe(case, seed):
    raws, router, x = _moe_inputs(case, seed)
    ops.select_geometry(0)
    gu, dn, sgu, sdn = _pack_experts(raws, case["gu"], case["dn"])
    scratch = torch.empty(ops.inference_moe_workspace_bytes(case["rows"]), dtype=torch.uint8,
                          device="cuda")
    out = torch.empty_like(x)
    args = (x, ops.moe_shuffle_router(router),
            ops.KQuantExpertWeight(*gu, None, case["gu"]),
            ops.KQuantExpertWeight(*dn, None, case["dn"]),
            ops.KQuantProjWeight(*sgu, case["gu"]), ops.KQuantProjWeight(*sdn, case["dn"]),
            out, scratch)
    return dict(kind="moe", args=args, out=out)


def _run_moe(s):
    ops.inference_moe(*s["args"])
    return s["out"]


def _swiglu(x, gate_up, down):
    f = gate_up.shape[0] // 2
    a, u = x @ gate_up[:f].T, x @ gate_up[f:].T
    return (a * torch.sigmoid(a) * u) @ down.T


def _exact_moe_block(x, raws, router, gu, dn):
    h, f = MOE["hidden"], EXPERT_FFN
    logits = x @ router.double().T
    w, ids = logits[:, :EXPERTS].softmax(-1).topk(TOPK, -1)
    w = w / w.sum(-1, keepdim=True)
    out = torch.sigmoid(logits[:, EXPERTS:]) * _swiglu(
        x, _decode(gu, raws[2], 2 * f, h), _decode(dn, raws[3], h, f))
    gb, db = raws[0].numel() // EXPERTS, raws[1].numel() // EXPERTS
    for e in ids.unique().tolist():
        r, k = (ids == e).nonzero(as_tuple=True)
        y = _swiglu(x[r], _decode(gu, raws[0][e * gb:(e + 1) * gb], 2 * f, h),
                    _decode(dn, raws[1][e * db:(e + 1) * db], h, f))
        out.index_add_(0, r, w[r, k].unsqueeze(1) * y)
    return out


def _exact_moe(case, seed):
    raws, router, x = _moe_inputs(case, seed)
    return _exact_moe_block(x.double(), raws, router, case["gu"], case["dn"])


# ------------------------------------------------------------------------------------------
# attention block
# ------------------------------------------------------------------------------------------
def _exact_rms(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.double()


def _exact_rope(x, cos, sin, half):
    a, b = x[..., :half], x[..., half:2 * half]
    c, s = cos.unsqueeze(1), sin.unsqueeze(1)
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * half:]], -1)


def _angles(positions, shape, dtype):
    half = shape["rot_half"]
    inv = 1.0 / shape["rope_theta"] ** (torch.arange(half, device="cuda", dtype=torch.float32)
                                        / half)
    # the tables are single precision, the angle a single-precision product
    a = positions.float().unsqueeze(1) * inv
    return a.to(dtype).cos(), a.to(dtype).sin()


def _exact_attention(shape, proj, q_gamma, k_gamma, cos, sin, kp, vp, table, contexts, masks):
    """softmax(q k^T / sqrt(d)) v over the paged context and the block's visible rows."""
    hq, hk, d, half = shape["heads"], shape["kv_heads"], shape["head_dim"], shape["rot_half"]
    t = len(masks)
    rows = proj.shape[0]
    q = _exact_rope(_exact_rms(proj[:, :hq * d].view(rows, hq, d), q_gamma), cos, sin, half)
    k = _exact_rope(_exact_rms(proj[:, hq * d:(hq + hk) * d].view(rows, hk, d), k_gamma), cos, sin,
                    half)
    v = proj[:, (hq + hk) * d:].view(rows, hk, d)
    bits = torch.tensor([[(m >> j) & 1 for j in range(t)] for m in masks], device="cuda").bool()
    out = torch.empty(rows, hq, d, dtype=torch.float64, device="cuda")
    for b, ctx in enumerate(contexts):
        pages = table[b, :(ctx + 15) // 16].long()
        kc = kp[pages].permute(0, 3, 1, 2, 4).reshape(-1, hk, d)[:ctx]
        vc = vp[pages].permute(0, 2, 4, 1, 3).reshape(-1, hk, d)[:ctx]
        rs = slice(b * t, (b + 1) * t)
        for h in range(hk):
            keys = torch.cat([kc[:, h].double(), k[rs, h]])
            vals = torch.cat([vc[:, h].double(), v[rs, h]])
            grp = slice(h * hq // hk, (h + 1) * hq // hk)
            scores = (q[rs, grp].reshape(-1, d) @ keys.T * d ** -0.5).view(t, -1, ctx + t)
            scores[:, :, ctx:].masked_fill_(~bits.unsqueeze(1), -math.inf)
            out[rs, grp] = (scores.softmax(-1).view(-1, ctx + t) @ vals).view(t, -1, d)
    return out.view(rows, -1)


def _attn_inputs(case, seed):
    shape = MOE if case["moe"] else DENSE
    g = _gen(seed)
    hq, hk, d = shape["heads"], shape["kv_heads"], shape["head_dim"]
    rows = case["requests"] * case["block"]
    pages = (case["context"] + case["block"] + 15) // 16
    contexts, depths = _contexts(case, seed), _depths(case)
    positions = torch.tensor([c + x for c in contexts for x in depths], device="cuda")
    w = _blocks(case["fmt"], shape["hidden"], hq * d, g)
    proj = _rand(g, rows, (hq + 2 * hk) * d).bfloat16()
    gammas = _gamma(g, d), _gamma(g, d)
    table = _pages(g, case["requests"], pages)
    kp, vp = _pools(g, case["requests"] * pages + 8, hk, d)
    return shape, rows, contexts, positions, w, proj, gammas, table, kp, vp


def _prepare_attn(case, seed):
    shape, rows, contexts, positions, w, proj, gammas, table, kp, vp = _attn_inputs(case, seed)
    hq, hk, d, hidden = (shape[n] for n in ("heads", "kv_heads", "head_dim", "hidden"))
    t = case["block"]
    cos, sin = _angles(positions, shape, torch.float32)
    at = torch.tensor([c + j for c in contexts for j in range(t)], device="cuda")
    req = torch.arange(case["requests"], device="cuda").repeat_interleave(t)
    tree = None
    if case["tree"]:
        tree = torch.tensor(_masks(case) * case["requests"], dtype=torch.int64, device="cuda")
    u8 = dict(dtype=torch.uint8, device="cuda")
    return dict(
        kind="attn", shape=shape, rows=rows, fmt=case["fmt"], proj=proj, gammas=gammas, cos=cos,
        sin=sin, kp=kp, vp=vp, table=table, tree=tree,
        slots=(table[req, at // 16] * 16 + at % 16).int(),
        lens=torch.tensor([c + t for c in contexts], dtype=torch.int32, device="cuda"),
        attn=torch.empty(rows, hq, d, dtype=torch.bfloat16, device="cuda"),
        out=torch.empty(rows, hidden, dtype=torch.bfloat16, device="cuda"),
        scratch=torch.empty(ops.paged_attention_explicit_scratch_bytes(case["requests"], t, hq, hk,
                                                                       d), **u8),
        ws=torch.empty(ops.gemm_kquant_a_ws_bytes(rows, hq * d), **u8),
        o=_pack(case["fmt"], w, hidden, hq * d))


def _run_attn(s):
    shape, rows = s["shape"], s["rows"]
    hq, d, hidden = shape["heads"], shape["head_dim"], shape["hidden"]
    # with 256-wide heads the attention also writes the projection's operands
    wide = d == 256
    ops.paged_attention_qk(s["proj"], *s["gammas"], s["cos"], s["sin"], EPS, s["slots"], s["kp"],
                           s["vp"], s["attn"], s["table"], s["lens"], d ** -0.5, s["scratch"],
                           num_heads=hq, num_kv_heads=shape["kv_heads"], tree=s["tree"],
                           ws_out=s["ws"] if wide else None)
    if wide:
        ops.gemm_kquant_a_prepared(s["fmt"], *s["o"], s["out"], rows, hidden, hq * d, s["ws"])
    else:
        ops.gemm_kquant_a(s["fmt"], s["attn"].view(rows, -1), *s["o"], s["out"], rows, hidden,
                          hq * d, s["ws"])
    return dict(attn=s["attn"].view(rows, -1), out=s["out"], k_pool=s["kp"], v_pool=s["vp"])


def _exact_attn(case, seed):
    shape, rows, contexts, positions, w, proj, gammas, table, kp, vp = _attn_inputs(case, seed)
    cos, sin = _angles(positions, shape, torch.float64)
    attn = _exact_attention(shape, proj.double(), *gammas, cos, sin, kp, vp, table, contexts,
                            _masks(case))
    o = _decode(case["fmt"], w, shape["hidden"], attn.shape[1])
    return dict(attn=attn, out=attn @ o.T, k_pool=None, v_pool=None)


# ------------------------------------------------------------------------------------------
# whole step
# ------------------------------------------------------------------------------------------
def _step_inputs(case, seed):
    """The raw weights of the step's model (GGUF blocks, 16-bit embedding, router and head)."""
    shape = MOE if case["moe"] else DENSE
    h, hq, hk, d = (shape[n] for n in ("hidden", "heads", "kv_heads", "head_dim"))
    g = _gen(seed)
    out = []
    for _ in range(case["layers"]):
        w = dict(in_norm=_gamma(g, h), post_norm=_gamma(g, h), q_norm=_gamma(g, d),
                 k_norm=_gamma(g, d), qkv=_blocks(Q4_K, (hq + 2 * hk) * d, h, g),
                 o=_blocks(Q4_K, h, hq * d, g))
        if case["moe"]:
            w["experts"], w["router"] = _experts(g, Q4_K, Q4_K)
        else:
            w["gu"], w["dn"] = _blocks(Q4_K, 2 * FFN, h, g), _blocks(Q4_K, h, FFN, g)
        out.append(w)
    embed = _rand(g, VOCAB, h).half()
    head = (_rand(g, VOCAB, h) * h ** -0.5).half()
    return shape, out, embed, head, _gamma(g, h)


def _step_rows(case, seed):
    g = torch.Generator().manual_seed(int(seed) + 5)
    return torch.randint(0, VOCAB, (case["requests"], case["block"]), generator=g)


def _step_cache(case, seed, shape):
    pages = (case["context"] + case["block"] + 15) // 16
    g = _gen(seed, 1)
    table = _pages(g, case["requests"], pages)
    return table, [_pools(g, case["requests"] * pages + 8, shape["kv_heads"], shape["head_dim"])
                   for _ in range(case["layers"])]


def _install(model, raw, embed, head, final_norm):
    c = model.cfg
    h, qd = c.hidden, c.heads * c.head_dim
    model.layers = []
    for w in raw:
        lw = LayerWeights(in_norm=w["in_norm"], post_norm=w["post_norm"], q_norm=w["q_norm"],
                          k_norm=w["k_norm"], qkv=_pack(Q4_K, w["qkv"], c.qkv_n, h),
                          o=_pack(Q4_K, w["o"], h, qd))
        if c.moe:
            lw.router = layers.dense_shuffle(w["router"])
            lw.gu, lw.dn, lw.sh_gu, lw.sh_dn = _pack_experts(w["experts"], Q4_K, Q4_K)
        else:
            lw.gu, lw.dn = _pack(Q4_K, w["gu"], 2 * FFN, h), _pack(Q4_K, w["dn"], h, FFN)
        model.layers.append(lw)
    model.embed, model.lm_head, model.final_norm = embed, layers.dense_shuffle(head), final_norm


def _prepare_step(case, seed):
    shape, raw, embed, head, final_norm = _step_inputs(case, seed)
    extra = dict(experts=EXPERTS, expert_ffn=EXPERT_FFN, topk=TOPK) if case["moe"] else dict(ffn=FFN)
    cfg = VerifyConfig("step", layers=case["layers"], vocab=VOCAB, context=case["context"],
                       block=case["block"], eps=EPS, **shape, **extra)
    m = VerifyModel(cfg, batch=case["requests"],
                    weights=lambda model: _install(model, raw, embed, head, final_norm))
    table, pools = _step_cache(case, seed, shape)
    m.table.copy_(table)
    for i, (k, v) in enumerate(pools):
        m.k_pools[i].copy_(k)
        m.v_pools[i].copy_(v)
    m.set_batch(_step_rows(case, seed), _contexts(case, seed))
    # the step as a program keeps it: captured once, replayed for every block
    m.forward()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        m.forward()
    return dict(kind="step", model=m, graph=graph)


def _run_step(s):
    s["graph"].replay()
    m = s["model"]
    return dict(logits=m.logits, k=list(m.k_pools), v=list(m.v_pools))


def _exact_step(case, seed):
    shape, raw, embed, head, final_norm = _step_inputs(case, seed)
    h, hq, hk, d = (shape[n] for n in ("hidden", "heads", "kv_heads", "head_dim"))
    table, pools = _step_cache(case, seed, shape)
    contexts, t = _contexts(case, seed), case["block"]
    positions = torch.tensor([c + j for c in contexts for j in range(t)], device="cuda")
    cos, sin = _angles(positions, shape, torch.float64)
    x = embed[_step_rows(case, seed).view(-1).cuda()].double()
    res = torch.zeros_like(x)
    for w, (kp, vp) in zip(raw, pools):
        res = res + x
        proj = _exact_rms(res, w["in_norm"]) @ _decode(Q4_K, w["qkv"], (hq + 2 * hk) * d, h).T
        attn = _exact_attention(shape, proj, w["q_norm"], w["k_norm"], cos, sin, kp, vp, table,
                                contexts, _masks(case))
        res = res + attn @ _decode(Q4_K, w["o"], h, hq * d).T
        y = _exact_rms(res, w["post_norm"])
        if case["moe"]:
            x = _exact_moe_block(y, w["experts"], w["router"], Q4_K, Q4_K)
        else:
            x = _swiglu(y, _decode(Q4_K, w["gu"], 2 * FFN, h), _decode(Q4_K, w["dn"], h, FFN))
    y = _exact_rms(res + x, final_norm)
    none = [None] * case["layers"]
    return dict(logits=torch.cat([y @ part.double().T for part in head.split(16384)], 1), k=none,
                v=none)


# ------------------------------------------------------------------------------------------
# acceptance
# ------------------------------------------------------------------------------------------
def _target_logits(g, rows, vocab):
    """Logits as a language model's: a broad floor and some tens of likely tokens per row."""
    x = 2.0 * _rand(g, rows, vocab)
    part = vocab // 48   # one likely token in each 48th of the vocabulary: no id twice
    at = torch.randint(0, part, (rows, 48), device="cuda", generator=g)
    at += part * torch.arange(48, device="cuda")
    return x.scatter_add_(1, at, 4.0 + 8.0 * torch.rand(rows, 48, device="cuda", generator=g))


def _lists_inputs(case, seed):
    g = _gen(seed)
    b, t, v = case["requests"], case["block"], case["vocab"]
    logits = _target_logits(g, b * t, v)
    # the draft's 16 candidates: likely tokens of the target's rows, its probabilities noisy
    noisy = logits.view(b, t, v)[:, :t - 1] + 0.5 * _rand(g, b, t - 1, v)
    top, cand = noisy.topk(16, -1) if t > 1 else (noisy[..., :16], noisy[..., :16].long())
    q = top.softmax(-1)
    drafts = torch.empty(b, t - 1, dtype=torch.int64, device="cuda")
    if t > 1:
        pick = torch.multinomial(q.view(-1, 16), 1, generator=g).view(b, t - 1, 1)
        drafts = cand.gather(2, pick).squeeze(2)
    uniform = torch.rand(b, t, device="cuda", generator=g)
    temperature = (0.6 + 0.4 * torch.rand(b, 1, device="cuda", generator=g)).expand(b, t)
    return logits, cand.contiguous(), q.contiguous(), drafts.contiguous(), uniform, \
        temperature.reshape(-1).contiguous()


def _prepare_lists(case, seed):
    logits, cand, q, drafts, uniform, temperature = _lists_inputs(case, seed)
    b, t, v = case["requests"], case["block"], case["vocab"]
    n, k = b * t, case["top_k"] or ops.SAMPLING_MAX_K
    width = min(k, v)
    i64 = dict(dtype=torch.int64, device="cuda")
    return dict(
        kind="lists", logits=logits, cand=cand, q=q, drafts=drafts, uniform=uniform,
        temperature=temperature, width=width,
        top_k=torch.full((n,), k, dtype=torch.int32, device="cuda"),
        top_p=torch.full((n,), case["top_p"], device="cuda"),
        p=torch.empty(n, width, device="cuda"), ids=torch.empty(n, width, **i64),
        ws=torch.empty(ops.sample_workspace_bytes(n, v, width), dtype=torch.uint8, device="cuda"),
        slots=torch.arange(b, dtype=torch.int32, device="cuda"),
        valid=torch.ones(b, dtype=torch.int32, device="cuda"), out=torch.empty(b, t, **i64),
        accepted=torch.empty(b, **i64))


def _run_lists(s):
    ops.probabilities(s["logits"], s["top_k"], s["top_p"], s["temperature"], s["width"], s["p"],
                      s["ids"], s["ws"])
    ops.dflash.reject(s["p"], s["ids"], s["drafts"], s["cand"], s["q"], s["slots"], s["valid"],
                      s["uniform"], s["out"], s["accepted"])
    return dict(p=s["p"], ids=s["ids"], out=s["out"], accepted=s["accepted"])


def _exact_lists(case, seed):
    logits, _, _, _, _, temperature = _lists_inputs(case, seed)
    v = case["vocab"]
    k = min(case["top_k"] or v, v)
    p = (logits.double() / temperature.double().unsqueeze(1)).softmax(-1)
    p = p.sort(dim=-1, descending=True, stable=True)[0][:, :k]
    p = p / p.sum(-1, keepdim=True)
    if case["top_p"] < 1.0:
        p = p * (p.cumsum(-1) - p < case["top_p"])
        p = p / p.sum(-1, keepdim=True)
    return dict(p=p, ids=None, out=None, accepted=None)


def _accept_inputs(case, seed):
    g = _gen(seed)
    b, t, v = case["requests"], case["block"], case["vocab"]
    n = b * (t - 1)
    target = _target_logits(g, b * t, v)
    draft = target.view(b, t, v)[:, :t - 1].reshape(n, v) + 0.5 * _rand(g, n, v)
    hp, pred, succ = (0.2 * _rand(g, m, 256) for m in (n, v, v))
    anchor = torch.randint(0, v, (b,), device="cuda", generator=g)
    u = torch.rand(b, 2 * t - 1, device="cuda", generator=g)
    return target, draft, hp.bfloat16(), pred.bfloat16(), succ.bfloat16(), anchor, \
        u[:, :t - 1].contiguous(), u[:, t - 1:].contiguous()


def _prepare_accept(case, seed):
    target, draft, hp, pred, succ, anchor, select_u, uniform = _accept_inputs(case, seed)
    b, t = case["requests"], case["block"]
    acc = Acceptance(case["vocab"], list(range(t)), batch=b, block=t)
    acc.set_selector(hp, draft, pred, succ, anchor, torch.ones(b, device="cuda"), select_u,
                     uniform)
    return dict(kind="accept", acc=acc, target=target)


def _run_accept(s):
    acc = s["acc"]
    acc.propose()
    out, accepted = acc(s["target"])
    return dict(drafts=acc.drafts, candidates=acc.qid, q=acc.q, out=out, accepted=accepted)


def _exact_accept(case, seed):
    _, draft, hp, pred, succ, prev, select_u, _ = _accept_inputs(case, seed)
    b, k = case["requests"], case["block"] - 1
    top, cand = draft.view(b, k, -1).topk(16, -1)
    q = torch.empty(b, k, 16, dtype=torch.float64, device="cuda")
    for j in range(k):
        # the sampling walk rounds the product and the correction to bf16
        a = (pred[prev].float() * hp.view(b, k, -1)[:, j].float()).bfloat16().double()
        corr = (succ[cand[:, j]].double() @ a.unsqueeze(2)).squeeze(2).float().bfloat16().double()
        q[:, j] = (top[:, j].double() + corr).softmax(-1)
        pick = (q[:, j].cumsum(-1) <= select_u[:, j:j + 1].double()).sum(-1).clamp(max=15)
        prev = cand[:, j].gather(1, pick.unsqueeze(1)).squeeze(1)
    return dict(drafts=None, candidates=None, q=q, out=None, accepted=None)


def _markov_inputs(case, seed):
    g = _gen(seed)
    b, t, v, r = case["requests"], case["block"], case["vocab"], case["rank"]
    h = MOE["hidden"]
    w1, w2 = ((0.25 * _rand(g, v, r)).bfloat16() for _ in range(2))
    conf = 0.05 * _rand(g, h + r)
    rows = _rand(g, b * t, h).bfloat16()
    logits = _target_logits(g, b * t, v)
    return w1, w2, conf, 0.1 * _rand(g, 1), rows, logits, \
        torch.randint(0, v, (b,), device="cuda", generator=g)


def _prepare_markov(case, seed):
    w1, w2, conf_w, conf_b, rows, logits, anchor = _markov_inputs(case, seed)
    b, t = case["requests"], case["block"]
    return dict(kind="markov", head=MarkovHead(w1, w2, conf_w, conf_b), rows=rows, logits=logits,
                anchor=anchor, path=torch.empty(b, t, dtype=torch.int64, device="cuda"),
                confidence=torch.empty(b, t, device="cuda"))


def _run_markov(s):
    s["head"].propose(s["rows"], s["logits"], s["anchor"], s["path"], s["confidence"])
    return dict(path=s["path"], confidence=s["confidence"])


def _exact_markov(case, seed):
    w1, w2, conf_w, conf_b, rows, logits, prev = _markov_inputs(case, seed)
    b, t, h = case["requests"], case["block"], MOE["hidden"]
    w2, conf = w2.double(), torch.empty(b, t, dtype=torch.float64, device="cuda")
    for j in range(t):
        latent = w1[prev].double()
        z = torch.cat([rows.view(b, t, h)[:, j].double(), latent], 1) @ conf_w.double()
        conf[:, j] = torch.sigmoid(z + conf_b.double())
        bias = (latent @ w2.T).float().bfloat16().float()
        prev = (logits.view(b, t, -1)[:, j] + bias).argmax(-1)
    return dict(path=None, confidence=conf)


# ------------------------------------------------------------------------------------------
_KINDS = {
    "linear": (_prepare_linear, _run_linear, _exact_linear),
    "head": (_prepare_head, _run_head, _exact_head),
    "moe": (_prepare_moe, _run_moe, _exact_moe),
    "attn": (_prepare_attn, _run_attn, _exact_attn),
    "step": (_prepare_step, _run_step, _exact_step),
    "lists": (_prepare_lists, _run_lists, _exact_lists),
    "accept": (_prepare_accept, _run_accept, _exact_accept),
    "markov": (_prepare_markov, _run_markov, _exact_markov),
}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["kind"]][1](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def _weight(fmt, n, k):
    return n * k * 2 if fmt in (F16, BF16) else n * k // 256 * BLOCK_BYTES[fmt]


def _touched(rows):
    """Expected number of distinct experts of `rows` rows."""
    return EXPERTS * (1.0 - (1.0 - TOPK / EXPERTS) ** rows)


def _moe_work(rows, gu, dn):
    h, f = MOE["hidden"], EXPERT_FFN
    per_expert = _weight(gu, 2 * f, h) + _weight(dn, h, f)
    return ((_touched(rows) + 1) * per_expert + (EXPERTS + 1) * h * 2 + rows * h * 4,
            2.0 * rows * ((TOPK + 1) * 3 * f * h + (EXPERTS + 1) * h))


def _attn_work(case, shape):
    hq, hk, d = shape["heads"], shape["kv_heads"], shape["head_dim"]
    rows = case["requests"] * case["block"]
    spread = case.get("spread", 0.9)
    # the longest context, the others uniform below it
    tokens = case["context"] * (1 + (case["requests"] - 1) * (1 - spread / 2))
    return (tokens * hk * d * 4 + rows * (2 * hq + 4 * hk) * d * 2,
            4.0 * tokens * case["block"] * hq * d)


def work(case):
    """One pass's input read once and output written once, and its multiplications and additions."""
    kind = case["kind"]
    if kind in ("linear", "head"):
        n, k = (case["n"], case["k"]) if kind == "linear" else (VOCAB, MOE["hidden"])
        m, out = case["rows"], 2 if kind == "linear" else 4
        return dict(bytes=_weight(case["fmt"], n, k) + m * k * 2 + m * n * out,
                    flops=2.0 * m * n * k)
    if kind == "moe":
        nbytes, flops = _moe_work(case["rows"], case["gu"], case["dn"])
        return dict(bytes=nbytes, flops=flops)
    if kind == "attn":
        shape = MOE if case["moe"] else DENSE
        nbytes, flops = _attn_work(case, shape)
        rows, n, k = (case["requests"] * case["block"], shape["hidden"],
                      shape["heads"] * shape["head_dim"])
        return dict(bytes=nbytes + _weight(case["fmt"], n, k) + rows * n * 2,
                    flops=flops + 2.0 * rows * n * k)
    if kind == "step":
        shape = MOE if case["moe"] else DENSE
        h, hq, hk, d = (shape[n] for n in ("hidden", "heads", "kv_heads", "head_dim"))
        rows = case["requests"] * case["block"]
        a_bytes, a_flops = _attn_work(case, shape)
        if case["moe"]:
            f_bytes, f_flops = _moe_work(rows, Q4_K, Q4_K)
        else:
            f_bytes, f_flops = 3 * _weight(Q4_K, FFN, h), 6.0 * rows * FFN * h
        qkv = (hq + 2 * hk) * d
        layer = a_bytes + f_bytes + _weight(Q4_K, qkv, h) + _weight(Q4_K, h, hq * d)
        flops = a_flops + f_flops + 2.0 * rows * h * (qkv + hq * d)
        return dict(bytes=case["layers"] * layer + VOCAB * h * 2 + rows * (h * 2 + VOCAB * 4),
                    flops=case["layers"] * flops + 2.0 * rows * VOCAB * h)
    b, t, v = case["requests"], case["block"], case["vocab"]
    if kind == "lists":
        width = min(case["top_k"] or v, v)
        return dict(bytes=b * t * (v * 4 + width * 12), flops=8.0 * b * t * v)
    if kind == "accept":
        return dict(bytes=b * ((2 * t - 1) * v * 4 + (t - 1) * 33 * 512), flops=16.0 * b * t * v)
    return dict(bytes=v * case["rank"] * 2 + b * t * v * 4, flops=2.0 * b * t * v * case["rank"])


def tolerance(case):
    """Integer lists and the acceptance's probabilities are canonical: every implementation gives
    the same bits. The rest has bf16 in and out and 32-bit sums, and states about four times
    what the outputs are off the 64-bit values: 1.7e-3 for one bf16 rounding (a projection),
    2.9e-3 for the attention block, 3.9e-3 for the MoE block, 6e-3 for a whole step, where a
    routing tie may turn as well. The head's logits and the confidences stay in 32 bits."""
    kind = case["kind"]
    if kind in ("lists", "accept"):
        return "exact"
    if kind in ("markov", "head"):
        return {"rel": 1e-5, "max": 1e-4}
    rel = {"linear": 7e-3, "attn": 1.2e-2, "moe": 1.6e-2, "step": 2.4e-2}[kind]
    return {"rel": rel, "max": 0.5 if kind == "step" else 0.08}
