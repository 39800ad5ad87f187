"""Draft-side proposal heads on the GPU: the DSpark Markov walk (snowllm_dspark_markov) against
oracle/dspark.py -- picks bit for bit, confidence within 1e-5 as the reference's own check
(tests/test_lfm2_dspark_reference.py:158-163) -- and the DFlash 2 selector's hidden projection
(SELECTOR_HIDDEN, models/qwen3_5/dflash_draft.py:187-204) within the matmul tolerance, feeding
the selector walk bit-exactly against the C oracle."""
import numpy as np
import pytest
import torch

from oracle import accept as A
from oracle import dspark as D
from oracle import quant as Q

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _markov_case(V, rank, b, block, seed, stride_pad=0):
    g = torch.Generator().manual_seed(seed)
    W1 = (torch.randn(V, rank, generator=g) * .25).bfloat16()
    W2 = (torch.randn(V, rank, generator=g) * .25 * (256 / rank) ** .5).bfloat16()
    base = torch.randn(b * block, V + stride_pad, generator=g)
    anchor = torch.randint(0, V, (b,), generator=g)
    H = 512
    hidden = torch.randn(b * block, H, generator=g).bfloat16()
    conf_w = torch.randn(H + rank, generator=g) * .05
    conf_b = torch.tensor([.3])
    return W1, W2, base, anchor, hidden, conf_w, conf_b


CASES = [
    # V, rank, b, block, stride pad, fp32 bias
    (151936, 256, 1, 8, 0, False),    # the 35B-A3B vocabulary, Markov rank 256, block 8
    (1000, 64, 3, 5, 24, False),      # a partial last tile, padded logit rows
    (4096, 128, 16, 4, 0, False),     # the largest batch
    (2048, 512, 2, 16, 0, True),      # the largest rank, fp32 bias
]


@pytest.mark.parametrize("V,rank,b,block,pad,fp32", CASES)
def test_markov_equals_oracle(gpu, V, rank, b, block, pad, fp32):
    from snowllm_amd.draft_heads import MarkovHead
    _say(f"dspark markov V={V} rank={rank} b={b} block={block} pad={pad} fp32={fp32}")
    W1, W2, base, anchor, hidden, conf_w, conf_b = _markov_case(V, rank, b, block, V + rank, pad)
    if b == 16:
        anchor[3], anchor[7] = -1, V + 9        # outside the table: a zero latent
        base[5, :] = float("nan")               # a row of NaN: index 0
        base[6, 10:20] = 50.0                   # a plateau the bias decides
    head = MarkovHead(W1.cuda(), W2.cuda(), conf_w.cuda(), conf_b.cuda())
    path = torch.full((b, block), -7, dtype=torch.int64, device="cuda")
    conf = torch.full((b, block), -1.0, device="cuda")
    logits = base.cuda()[:, :V] if pad else base.cuda()
    head.propose(hidden.cuda(), logits, anchor.cuda(), path, conf, fp32_bias=fp32)
    torch.cuda.synchronize()
    want_path, want_conf = D.markov(base[:, :V].numpy(), _bits(W1), _bits(W2), anchor.numpy(),
                                    block, pre_head=_bits(hidden), conf_w=conf_w.numpy(),
                                    conf_b=float(conf_b), fp32_bias=fp32)
    assert np.array_equal(path.cpu().numpy(), want_path)
    assert np.abs(conf.cpu().double().numpy() - want_conf).max() < 1e-5
    if b == 16:
        assert path[1, 1].item() == 0 and 10 <= path[1, 2].item() < 20


@pytest.mark.parametrize("kind", ["plain", "-inf", "lowest", "equal", "zeros", "infinite", "tiny"])
@pytest.mark.parametrize("V,rank,b", [(77, 8, 16), (9000, 72, 5), (1290, 264, 3), (140000, 40, 1)])
def test_markov_bounds_keep_the_pick(gpu, V, rank, b, kind):
    """Ranks and vocabularies off the tile sizes, and rows whose bounds say little: masked logits,
    equal scores (more candidates than a workgroup sums one by one, and than it keeps), infinities,
    values below the normal range. The picks are the fp64 oracle's, bit for bit."""
    from snowllm_amd.draft_heads import MarkovHead
    _say(f"dspark markov bounds V={V} rank={rank} b={b} {kind}")
    block = 3
    W1, W2, base, anchor, *_ = _markov_case(V, rank, b, block, V + rank)
    if kind in ("-inf", "lowest"):
        low = float("-inf") if kind == "-inf" else torch.finfo(torch.float32).min
        base[:, :-3] = low
        base[1] = low                           # a row with nothing left
    elif kind == "equal":
        W2[:] = W2[0].clone()
        base[:] = 1.5
    elif kind == "zeros":
        W1.zero_(), base.zero_()
    elif kind == "infinite":
        W2[5, 1], W2[9, 3], base[0, 4], base[2, 6] = float("inf"), float("nan"), float("inf"), float("nan")
    elif kind == "tiny":
        W1[:], base[:] = W1 * 2.0 ** -133, base * 2.0 ** -20
        W2[:] = W2 * 2.0 ** 110
    head = MarkovHead(W1.cuda(), W2.cuda())
    path = torch.full((b, block), -7, dtype=torch.int64, device="cuda")
    head.propose(None, base.cuda(), anchor.cuda(), path)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        want = D.markov(base.numpy(), _bits(W1), _bits(W2), anchor.numpy(), block)
    want = want[0] if isinstance(want, tuple) else want
    assert np.array_equal(path.cpu().numpy(), want)


# ranks that end inside a 32-value step of every kernel form, vocabularies that end inside a 16-row
# unit (17 and 1 rows of the last 64-row tile)
@pytest.mark.parametrize("V,rank", [(1041, 8), (1041, 40), (1025, 72), (1041, 136), (1025, 264)])
def test_markov_does_not_read_past_the_weight(gpu, V, rank):
    """Chunks past the rank and rows past the vocabulary are zeros: NaN right behind the packed
    weight changes neither the picks nor which rows the bounds leave."""
    from snowllm_amd.draft_heads import MarkovHead
    _say(f"dspark markov end V={V} rank={rank}")
    b, block = 3, 4
    W1, W2, base, anchor, *_ = _markov_case(V, rank, b, block, V + rank)
    head = MarkovHead(W1.cuda(), W2.cuda())
    size = head.w2.numel() * head.w2.element_size()
    behind = torch.full((size + 65536,), 0xff, dtype=torch.uint8, device="cuda")
    behind[:size].copy_(head.w2.view(-1).view(torch.uint8))
    head.w2 = behind[:size].view(head.w2.dtype).view(head.w2.shape)
    path = torch.full((b, block), -7, dtype=torch.int64, device="cuda")
    head.propose(None, base.cuda(), anchor.cuda(), path)
    want = D.markov(base.numpy(), _bits(W1), _bits(W2), anchor.numpy(), block)
    want = want[0] if isinstance(want, tuple) else want
    assert np.array_equal(path.cpu().numpy(), want)


def test_markov_without_confidence_and_graph_replay(gpu):
    """No confidence output; the arrival counter carries across captured replays."""
    from snowllm_amd.draft_heads import MarkovHead
    V, rank, b, block = 4096, 256, 2, 8
    W1, W2, base, anchor, hidden, conf_w, conf_b = _markov_case(V, rank, b, block, 3)
    head = MarkovHead(W1.cuda(), W2.cuda())
    logits = torch.empty(b * block, V, device="cuda")
    anchors = anchor.cuda()
    path = torch.empty(b, block, dtype=torch.int64, device="cuda")
    logits.copy_(base)
    head.propose(None, logits, anchors, path)          # eager once (allocates the workspace)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        head.propose(None, logits, anchors, path)
    g = torch.Generator().manual_seed(11)
    for i in range(4):
        _say(f"markov graph replay {i}")
        fresh = torch.randn(b * block, V, generator=g)
        logits.copy_(fresh)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want, _ = D.markov(fresh.numpy(), _bits(W1), _bits(W2), anchor.numpy(), block)
        assert np.array_equal(path.cpu().numpy(), want)


@pytest.mark.parametrize("fmt,n", [(0, 8), (0, 24), (4, 8), (8, 40)])
def test_selector_hidden_projection(gpu, fmt, n):
    """hp = hidden W^T against fp32 (W bf16, or dequantised Q4_K / Q8_0), then the selector
    walk on the projected rows equals the C oracle's walk on them."""
    from snowllm_amd import dflash
    from snowllm_amd.draft_heads import SelectorHead
    from snowllm_amd.verify import gguf_random
    H, V, R = 2048, 4096, 256
    _say(f"selector hidden projection fmt={fmt} rows={n}")
    g = torch.Generator().manual_seed(n + fmt)
    hidden = (torch.randn(n, H, generator=g)).bfloat16()
    pred = (torch.randn(V, R, generator=g) * .2).bfloat16()
    succ = (torch.randn(V, R, generator=g) * .2).bfloat16()
    if fmt:
        raw = gguf_random(fmt, R, H, seed=n, centered=fmt == 4)
        w_ref = torch.from_numpy((Q.dequant_q4_k if fmt == 4 else Q.dequant_q8_0)(
            raw.cpu().numpy(), R, H))
        head = SelectorHead(H, raw, pred.cuda(), succ.cuda(), fmt=fmt)
    else:
        w = (torch.randn(R, H, generator=g) * H ** -.5).bfloat16()
        w_ref = w.float()
        head = SelectorHead(H, w.cuda(), pred.cuda(), succ.cuda())
    assert dflash.proj_shape(dflash.Proj.SELECTOR_HIDDEN) == (R, H)
    hp = head.project(hidden.cuda())
    torch.cuda.synchronize()
    ref = hidden.float() @ w_ref.T
    got = hp.float().cpu()
    rel = float((got - ref).norm() / ref.norm())
    _say(f"  hp rel L2 {rel:.2e} vs fp32")
    assert rel < 3e-3                                   # bf16 output rounding: ~1.1e-3
    assert float((got - ref.bfloat16().float()).norm() / ref.norm()) < 1e-3
    # the walk on the projected rows: n / 8 requests of 8 rows, greedy
    b = n // 8
    logits = torch.randn(n, V, generator=g).cuda()
    anchor = torch.arange(b, device="cuda") * 7 + 3
    path = torch.empty(b, 8, dtype=torch.int64, device="cuda")
    hp2 = head.propose(hidden.cuda(), logits, anchor, path)
    torch.cuda.synchronize()
    assert torch.equal(hp2, hp)
    want, _, _ = A.select(hp.cpu(), logits.cpu().numpy(), pred, succ, anchor.cpu().numpy())
    assert np.array_equal(path.cpu().numpy(), want)


def test_other_draft_projections_are_refused(gpu):
    from snowllm_amd import dflash
    from snowllm_amd.errors import SnowLLMError
    dflash.select(type("S", (), {"hidden": 2048})())
    for which in (dflash.Proj.FC, dflash.Proj.QKV, dflash.Proj.DOWN):
        with pytest.raises(SnowLLMError):
            dflash.proj_shape(which)
