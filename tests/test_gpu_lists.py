"""Candidate lists and rejection at the edges of their kernels' rules, bit-exact against the
oracle: lists within one workgroup (up to 1024) and wider ones, ties, masked rows, rows that the
LDS buffers do not hold, odd vocabularies (unaligned rows), and the search of draft tokens."""
import numpy as np
import pytest
import torch

from oracle import accept as A

pytestmark = pytest.mark.gpu


def _rows(V, seed):
    """Logit rows: plain, narrow (crowded probabilities), few distinct values (ties), masked by
    -inf, masked by the lowest value, all equal, one NaN and an infinity."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(7, V, generator=g) * 2
    x[1] *= 0.05
    x[2] = (x[2] * 2).round() / 2
    keep = torch.randperm(V, generator=g)[:max(1, V // 50)]
    for r, low in ((3, float("-inf")), (4, torch.finfo(torch.float32).min)):
        m = torch.full((V,), low)
        m[keep] = x[r, keep]
        x[r] = m
    x[5] = 1.25
    x[6, V // 3] = float("nan")
    x[6, V // 2] = float("-inf")
    return x


def _check(V, top_k, top_p, seed):
    _check_rows(_rows(V, seed), top_k, top_p)


def _check_rows(x, top_k, top_p):
    from snowllm_amd import ops
    n, V = x.shape
    width = max(min(k, V) if k > 0 else V for k in top_k)
    k = torch.tensor(top_k, dtype=torch.int32)
    p = torch.tensor(top_p)
    temp = torch.linspace(0.5, 1.5, n)
    out = torch.empty(n, width, device="cuda")
    ids = torch.empty(n, width, dtype=torch.int64, device="cuda")
    ws = torch.empty(ops.sample_workspace_bytes(n, V, width), dtype=torch.uint8, device="cuda")
    print(f"lists V={V} top_k={top_k} width={width}", flush=True)
    for _ in range(2):   # a second call on the used workspace
        ops.probabilities(x.cuda(), k.cuda(), p.cuda(), temp.cuda(), width, out, ids, ws)
    want_p, want_ids = A.probabilities(x.numpy(), k.numpy(), p.numpy(), temp.numpy(), width)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want_p.view(np.uint32))


@pytest.mark.parametrize("V", [3, 1024, 1030, 4099, 8195, 50257, 151936])
@pytest.mark.parametrize("k", [1, 20, 257, 1024])
def test_short_lists(gpu, V, k):
    _check(V, [min(k, V)] * 7, [0.9, 1.0, 0.95, 0.8, 0.7, 0.5, 0.99], V + k)


@pytest.mark.parametrize("V", [1030, 50257])
@pytest.mark.parametrize("k", [65, 100, 300, 1000])
def test_short_lists_of_several_waves_cut_by_top_p(gpu, V, k):
    """More list slots than one wave holds (and fewer than the workgroup's threads), cut within the
    first wave, at its end and waves later: the prefix scan and the kept sum run in every wave."""
    _check(V, [k] * 7, [0.02, 0.3, 0.001, 0.1, 0.6, 64.0 / k, 0.9], V + k)


@pytest.mark.parametrize("V", [1100, 8193, 32000, 151937])
def test_wide_lists(gpu, V):
    """The whole vocabulary with top-p, widths between, short lists beside them."""
    _check(V, [0, V, 0, 1025, 0, 0, 0], [0.9, 0.5, 0.95, 1.0, 0.8, 0.3, 0.999], V)
    _check(V, [1026, 20, V - 1, 0, 0, 1050, 7], [0.9, 0.5, 1.0, 0.9, 1.0, 0.95, 1.0], V + 1)


@pytest.mark.parametrize("V", [12000, 50257, 151936])
def test_wide_lists_of_crowded_rows(gpu, V):
    """More nearly equal probabilities than a workgroup sorts in LDS, so that several share a range:
    distinct ones in one bucket and in neighbouring ones, a few values many times each, two heavy
    values, one value, and one beside a peak."""
    g = torch.Generator().manual_seed(V)
    x = torch.randn(8, V, generator=g)
    x[0] *= 0.001
    x[1] *= 0.01
    x[2] *= 0.0001
    x[3] = (x[3] * 2).round() * 0.003
    x[4] = torch.where(torch.rand(V, generator=g) < 0.5, 0.0, -0.004)
    x[5] = 1.25
    x[6] = torch.where(torch.arange(V) == V // 3, 40.0, 0.0)
    x[7] = torch.where(torch.rand(V, generator=g) < 0.7, 1.0, 0.05 * x[7])
    _check_rows(x, [0] * 8, [0.9, 0.5, 0.95, 0.3, 0.8, 0.6, 0.999, 0.7])
    _check_rows(x, [V - 5, 1500, V, 9000, 0, 2000, 11000, 0], [1.0, 0.9, 0.2, 1.0, 0.99, 1.0, 0.9, 1.0])


@pytest.mark.parametrize("k", [200, 1000])
def test_short_lists_of_many_candidates(gpu, k):
    """Large distinct values in a few threads' words: more elements lie above the threshold than LDS
    holds, and the exact selection takes over (k at or below 256 keeps one key per thread, two
    above)."""
    V = 151936
    g = torch.Generator().manual_seed(k)
    x = torch.randn(2, V, generator=g)
    heavy = (torch.arange(V) // 4) % 1024 < 150
    x = torch.where(heavy, x.abs() + 6, x)
    _check_rows(x, [k, k], [1.0, 0.9])


@pytest.mark.parametrize("p_width,q_width", [(1, 16), (20, 16), (4096, 16), (4097, 70), (9000, 9000)])
def test_reject_searches(gpu, p_width, q_width):
    """Draft tokens in unordered lists, present, absent and repeated (their sum), with stale
    proposals, at the widths where the search changes form."""
    from snowllm_amd import ops
    g = torch.Generator().manual_seed(p_width + q_width)
    b, k, V = 5, 4, 20000
    p = torch.rand(b * (k + 1), p_width, generator=g)
    p /= p.sum(-1, keepdim=True)
    ids = torch.stack([torch.randperm(V, generator=g)[:p_width] for _ in range(b * (k + 1))])
    cand = torch.stack([torch.randperm(V, generator=g)[:q_width] for _ in range(b * k)])
    q = torch.rand(b * k, q_width, generator=g)
    q /= q.sum(-1, keepdim=True)
    rows = [r * (k + 1) + j for r in range(b) for j in range(k)]
    drafts = ids[rows][:, p_width // 2].clone()         # in the target's list
    cand[:, q_width // 3] = drafts                      # and in the proposal's
    drafts[1], drafts[6] = V + 5, -1                    # nowhere
    if p_width > 8:
        ids[0, 3] = ids[0, p_width - 2] = drafts[0]     # repeated ids add up
    ids[2 * (k + 1)] = torch.arange(p_width)            # a list in vocabulary order
    drafts[2 * k] = p_width - 1
    args = [p, ids, drafts.view(b, k), cand.view(b, k, q_width), q.view(b, k, q_width),
            torch.tensor([4, 3, 2, 1, 0], dtype=torch.int32),
            torch.tensor([1, 1, 1, 0, 1], dtype=torch.int32)]
    out = torch.empty(b, k + 1, dtype=torch.int64, device="cuda")
    acc = torch.empty(b, dtype=torch.int64, device="cuda")
    for u in (torch.rand(b, k + 1, generator=g), torch.rand(b, k + 1, generator=g) * 0.02,
              torch.zeros(b, k + 1)):
        print(f"reject p_width={p_width} q_width={q_width}", flush=True)
        ops.dflash.reject(*[x.cuda() for x in args], u.cuda(), out, acc)
        want, wacc = A.reject(*[x.numpy() for x in args], u.numpy())
        assert np.array_equal(acc.cpu().numpy(), wacc)
        assert np.array_equal(out.cpu().numpy(), want)


def test_reject_of_a_block_past_the_search_array(gpu):
    """A block of more draft rows than the array of matches holds, with target lists wider than a
    chunk: the waves search the lists themselves."""
    from snowllm_amd import ops
    k, p_width, q_width = 2060, 4097, 16
    g = torch.Generator().manual_seed(5)
    print(f"reject block={k} p_width={p_width}", flush=True)
    p = torch.rand(k + 1, p_width, generator=g)
    p /= p.sum(-1, keepdim=True)
    ids = (torch.arange(p_width) * 5 + torch.arange(k + 1).unsqueeze(1) * 3) % 30000
    drafts = ids[torch.arange(k), torch.randint(0, p_width, (k,), generator=g)].view(1, k).clone()
    cand = torch.randint(0, 30000, (1, k, q_width), generator=g)
    cand[0, :, 3] = drafts[0]
    q = torch.rand(1, k, q_width, generator=g) * 1e-4
    one = torch.ones(1, dtype=torch.int32)
    args = [p, ids.contiguous(), drafts, cand, q, one * 0, one]
    out = torch.empty(1, k + 1, dtype=torch.int64, device="cuda")
    acc = torch.empty(1, dtype=torch.int64, device="cuda")
    u = torch.rand(1, k + 1, generator=g)
    for u in (u * 1e-3, u, u * 0.0):
        ops.dflash.reject(*[x.cuda() for x in args], u.cuda(), out, acc)
        want, wacc = A.reject(*[x.numpy() for x in args], u.numpy())
        assert np.array_equal(acc.cpu().numpy(), wacc)
        assert np.array_equal(out.cpu().numpy(), want)
