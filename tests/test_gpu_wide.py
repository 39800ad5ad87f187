"""GPU kernels over more than 16 rows at the edges of their tiles and dispatch rules: the bits of
the 16-row launches and the fp64 product."""
import numpy as np
import pytest
import torch

from tests.test_gpu_batch import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt", [1, 2])
# two row groups with a short second one and a partial last tile; column tiles past the last of
# a workgroup; superblocks that do not divide over the waves (eight waves, then four); the two
# sides of the narrow outputs' rule (4096 columns) at two, three and five row tiles
@pytest.mark.parametrize("M,N,K", [(17, 2064, 3072), (113, 2000, 2304), (129, 2032, 4096),
                                   (145, 4112, 768), (250, 2050, 1024), (32, 4096, 2304),
                                   (17, 4112, 768), (33, 4096, 2048), (33, 4112, 2304),
                                   (72, 4080, 768), (65, 4100, 4096)])
def test_dense_gemv_wide_edges(gpu, wt, M, N, K):
    from snowllm_amd import layers as L, ops
    print(f"dense_gemv wide wt={wt} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.02).to(
        torch.float16 if wt == 1 else torch.bfloat16)
    packed = L.dense_shuffle(w)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    x[0] *= 1e4   # rows of different operand scales
    act = x
    if wt == 1:
        act = torch.empty(ops.gemm_kquant_a_ws_bytes(M, K), dtype=torch.uint8, device="cuda")
        ops.gemm_kquant_prepare_a(x, act)
    out = torch.full((M, N), float("nan"), device="cuda")
    L.dense_gemv(wt, packed, act, out, M, N, K)
    tiles = torch.empty_like(out)
    tb = ops.gemm_kquant_a_ws_bytes(16, K)
    for r0 in range(0, M, 16):
        n = min(16, M - r0)
        L.dense_gemv(wt, packed, act[(r0 // 16) * tb:] if wt == 1 else x[r0:r0 + n],
                     tiles[r0:r0 + n], n, N, K)
    torch.cuda.synchronize()
    assert torch.equal(out, tiles)
    # exact products summed in 32 bits: K roundings of 2^-24 at most
    assert rel(out.cpu(), x.double().cpu() @ w.double().cpu().T) < K * 2.0 ** -24


@pytest.mark.parametrize("wt", [1, 2])
# up to 16 rows of a head's columns, at the edge of that rule: the bits of the narrow launches;
# a lone last tile, a partial one, waves without a superblock, several superblocks per wave
@pytest.mark.parametrize("M,N,K", [(1, 65520, 256), (9, 65521, 768), (16, 65536, 2304),
                                   (13, 65550, 2048)])
def test_dense_gemv_of_a_head(gpu, wt, M, N, K):
    from snowllm_amd import layers as L, ops
    print(f"dense_gemv head wt={wt} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.02).to(
        torch.float16 if wt == 1 else torch.bfloat16)
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    x[0] *= 1e4   # rows of different operand scales
    act = x
    if wt == 1:
        act = torch.empty(ops.gemm_kquant_a_ws_bytes(M, K), dtype=torch.uint8, device="cuda")
        ops.gemm_kquant_prepare_a(x, act)
    out = torch.full((M, N), float("nan"), device="cuda")
    L.dense_gemv(wt, L.dense_shuffle(w), act, out, M, N, K)
    for n0 in range(0, N, 32768):
        n = min(32768, N - n0)
        part = torch.empty(M, n, device="cuda")
        L.dense_gemv(wt, L.dense_shuffle(w[n0:n0 + n].contiguous()), act, part, M, n, K)
        assert torch.equal(out[:, n0:n0 + n], part)
    # exact products summed in 32 bits: K roundings of 2^-24 at most
    assert rel(out.cpu(), x.double().cpu() @ w.double().cpu().T) < K * 2.0 ** -24


@pytest.mark.parametrize("m", [16, 33])
def test_q6k_every_scale_is_exact(gpu, m):
    """Q6_K scales over the whole of int8 against quants 0, 63 and random ones: rows with a single
    1 read single weights d sc (q - 32), whose integer part is exact, so one rounding is left."""
    from oracle import quant as Q
    from snowllm_amd import ops
    n, k = 64, 1024
    print(f"q6k scales m={m}", flush=True)
    raw = Q.make_q6_k(n, k, seed=m)
    b = raw.reshape(-1, 210)
    b[:, 192:208] = np.arange(b.shape[0] * 16, dtype=np.uint8).reshape(-1, 16)
    b[0::3, :192], b[1::3, :192] = 0x00, 0xff
    x = torch.zeros(m, k)
    at = (torch.arange(m) * 37) % k
    x[torch.arange(m), at] = 1.0
    quant, meta = ops.gemm_kquant_shuffle_b(6, torch.from_numpy(raw).cuda(), n, k)
    ws = torch.empty(ops.gemm_kquant_a_ws_bytes(m, k), dtype=torch.uint8, device="cuda")
    out = torch.empty(m, n, device="cuda")
    ops.gemm_kquant_a(6, x.bfloat16().cuda(), quant, meta, out, m, n, k, ws)
    torch.cuda.synchronize()
    want = torch.from_numpy(Q.dequant(raw, 6, n, k)).double()[:, at].T
    assert ((out.cpu().double() - want).abs() <= want.abs() * 2.0 ** -23).all()


@pytest.mark.parametrize("fmt", [4, 5, 6, 8])
@pytest.mark.parametrize("m,n,k", [(235, 2000, 4096), (241, 2000, 4352), (200, 2000, 4096),
                                   (113, 2000, 4352), (33, 2000, 4352), (250, 2000, 2048),
                                   (113, 2000, 2048), (200, 6160, 1280), (33, 512, 512)])
def test_wide_rows_equal_single_row_tiles(gpu, fmt, m, n, k):
    """Blocks of two row tiles by four or two column tiles (a last pair of one tile, a last group
    of one column tile, waves with one, two and three superblocks), and blocks of one row tile (eight
    and four waves) against 16-row calls, bit for bit."""
    from oracle import quant as Q
    from snowllm_amd import ops
    print(f"wide rows fmt={fmt} m={m} n={n} k={k}", flush=True)
    make = {4: Q.make_q4_k, 5: Q.make_q5_k, 6: Q.make_q6_k, 8: Q.make_q8_0}[fmt]
    quant, meta = ops.gemm_kquant_shuffle_b(fmt, torch.from_numpy(make(n, k, seed=m)).cuda(), n, k)
    x = Q.make_activations(m, k, seed=k).cuda()
    ws = torch.empty(ops.gemm_kquant_a_ws_bytes(m, k), dtype=torch.uint8, device="cuda")
    out, want = torch.empty(m, n, device="cuda"), torch.empty(m, n, device="cuda")
    ops.gemm_kquant_a(fmt, x, quant, meta, out, m, n, k, ws)
    for r in range(0, m, 16):
        c = min(16, m - r)
        ops.gemm_kquant_a(fmt, x[r:r + c], quant, meta, want[r:r + c], c, n, k,
                          ws[:ops.gemm_kquant_a_ws_bytes(c, k)])
    assert torch.equal(out, want)


@pytest.mark.parametrize("fmt", [4, 5, 6, 8])
# one launch at the depths that the 16-row kernel has unrolled forms for (8 and 16 superblocks: odd
# pair counts, a last row tile of one row) and around them; the sizes where the rule changes sides
@pytest.mark.parametrize("m,f,k", [(57, 272, 4096), (113, 144, 2048), (113, 1040, 1280),
                                   (256, 16, 256), (33, 176, 512), (17, 272, 4096),
                                   (33, 144, 2048), (33, 12400, 512), (20, 12288, 4096),
                                   (45, 6144, 2048)])
def test_gate_up_rows_equal_row_chunks(gpu, fmt, m, f, k):
    """Gate/up over many rows in one launch (a last pair of one row tile, a last group of one
    column pair, a wave without a superblock) against 16-row launches, bit for bit, and against the
    fp64 products with the projections rounded to bf16."""
    from oracle import quant as Q
    from snowllm_amd import layers as L, ops
    print(f"gate_up rows fmt={fmt} m={m} f={f} k={k}", flush=True)
    make = {4: Q.make_q4_k, 5: Q.make_q5_k, 6: Q.make_q6_k, 8: Q.make_q8_0}[fmt]
    host = make(2 * f, k, seed=m)
    quant, meta = ops.gemm_kquant_shuffle_b(fmt, torch.from_numpy(host).cuda(), 2 * f, k)
    x = Q.make_activations(m, k, seed=k).cuda()
    ws = torch.empty(ops.gemm_kquant_a_ws_bytes(m, k), dtype=torch.uint8, device="cuda")
    ops.gemm_kquant_prepare_a(x, ws)
    out = torch.empty(m, f, dtype=torch.bfloat16, device="cuda")
    want = torch.empty_like(out)
    L.gate_up_swiglu_rows(fmt, quant, meta, ws, out, m, f, k)
    tile = ops.gemm_kquant_a_ws_bytes(16, k)
    for r in range(0, m, 16):
        c = min(16, m - r)
        L.gate_up_swiglu(fmt, quant, meta, ws[r // 16 * tile:], want[r:r + c], c, f, k)
    assert torch.equal(out, want)
    if f <= 1040:
        w = torch.from_numpy(Q.dequant(host, fmt, 2 * f, k)).double()
        y = (x.cpu().double() @ w.T).bfloat16().double()
        exact = y[:, :f] * torch.sigmoid(y[:, :f]) * y[:, f:]
        # the result's rounding to bf16 is 2^-9 at most; a projection that rounds the other way
        # shifts its element by 2^-8, rarely
        assert rel(out.cpu(), exact) < 2.0 ** -8
