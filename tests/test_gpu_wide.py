"""GPU kernels over more than 16 rows at the edges of their tiles and dispatch rules: the bits of
the 16-row launches and the fp64 product."""
import pytest
import torch

from tests.test_gpu_batch import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt", [1, 2])
# two row groups with a short second one and a partial last tile; column tiles past the last of
# a workgroup; superblocks that do not divide over the waves (eight waves, then four)
@pytest.mark.parametrize("M,N,K", [(17, 2064, 3072), (113, 2000, 2304), (129, 2032, 4096),
                                   (145, 4112, 768), (250, 2050, 1024)])
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
