"""One selection per head or per query: vectors of every length around the kernels' sizes, rows that fit one workgroup and rows whose
maxima come in parts, against the oracle."""
import pytest
import torch

from oracle import mem_cache as omc
from oracle import retrieval as oret
from oracle import rotary as orot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,T,k", [(1, 1, 1), (64, 32, 64), (65, 33, 3), (256, 70, 8), (257, 31, 4), (257, 12, 4), (300, 13, 5),
                                   (1024, 129, 5), (1025, 5, 2), (2048, 34, 64), (2049, 34, 7)])
def test_per_head_picks_match_the_oracle(n, T, k, dtype):
    from landmark_hip.retrieval import retrieve_topk
    print(f"case per head: {n} blocks T{T} top {k} {dtype}", flush=True)
    B, H, D, block = 1, 2, 64, 16
    g = torch.Generator().manual_seed(n + T)
    q = (torch.randn(B, H, T, D, generator=g) * 0.5).to(dtype)
    kc = (torch.randn(B, H, n * block, D, generator=g) * 0.5).to(dtype)
    cos, sin = orot.rotary_tables((n + k + 2) * block, D, dtype)
    idx = retrieve_topk(q.cuda(), kc.cuda(), cos.cuda(), sin.cuda(), block, k, aggregate="max_over_tokens").cpu()
    want = oret.select_topk(oret.aggregate_max_over_tokens(oret.landmark_scores(q, kc, cos, sin, block, k)), k)
    assert torch.equal(idx.reshape(want.shape), want)


@pytest.mark.parametrize("method,code", [("max_over_heads", 1), ("max_over_tokens", 2)])
@pytest.mark.parametrize("n,oldest,H,T,k", [(1, 0, 3, 2, 1), (8, 3, 33, 5, 4), (64, 17, 12, 40, 4), (65, 64, 2, 33, 64), (300, 7, 32, 3, 5),
                                                  (270, 7, 32, 260, 3)])
def test_ring_picks_match_the_oracle(n, oldest, H, T, k, method, code):
    from landmark_hip import _lib
    print(f"case ring {method}: {n} blocks, oldest {oldest}, H{H} T{T} top {k}", flush=True)
    B, D, block = 2, 64, 8
    g = torch.Generator().manual_seed(n + T)
    q = (torch.randn(B, H, T, D, generator=g) * 0.5).bfloat16()
    ring = (torch.randn(B, n, block, H, D, generator=g) * 0.5).bfloat16()
    cos, sin = orot.rotary_tables((k + 2) * block, D, torch.bfloat16)
    want = omc.select_blocks(omc.ring_scores(q, ring, n, oldest, k, cos, sin), oldest, k, method)
    q, ring, cos, sin = (t.cuda() for t in (q, ring, cos, sin))
    lib = _lib.lib()
    nbytes = lib.lmk_retrieve_workspace_bytes(B, H, T, n * block, D, block)
    idx = torch.empty((B, T, k) if code == 1 else (B, H, k), device="cuda", dtype=torch.int64)
    ws = torch.full((nbytes,), 255, device="cuda", dtype=torch.uint8)
    rc = lib.lmk_ring_retrieve_topk(_lib.tensor4(q), _lib.tensor4(ring.flatten(1, 2).transpose(1, 2)), cos.data_ptr(), sin.data_ptr(),
                                    cos.stride(0), cos.shape[0], idx.data_ptr(), ws.data_ptr(), nbytes, B, H, T, n, D, block, k, oldest,
                                    code, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    idx = idx.cpu()
    assert torch.equal(idx[:, None].expand_as(want) if code == 1 else idx[:, :, None].expand_as(want), want)
