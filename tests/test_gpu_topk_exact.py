"""The selection by exact scores: a block per lane (up to 64 blocks), tiles of 64 by 16 rows (up to 256) -- around
every size where the kernel changes, every remainder of the rows a wave takes, equal scores, scores that overflow, rows that pick
all blocks, against the oracle's scores; and the ring's order of age likewise."""
import pytest
import torch

from oracle import mem_cache as omc
from oracle import retrieval as oret
from oracle import rotary as orot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n,T,k", [(1, 17, 1), (2, 513, 2), (40, 530, 4), (63, 515, 63), (64, 516, 5), (64, 37, 64), (65, 514, 5), (128, 545, 16), (128, 545, 17), (129, 529, 3),
                                   (256, 515, 16), (200, 1026, 1), (257, 519, 4), (1000, 531, 64), (1024, 514, 1), (1025, 514, 5), (2300, 515, 64)])
def test_picks_match_the_oracle(n, T, k, D, dtype):
    from landmark_hip.retrieval import retrieve_topk
    print(f"case {n} blocks T{T} top {k} D{D} {dtype}", flush=True)
    B, H, block = 1, 2, 32
    g = torch.Generator().manual_seed(n + T)
    q = (torch.randn(B, H, T, D, generator=g) * 0.5).to(dtype)
    kc = (torch.randn(B, H, n * block, D, generator=g) * 0.5).to(dtype)
    cos, sin = orot.rotary_tables((n + k + 2) * block, D, dtype)
    idx = retrieve_topk(q.cuda(), kc.cuda(), cos.cuda(), sin.cuda(), block, k).cpu()
    want = oret.select_topk(oret.landmark_scores(q, kc, cos, sin, block, k), k)
    assert torch.equal(idx, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n", [2, 100, 300])
def test_quotients_of_every_value_rank_as_division_ranks_them(n, D, dtype):
    """Two blocks score a finite 16-bit number and the next one, the others the lowest: the second is picked where the quotients by
    sqrt(D), divided in fp32 and rounded, differ.  A quotient one place off would turn a tie into a difference, or the reverse."""
    from landmark_hip.retrieval import retrieve_topk
    block = 4
    bits = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype)
    x = x[x.isfinite()].float().sort().values.to(dtype)                 # -0 and +0 side by side
    q = torch.zeros(1, 1, x.numel() - 1, D, dtype=dtype)
    q[0, 0, :, 0], q[0, 0, :, 1], q[0, 0, :, 2] = x[:-1], x[1:], x[-1]
    kc = torch.zeros(1, 1, n * block, D, dtype=dtype)
    kc[0, 0, block - 1, 0], kc[0, 0, 2 * block - 1, 1], kc[0, 0, 3 * block - 1::block, 2] = 1, 1, -1
    cos, sin = torch.ones((n + 2) * block, D, dtype=dtype), torch.zeros((n + 2) * block, D, dtype=dtype)
    idx = retrieve_topk(q.cuda(), kc.cuda(), cos.cuda(), sin.cuda(), block, 1).cpu()[0, 0, :, 0]
    c = (x.float() / torch.tensor(float(D)).sqrt()).to(dtype)
    assert torch.equal(idx, (c[1:] > c[:-1]).long())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [50, 128, 200, 1024, 1100])
def test_equal_scores_go_to_the_lowest_block(n, dtype):
    from landmark_hip.retrieval import retrieve_topk
    q = torch.zeros(1, 1, 1030, 64, dtype=dtype)                # every score is zero, half of them negative
    kc = torch.randn(1, 1, n * 32, 64).to(dtype)
    cos, sin = orot.rotary_tables((n + 2) * 32, 64, dtype)
    idx = retrieve_topk(q.cuda(), kc.cuda(), cos.cuda(), sin.cuda(), 32, 6).cpu()
    assert torch.equal(idx, torch.arange(6).expand_as(idx))


@pytest.mark.parametrize("n", [60, 100, 250])
def test_scores_that_overflow(n):
    """fp16 scores of +-infinity rank like numbers, equal ones by block; a row of NaN picks blocks of the cache."""
    from landmark_hip.retrieval import retrieve_topk
    B, H, T, D, block, k = 1, 1, 1031, 64, 32, 7
    g = torch.Generator().manual_seed(n)
    q = (torch.randn(B, H, T, D, generator=g) * 100).half()
    kc = (torch.randn(B, H, n * block, D, generator=g) * 60).half()
    q[:, :, 9:12] *= 10
    q[:, :, 12] = -kc[:, :, block - 1, :].sign() * 60000            # block 0's score (and most others) far below the range
    cos, sin = orot.rotary_tables((n + 2) * block, D, torch.float16)
    want = oret.select_topk(oret.landmark_scores(q, kc, cos, sin, block, k), k)
    q[:, :, 20] = float("nan")
    idx = retrieve_topk(q.cuda(), kc.cuda(), cos.cuda(), sin.cuda(), block, k).cpu()
    keep = [t for t in range(T) if t != 20]
    assert torch.equal(idx[:, :, keep], want[:, :, keep])
    assert ((idx >= 0) & (idx < n)).all()


@pytest.mark.parametrize("n,oldest,T,k,block,D", [(1, 0, 3, 1, 32, 64), (40, 0, 255, 4, 51, 64), (64, 63, 130, 4, 51, 128),
                                                  (64, 17, 33, 64, 32, 64), (65, 17, 213, 4, 32, 64), (300, 299, 190, 4, 8, 128), (7, 3, 18, 7, 64, 128)])
def test_ring_picks_match_the_oracle(n, oldest, T, k, block, D):
    from landmark_hip import _lib
    print(f"case ring {n} blocks, oldest {oldest}, T{T} top {k} block {block} D{D}", flush=True)
    B, H = 2, 3
    g = torch.Generator().manual_seed(n + T)
    q = (torch.randn(B, H, T, D, generator=g) * 0.5).bfloat16()
    ring = (torch.randn(B, n, block, H, D, generator=g) * 0.5).bfloat16()
    cos, sin = orot.rotary_tables((k + 2) * block, D, torch.bfloat16)
    want = omc.select_blocks(omc.ring_scores(q, ring, n, oldest, k, cos, sin), oldest, k, "per_token_and_head")
    q, ring, cos, sin = (t.cuda() for t in (q, ring, cos, sin))
    kring = ring.flatten(1, 2).transpose(1, 2)
    lib = _lib.lib()
    nbytes = lib.lmk_retrieve_workspace_bytes(B, H, T, n * block, D, block)
    idx = torch.empty(B, H, T, k, device="cuda", dtype=torch.int64)
    ws = torch.empty(nbytes, device="cuda", dtype=torch.uint8)
    rc = lib.lmk_ring_retrieve_topk(_lib.tensor4(q), _lib.tensor4(kring), cos.data_ptr(), sin.data_ptr(), cos.stride(0), cos.shape[0],
                                    idx.data_ptr(), ws.data_ptr(), nbytes, B, H, T, n, D, block, k, oldest, 0, 0,
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(idx.cpu(), want)
