"""The decode step's gather: one block, several and as many as a row can pick, waves that walk one block and several, every
number of waves the rows ask for, a window of one token and of a whole block; first and last head against the oracle on the same
16-bit inputs (heads are independent).
"""
import pytest
import torch

from oracle import retrieval as oret
from oracle import rotary as orot

pytestmark = pytest.mark.gpu

TOL = 2e-2      # 16-bit weights, output and (oracle) rotated keys, values up to about 2

# B, H, T, cached blocks, cached tokens behind them, block, top_k, D
CASES = [(1, 3, T, n, tail, block, k, D)
         for D in (64, 128)
         for block in (32, 64, 128)
         for T, n, tail, k in ((1, 1, 0, 1), (1, 9, block - 1, 9), (4, 5, block - 4, 3), (2, 17, 16, 17))]
CASES += [(1, 2, 1, 70, 5, 32, 64, 64), (1, 2, 1, 66, 40, 64, 64, 128), (1, 2, 3, 300, 1, 32, 8, 128), (1, 2, 1, 9, 21, 128, 5, 128), (1, 2, 1, 11, 90, 128, 10, 128)]
CASES += [(B, 32, 1, 9, 21, block, 5, D) for B in (9, 17, 25, 33) for block, D in ((32, 128), (64, 64), (128, 128))]
CASES += [(33, 32, 2, 6, 3, 64, 4, 128), (33, 32, 2, 6, 3, 128, 4, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,T,n,tail,block,k,D", CASES)
def test_decode_step_matches_the_oracle(B, H, T, n, tail, block, k, D, dtype):
    from landmark_hip.retrieval import retrieve_and_attend
    print(f"case {B} {H} {T} {n} {tail} block {block} top {k} D{D} {dtype}", flush=True)
    S = n * block + tail
    g = torch.Generator().manual_seed(S + D + k)
    make = lambda rows: (torch.randn(B, H, rows, D, generator=g) * 0.5).to(dtype)
    q, kc, vc, kl, vl = (make(r) for r in (T, S, S, T, T))
    cos, sin = orot.rotary_tables(S + T, D, dtype)
    dev = [t.cuda() for t in (q, kc, vc, kl, vl, cos, sin)]
    out, idx = retrieve_and_attend(dev[0], (dev[1], dev[2]), *dev[3:], block, k)
    mem = ((torch.arange(T) + tail) % block == block - 1)[None]
    for b, h in {(0, 0), (B - 1, H - 1)}:
        s = (slice(b, b + 1), slice(h, h + 1))
        want, want_idx = oret.retrieve_and_attend(q[s], kc[s], vc[s], kl[s], vl[s], mem, cos, sin, block, k,
                                                   n_buckets=128)    # 64 hold the window's group and 63 picked blocks
        assert torch.equal(idx[s].cpu(), want_idx)
        assert (out[s].float().cpu() - want.float()).abs().max() <= TOL


@pytest.mark.parametrize("B,H,T,n,tail,block,D", [(1, 2, 1, 1, 5, 32, 64), (1, 3, 1, 3, 7, 64, 128), (1, 3, 1, 12, 7, 32, 64), (3, 11, 40, 1, 0, 64, 128),
                                                  (1, 3, 40, 2, 0, 32, 64)])
def test_a_first_block_behind_a_landmark_of_minus_infinity_weighs_nothing(B, H, T, n, tail, block, D):
    """Every block is picked; the landmark of block 0, the first a wave takes, scores -infinity for every query.  Decode steps (a wave
    for each block, for some of them) and chunks row by row (one row per wave, waves that share a row out)."""
    from landmark_hip.retrieval import gather_attend
    print(f"case {B} {H} {T} {n} {tail} block {block} D{D}", flush=True)
    S = n * block + tail
    g = torch.Generator().manual_seed(S + D)
    make = lambda rows: (torch.randn(B, H, rows, D, generator=g) * 0.5).bfloat16()
    q, kc, vc, kl, vl = (make(r) for r in (T, S, S, T, T))
    q = q.abs()
    kc[:, :, block - 1, 3] = -float("inf")                                  # both partners of its rotation by 0.5
    cos, sin = (f(torch.full((S + T, D), 0.5)).bfloat16() for f in (torch.cos, torch.sin))
    idx = torch.arange(n).expand(B, H, T, n).contiguous()
    mem = ((torch.arange(T) + tail) % block == block - 1)[None].expand(B, T)
    want, _ = oret.retrieve_and_attend(q, kc, vc, kl, vl, mem, cos, sin, block, n, idx=idx)
    out = gather_attend(*(t.cuda() for t in (q, kc, vc, idx, kl, vl, cos, sin)), block, n)
    assert (out.float().cpu() - want.float()).abs().max() <= TOL
