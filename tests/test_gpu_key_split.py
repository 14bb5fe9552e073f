"""The forward, dQ and dK/dV kernels with 64 rows per workgroup (blocks of 64 and 128 slots): both numbers of parts and the
kernels on the other side of the dispatch, at the edges of tiles, stages and blocks, against the fp32 oracle on
the same 16-bit inputs.  Heads are independent, so the first and the last stand for the rest.
"""
import pytest
import torch

from tests.util import make_qkv, oracle_forward, oracle_grads

pytestmark = pytest.mark.gpu

TOL = 2e-2

# B, H, Lq, Lk, D, block: few workgroups (four parts), more than compute units (two parts), more than they pay for (256 rows)
CASES = [(1, 2, n, n, D, block) for D, block in ((128, 64), (64, 64), (128, 128), (64, 128), (128, 51), (64, 100), (128, 2))
         for n in (1, block + 1, 4 * block, 5 * block + 33)]
CASES += [(1, 2, 70, 70 + 67 * 64, 128, 64), (1, 1, 40, 40 + 65 * 51, 64, 51)]     # more landmarks than one pass holds
CASES += [(6, 50, 97, 97, 128, 64), (6, 50, 130, 130 + 128, 64, 128), (6, 50, 140, 140, 128, 51), (5, 60, 300, 300, 64, 100)]
CASES += [(7, 55, 200, 200, 128, 64), (7, 55, 200, 328, 128, 128), (5, 41, 1089, 1089, 64, 64), (5, 41, 1000, 1000, 128, 51)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Lq,Lk,D,block", CASES)
def test_forward_matches_the_oracle_on_every_side_of_the_dispatch(B, H, Lq, Lk, D, block, dtype):
    from ltriton.flash_landmark_attention import fused_landmark_attention
    print(f"case {B} {H} {Lq} {Lk} D{D} block {block} {dtype}", flush=True)
    q, k, v = make_qkv(B, H, Lq, Lk, D, seed=Lk + D, dtype=dtype)
    with torch.no_grad():
        out = fused_landmark_attention(q.cuda(), k.cuda(), v.cuda(), None, block_size=block).float().cpu()
    for b, h in {(0, 0), (B - 1, H - 1)}:
        s = (slice(b, b + 1), slice(h, h + 1))
        want = oracle_forward(q[s], k[s], v[s], block)[0]
        assert (out[s] - want).abs().max() <= TOL


# the backward's kernels: the same two numbers of parts, and (last two) whole blocks of 64 with many long rows
GRAD_CASES = [(1, 2, n * block, n * block, D, block) for D, block in ((128, 64), (64, 64), (128, 128), (64, 128), (128, 51), (64, 100))
              for n in (1, 2, 5)]
GRAD_CASES += [(1, 2, 128, 128 + 3 * 64, 128, 64), (1, 1, 200, 1200, 64, 100)]
GRAD_CASES += [(6, 50, 128, 128, 128, 64), (6, 50, 128, 256, 64, 128), (6, 50, 153, 153, 128, 51), (5, 60, 300, 300, 64, 100)]
GRAD_CASES += [(2, 52, 1088, 1088, 128, 64), (2, 52, 1088, 1152, 64, 64)]
# dK/dV with 128 keys per workgroup: whole rounds of compute units, long walks of few workgroups; a history of several blocks
GRAD_CASES += [(4, 32, 512, 512, 128, 64), (1, 12, 4096, 4096, 64, 64), (1, 3, 256, 640, 128, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Lq,Lk,D,block", GRAD_CASES)
def test_gradients_match_the_oracle_on_every_side_of_the_dispatch(B, H, Lq, Lk, D, block, dtype):
    from ltriton.flash_landmark_attention import fused_landmark_attention
    print(f"case {B} {H} {Lq} {Lk} D{D} block {block} {dtype}", flush=True)
    q, k, v = make_qkv(B, H, Lq, Lk, D, seed=Lk + D, dtype=dtype)
    do = make_qkv(B, H, Lq, Lq, D, seed=Lk + D + 1, dtype=dtype)[0]
    qkv = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    out = fused_landmark_attention(*qkv, None, block_size=block)
    grads = [g.float().cpu() for g in torch.autograd.grad(out, qkv, do.cuda())]
    for b, h in {(0, 0), (B - 1, H - 1)}:
        s = (slice(b, b + 1), slice(h, h + 1))
        for got, want in zip(grads, oracle_grads(q[s], k[s], v[s], do[s], block)):
            assert (got[s] - want).abs().max() <= TOL
