"""Gather + attend by block against float64 and against the gather by row, through the C ABI: groups of one and of several
picks of a rank, more picks than one search holds, more rows than the workspace holds, blocks of every slot count, a ring
that has wrapped, shared selections, indices outside the cache.
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# B, H, T, n_blocks, block, k, D, ring_start, method (0 a selection per row, 1 shared by the heads, 2 by the queries), dtype
CASES = [
    (1, 32, 65, 8, 64, 4, 128, 0, 0, torch.bfloat16),
    (1, 32, 130, 9, 32, 4, 128, 5, 0, torch.bfloat16),
    (2, 12, 255, 40, 51, 4, 64, 13, 0, torch.float16),
    (1, 8, 140, 5, 128, 5, 128, 0, 0, torch.float16),          # every block picked by every row
    (1, 8, 500, 7, 100, 3, 64, 6, 0, torch.bfloat16),
    (1, 16, 65, 64, 33, 64, 64, 1, 0, torch.bfloat16),         # the most ranks there are
    (1, 32, 600, 70, 32, 4, 64, 0, 0, torch.bfloat16),         # more picks than one search holds
    (1, 33, 1000, 24, 64, 16, 128, 0, 0, torch.bfloat16),      # more rows than the workspace holds
    (2, 12, 255, 40, 51, 4, 64, 39, 1, torch.bfloat16),
    (2, 12, 255, 40, 51, 4, 64, 39, 2, torch.bfloat16),
    (1, 40, 257, 6, 128, 1, 64, 2, 2, torch.float16),
    (1, 16, 512, 3, 2, 3, 128, 0, 0, torch.bfloat16),          # too little to read for a second launch: by row
]


def _float64(q, k, v, idx, cos, sin, o_loc, L, M, block, start, heads):
    """What the rows of `heads` attend to: the picked blocks in float64, merged with the local window."""
    n, D = k.shape[2] // block, k.shape[-1]
    top_k = idx.shape[-1]
    out = torch.empty(len(heads), q.shape[2], D, dtype=torch.float64, device=q.device)
    tok = torch.arange(block, device=q.device)
    for i, (b, h) in enumerate(heads):
        rows = idx[b, h].clamp(0, n - 1)                                             # (T, k)
        newest = ((rows - start) % n) >= n - top_k
        pos = (torch.arange(top_k, device=q.device)[None] + newest)[..., None] * block + tok        # (T, k, block)
        kb, vb = (x[b, h].double().view(n, block, D)[rows] for x in (k, v))          # (T, k, block, D)
        half = torch.cat((-kb[..., D // 2:], kb[..., :D // 2]), -1)
        kb = kb * cos.double()[pos] + half * sin.double()[pos]
        s = (kb @ q[b, h].double()[:, None, :, None])[..., 0] / math.sqrt(D)         # (T, k, block)
        inner = (s[..., :-1].softmax(-1)[..., None] * vb[..., :-1, :]).sum(-2)       # (T, k, D)
        w = torch.cat((s[..., -1], (M[b, h] + L[b, h].log()).double()[:, None]), -1).softmax(-1)
        out[i] = (w[:, :-1, None] * inner).sum(1) + w[:, -1:] * o_loc[b, h].double()
    return out


@pytest.mark.parametrize("B,H,T,n,block,k,D,start,method,dtype", CASES)
def test_gather_by_block_is_as_exact_as_the_gather_by_row(B, H, T, n, block, k, D, start, method, dtype):
    from landmark_hip import _lib
    print(f"case {B} {H} {T} {n} {block} {k} D{D} start {start} method {method} {dtype}", flush=True)
    lib, dev = _lib.lib(), torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(T + n)
    make = lambda *shape: torch.randn(*shape, device=dev, generator=g).mul_(0.7).to(dtype)
    q, o_loc = make(B, H, T, D), make(B, H, T, D)
    kc, vc = make(B, H, n * block, D), make(B, H, n * block, D)
    M = torch.randn(B, H, T, device=dev, generator=g)
    L = torch.rand(B, H, T, device=dev, generator=g) * 20 + 1
    angle = torch.outer(torch.arange((k + 1) * block, device=dev).float(), 1e4 ** (-torch.arange(0, D, 2, device=dev).float() / D))
    cos, sin = (torch.cat((x, x), -1).to(dtype) for x in (angle.cos(), angle.sin()))
    shape = ((B, H, T), (B, T), (B, H))[method]
    idx = torch.rand(*shape, n, device=dev, generator=g).argsort(-1)[..., :k].sort(-1).values.contiguous()
    idx.view(-1)[0], idx.view(-1)[-1] = -3, n + 5                                    # read as the first and the last block
    out = [torch.empty_like(q) for _ in range(2)]
    need = lib.lmk_gather_blocks_workspace_bytes(B, H, T, n, D, block, k, int(method == 2))
    assert (need == 0) == (block == 2)
    if need:
        assert need <= (256 << 20) + 256 and (need < B * H * T * k * (D + 1) * 4) == (T == 1000)
    ws = torch.empty(max(need, 16), device=dev, dtype=torch.uint8)
    for i, nbytes in enumerate((0, need)):
        _lib.check(lib.lmk_ring_gather_attend_blocks(
            _lib.tensor4(q), _lib.tensor4(kc), _lib.tensor4(vc), idx.data_ptr(), cos.data_ptr(), sin.data_ptr(), cos.stride(0),
            cos.shape[0], _lib.tensor4(o_loc), L.data_ptr(), M.data_ptr(), T, _lib.tensor4(out[i]), ws.data_ptr(), nbytes, B, H, T, n,
            D, 1 / math.sqrt(D), block, k, start, method, _lib.DTYPE_CODES[dtype], _lib.current_stream(dev)))
    rows = (idx, idx[:, None], idx[:, :, None])[method].expand(B, H, T, k)
    heads = sorted({(0, 0), (B - 1, H - 1)})
    want = _float64(q, kc, vc, rows, cos, sin, o_loc, L, M, block, start, heads)
    by_row, by_block = ((torch.stack([o[b, h] for b, h in heads]).double() - want) for o in out)
    # both round the weights and the output to 16 bits: 2^-9 (2^-12) of values up to about 3
    bound = 2e-2 if dtype == torch.bfloat16 else 2.5e-3
    assert by_block.abs().max() <= bound
    assert by_block.norm() <= 1.01 * by_row.norm()
    print("error by row / by block", (by_row.norm() / want.norm()).item(), (by_block.norm() / want.norm()).item(), flush=True)


@pytest.mark.parametrize("dtype,q_scale,k_scale", [(torch.bfloat16, 60, 60), (torch.float16, 60, 60), (torch.float16, 8000, 0.25),
                                                   (torch.float16, 8000, 2.0 ** -12)])       # parts below the normal numbers
def test_rotated_keys_keep_the_bits_of_fp32(dtype, q_scale, k_scale):
    """Scores in the thousands that differ by a few: a key's bits below 16 decide the weights.  One rotation for all positions, keys
    that are a common vector but for a place in some dimensions.  2^-17 of a product of 3600 would move a weight by 2 to 3 %."""
    from landmark_hip import _lib
    print(f"case {dtype} q {q_scale} k {k_scale}", flush=True)
    lib, dev = _lib.lib(), torch.device("cuda")
    B, H, T, n, block, k, D = 1, 16, 130, 6, 64, 4, 128
    g = torch.Generator(device=dev).manual_seed(7)
    q = torch.randn(B, H, T, D, device=dev, generator=g).mul_(q_scale).to(dtype)
    common = torch.randn(B, H, 1, D, device=dev, generator=g).mul_(k_scale).to(dtype).expand(B, H, n * block, D)
    step = (torch.rand(B, H, n * block, D, device=dev, generator=g) < 1 / 64).to(torch.int16)
    kc = (common.contiguous().view(torch.int16) + step).view(dtype)                  # the next number up or down
    vc = torch.randn(B, H, n * block, D, device=dev, generator=g).to(dtype)
    o_loc = torch.randn(B, H, T, D, device=dev, generator=g).to(dtype)
    angle = torch.rand(D // 2, device=dev, generator=g).mul_(6.28).repeat(2).expand((k + 1) * block, D)
    cos, sin = angle.cos().to(dtype).contiguous(), angle.sin().to(dtype).contiguous()
    idx = torch.rand(B, H, T, n, device=dev, generator=g).argsort(-1)[..., :k].sort(-1).values.contiguous()
    # the local window weighs as much as a picked block
    half = torch.cat((-common[..., :1, D // 2:], common[..., :1, :D // 2]), -1)
    M = (q.double() * (common[..., :1, :].double() * cos[0].double() + half.double() * sin[0].double())).sum(-1).div(math.sqrt(D)).float()
    L = torch.ones_like(M)
    out = [torch.empty_like(q) for _ in range(2)]
    need = lib.lmk_gather_blocks_workspace_bytes(B, H, T, n, D, block, k, 0)
    assert need > 0
    ws = torch.empty(need, device=dev, dtype=torch.uint8)
    for o, nbytes in zip(out, (0, need)):
        _lib.check(lib.lmk_ring_gather_attend_blocks(
            _lib.tensor4(q), _lib.tensor4(kc), _lib.tensor4(vc), idx.data_ptr(), cos.data_ptr(), sin.data_ptr(), cos.stride(0),
            cos.shape[0], _lib.tensor4(o_loc), L.data_ptr(), M.data_ptr(), T, _lib.tensor4(o), ws.data_ptr(), nbytes, B, H, T, n, D,
            1 / math.sqrt(D), block, k, 0, 0, _lib.DTYPE_CODES[dtype], _lib.current_stream(dev)))
    heads = [(0, h) for h in range(0, H, 5)]
    want = _float64(q, kc, vc, idx, cos, sin, o_loc, L, M, block, 0, heads)
    by_row, by_block = ((torch.stack([o[b, h] for b, h in heads]).double() - want).norm() / want.norm() for o in out)
    print("error by row / by block", by_row.item(), by_block.item(), flush=True)
    # what they share is the rounding of weights and output to 16 bits, and sums of fp32 in two orders
    assert by_block <= 1.02 * by_row


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_keys_that_are_not_finite(dtype):
    """Infinite keys, NaN and the type's largest values: the rows they make NaN, and those whose weights they only take to 0 or 1."""
    from landmark_hip import _lib
    lib, dev = _lib.lib(), torch.device("cuda")
    B, H, T, n, block, k, D = 1, 16, 130, 6, 64, 4, 128
    g = torch.Generator(device=dev).manual_seed(3)
    make = lambda *shape: torch.randn(*shape, device=dev, generator=g).to(dtype)
    q, kc, vc, o_loc = make(B, H, T, D), make(B, H, n * block, D), make(B, H, n * block, D), make(B, H, T, D)
    inf, most = float("inf"), min(torch.finfo(dtype).max, 1e36)                                # sums of it stay finite
    kc[:, 0, 5, 9], kc[:, 1, block + 7, 100], kc[:, 2, 2 * block - 1, 3] = inf, -inf, inf     # the last a landmark
    kc[:, 3, 20, 30], kc[:, 4, 3 * block + 1, 64] = float("nan"), -float("nan")
    kc[:, 5, 70, 17], kc[:, 6, 2 * block + 9, 1], kc[:, 7, 6 * block - 1, 90] = most, -most, -most
    kc[:, 8, 33, 8], kc[:, 8, 33, 72] = inf, -inf                                             # both partners of a rotation
    M, L = torch.zeros(B, H, T, device=dev), torch.ones(B, H, T, device=dev)
    angle = torch.outer(torch.arange((k + 1) * block, device=dev).float() + 1, 1e2 ** (-torch.arange(0, D, 2, device=dev).float() / D))
    cos, sin = (torch.cat((x, x), -1).to(dtype) for x in (angle.cos(), angle.sin()))
    idx = torch.rand(B, H, T, n, device=dev, generator=g).argsort(-1)[..., :k].sort(-1).values.contiguous()
    need = lib.lmk_gather_blocks_workspace_bytes(B, H, T, n, D, block, k, 0)
    assert need > 0
    ws, out = torch.empty(need, device=dev, dtype=torch.uint8), [torch.empty_like(q) for _ in range(2)]
    for o, nbytes in zip(out, (0, need)):
        _lib.check(lib.lmk_ring_gather_attend_blocks(
            _lib.tensor4(q), _lib.tensor4(kc), _lib.tensor4(vc), idx.data_ptr(), cos.data_ptr(), sin.data_ptr(), cos.stride(0),
            cos.shape[0], _lib.tensor4(o_loc), L.data_ptr(), M.data_ptr(), T, _lib.tensor4(o), ws.data_ptr(), nbytes, B, H, T, n, D,
            1 / math.sqrt(D), block, k, 0, 0, _lib.DTYPE_CODES[dtype], _lib.current_stream(dev)))
    by_row, by_block = (o.double() for o in out)
    print("rows with NaN, of", T, by_row.isnan().any(-1).sum(-1).tolist(), by_block.isnan().any(-1).sum(-1).tolist(), flush=True)
    same = torch.equal(by_row.isnan()[:, torch.arange(H) != 2], by_block.isnan()[:, torch.arange(H) != 2])
    assert same and bool(by_row[:, :5].isnan().any()) and bool(by_row[:, :2].isfinite().any())
    # a landmark of -infinity takes its block's weight to 0; row by row its row is NaN if it is the first
    assert not bool((by_block.isnan() & ~by_row.isnan()).any())
    finite = by_row.isfinite()
    worst = (by_row - by_block)[finite].abs().max().item()
    assert worst <= (3e-2 if dtype == torch.bfloat16 else 4e-3)     # two roundings to 16 bits of values up to 4


# The same kernels behind the flat cache's entry points: B, H, T, cached blocks, tokens behind them, block, top_k, D.  Rows that select by
# slices, and others; chunks longer than a block, chunks behind a tail; every row stride of the window and its statistics counts.
FLAT = [(1, 8, 128, 60, 0, 32, 8, 128), (1, 32, 256, 128, 0, 64, 4, 128), (1, 32, 64, 6, 40, 128, 4, 128), (3, 32, 24, 4, 8, 32, 4, 128),
        (2, 37, 31, 4, 1, 32, 4, 128), (2, 32, 300, 20, 0, 64, 4, 64), (1, 12, 333, 70, 0, 128, 3, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,T,n,tail,block,k,D", FLAT)
def test_flat_cache_by_block_matches_the_oracle(B, H, T, n, tail, block, k, D, dtype):
    from landmark_hip import _lib
    from landmark_hip.retrieval import gather_attend, retrieve_and_attend
    from oracle import retrieval as oret
    from oracle import rotary as orot
    print(f"case {B} {H} {T} {n} {tail} block {block} top {k} D{D} {dtype}", flush=True)
    assert _lib.lib().lmk_gather_blocks_workspace_bytes(B, H, T, n, D, block, k, 0) > 0
    S = n * block + tail
    g = torch.Generator().manual_seed(S + D + k)
    make = lambda rows: (torch.randn(B, H, rows, D, generator=g) * 0.5).to(dtype)
    q, kc, vc, kl, vl = (make(r) for r in (T, S, S, T, T))
    cos, sin = orot.rotary_tables(S + T, D, dtype)
    dev = [t.cuda() for t in (q, kc, vc, kl, vl, cos, sin)]
    out, idx = retrieve_and_attend(dev[0], (dev[1], dev[2]), *dev[3:], block, k)
    apart = gather_attend(*dev[:3], idx, *dev[3:], block, k)
    assert torch.equal(apart, out)
    rows = sorted({0, 1, T // 2, T - 2, T - 1, min(T - 1, block - 1), min(T - 1, block)})
    for b, h in {(0, 0), (B - 1, H - 1)}:
        s = (slice(b, b + 1), slice(h, h + 1))
        want_idx = oret.select_topk(oret.landmark_scores(q[s], kc[s], cos, sin, block, k), k)
        assert torch.equal(idx[s].cpu(), want_idx)
        want = oret.retrieve_and_attend_s1(q[s], kc[s], vc[s], kl[s], vl[s], cos, sin, block, k, want_idx, tokens=rows)
        for (_, _, t), o in want.items():
            # 16-bit weights, output and (oracle) rotated keys, values up to about 2
            assert (out[b, h, t].float().cpu() - o).abs().max() <= (2e-2 if dtype == torch.bfloat16 else 2.5e-3), (b, h, t)
