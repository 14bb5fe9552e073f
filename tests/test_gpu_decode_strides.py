"""Decode steps whose row strides do not fit the decode gather's 32-bit offsets, through the C ABI: tables handed over back to
front (a negative stride from their last row) and a cache whose rows lie half a gigabyte apart.  Every address is inside its
tensor; the results are those of the same values in the usual layout.
"""
import math

import pytest
import torch

from oracle import retrieval as oret
from oracle import rotary as orot

pytestmark = pytest.mark.gpu

TOL = 2e-2      # 16-bit weights, output and (oracle) rotated keys, values up to about 2


def _step(q, kc, vc, kl, vl, cos, sin, table_row0, table_stride, block, k):
    """lmk_retrieve_and_attend; table row 0 is row table_row0 of cos and sin, the next one table_stride elements on."""
    from landmark_hip import _lib
    lib, (B, H, T, D), S = _lib.lib(), q.shape, kc.shape[2]
    out = torch.empty_like(q)
    idx = torch.empty(B, H, T, min(k, S // block), dtype=torch.int64, device=q.device)
    sizes = lib.lmk_retrieve_workspace_bytes(B, H, T, S, D, block), lib.lmk_attend_workspace_bytes(B, H, T, S, D, block)
    ws = [torch.empty(n, dtype=torch.uint8, device=q.device) for n in sizes]
    _lib.check(lib.lmk_retrieve_and_attend(
        *(_lib.tensor4(t) for t in (q, kc, vc, kl, vl)), cos[table_row0].data_ptr(), sin[table_row0].data_ptr(), table_stride,
        cos.shape[0], idx.data_ptr(), _lib.tensor4(out), ws[0].data_ptr(), sizes[0], 0, ws[1].data_ptr(), sizes[1], B, H, T, S, D,
        1 / math.sqrt(D), block, k, _lib.DTYPE_CODES[q.dtype], _lib.current_stream(q.device)))
    torch.cuda.synchronize()
    return out, idx


def _values(B, H, T, S, D, dtype):
    g = torch.Generator().manual_seed(S + D)
    make = lambda rows: (torch.randn(B, H, rows, D, generator=g) * 0.5).to(dtype)
    return [make(r) for r in (T, S, S, T, T)], orot.rotary_tables(S + T, D, dtype)


def _check(out, idx, tensors, cos, sin, tail, block, k):
    T = tensors[0].shape[2]
    want, want_idx = oret.retrieve_and_attend(*tensors, ((torch.arange(T) + tail) % block == block - 1)[None], cos, sin, block, k)
    assert torch.equal(idx.cpu(), want_idx)
    assert (out.float().cpu() - want.float()).abs().max() <= TOL


@pytest.mark.parametrize("block,D,T,tail,dtype", [(32, 128, 1, 7, torch.bfloat16), (32, 64, 2, 0, torch.float16),
                                                  (64, 128, 4, 60, torch.bfloat16), (128, 64, 1, 21, torch.bfloat16)])
def test_tables_back_to_front(block, D, T, tail, dtype):
    print(f"case block {block} D{D} T{T} tail {tail} {dtype}", flush=True)
    B, H, k, S = 1, 2, 3, 5 * block + tail
    tensors, (cos, sin) = _values(B, H, T, S, D, dtype)
    dev = [t.cuda() for t in tensors]
    last = cos.shape[0] - 1
    out, idx = _step(*dev, cos.flip(0).contiguous().cuda(), sin.flip(0).contiguous().cuda(), last, -D, block, k)
    _check(out, idx, tensors, cos, sin, tail, block, k)


def test_rows_half_a_gigabyte_apart():
    block, D, T, tail, k = 32, 64, 1, 2, 1
    B, H, S, row = 1, 1, block + tail, 1 << 28
    tensors, (cos, sin) = _values(B, H, T, S, D, torch.bfloat16)
    store = torch.empty((S - 1) * row + 2 * D, dtype=torch.bfloat16, device="cuda")       # 18 GB, written at the rows alone
    kc, vc = (store[i * D:].as_strided((B, H, S, D), (S * row, S * row, row, 1)) for i in (0, 1))
    kc.copy_(tensors[1]), vc.copy_(tensors[2])
    out, idx = _step(tensors[0].cuda(), kc, vc, *(t.cuda() for t in tensors[3:]), cos.cuda(), sin.cuda(), 0, D, block, k)
    _check(out, idx, tensors, cos, sin, tail, block, k)
    del store, kc, vc
    torch.cuda.empty_cache()
