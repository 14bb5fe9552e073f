"""Rows stored by kernels: the ring cache's store in one launch and the growing cache's append, against the restated
storage (oracle/mem_cache.py) and plain slices, bit for bit."""
import pytest
import torch

from oracle import mem_cache as omc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,block,chunks,hs", [
    (4, 3, [3, 3, 6, 3, 9], 8),                   # whole blocks, the ring wraps
    (4, 3, [5, 2, 8, 1, 1, 1, 13], 64),           # tails of every length, chunks that do not complete a block
    (3, 4, [40], 64),                             # more blocks than slots: the newest win
    (3, 4, [3, 20, 6, 1], 128),                   # a tail in front of more blocks than slots
    (5, 51, [51 * 7 + 13, 255, 38, 1], 64),       # the benchmark's blocks
])
def test_ring_store_matches_the_restated_storage(cap, block, chunks, hs):
    from landmark_hip.mem_cache import MemLMCacheStorage
    B, nh = 2, 3
    s = MemLMCacheStorage(B, cap, block - 1, nh, hs, dtype=torch.bfloat16, device="cuda")
    r = omc.RingStore(B, cap, block, nh, hs, dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(cap)
    seen = 0
    for i, T in enumerate(chunks):
        shape = (B, T, nh, hs) if i % 2 else (B, nh, T, hs)          # the projections' layout too
        k, v = (torch.randn(shape, generator=g).bfloat16() for _ in range(2))
        if i % 2:
            k, v = k.transpose(1, 2), v.transpose(1, 2)
        im = ((torch.arange(T) + seen) % block == block - 1)[None].expand(B, T)
        s.store_in_cache(k.cuda(), {"v": v.cuda(), "is_mem": im.cuda()})
        r.store(k, v, im)
        seen += T
        n, rest = r.filled, s.last_incomplete_len
        assert (s.cache_iter, s.cache_size, s.filled) == (r.cache_iter, r.cache_size, n)
        assert torch.equal(s.cache_mem_k[:, :n].cpu(), r.cache_k[:, :n]) and torch.equal(s.cache_mem_v[:, :n].cpu(), r.cache_v[:, :n])
        assert torch.equal(s.last_incomplete_k[:, :, :rest].cpu(), r.pending_k)
        assert torch.equal(s.last_incomplete_v[:, :, :rest].cpu(), r.pending_v)
        assert not s.last_incomplete_ismem[:, :rest].any()


def test_ring_store_still_rejects_a_landmark_in_the_wrong_place():
    from landmark_hip.mem_cache import MemLMCacheStorage
    s = MemLMCacheStorage(1, 4, 3, 2, 64, dtype=torch.float16, device="cuda")
    x = torch.zeros(1, 2, 6, 64, dtype=torch.float16, device="cuda")
    marks = torch.tensor([[False, False, False, True, False, True]], device="cuda")      # the tail's second token
    s.store_in_cache(x, {"v": x, "is_mem": marks})                   # shows only when its block is complete
    with pytest.raises(AssertionError):
        s.store_in_cache(x[:, :, :2], {"v": x[:, :, :2], "is_mem": torch.tensor([[False, True]], device="cuda")})


@pytest.mark.parametrize("D", [64, 128])
def test_append_by_kernel_equals_slices(D):
    from landmark_hip.cache import LandmarkKVCache
    cache = LandmarkKVCache(2, 3, D, torch.float16, "cuda", capacity=8)
    g = torch.Generator(device="cuda").manual_seed(0)
    ks, vs = [], []
    for t in (5, 1, 9, 40):
        k, v = (torch.randn((2, t, 3, D), generator=g, device="cuda").half().transpose(1, 2) for _ in range(2))
        ks.append(k)
        vs.append(v)
        cache.append(k, v)
    pk, pv = cache.past_key_value
    assert torch.equal(pk, torch.cat(ks, 2)) and torch.equal(pv, torch.cat(vs, 2))


def test_a_store_behind_a_refused_one_looks_at_the_tail_it_left():
    from landmark_hip.mem_cache import MemLMCacheStorage
    s = MemLMCacheStorage(1, 4, 3, 2, 64, dtype=torch.float16, device="cuda")
    x = torch.zeros(1, 2, 6, 64, dtype=torch.float16, device="cuda")
    marks = torch.tensor([[False, True, False, True, True, False]], device="cuda")       # the tail opens with a landmark
    with pytest.raises(AssertionError):
        s.store_in_cache(x, {"v": x, "is_mem": marks})
    with pytest.raises(AssertionError):
        s.store_in_cache(x[:, :, :2], {"v": x[:, :, :2], "is_mem": torch.tensor([[False, True]], device="cuda")})
