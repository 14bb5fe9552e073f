"""Host side of the ring cache's store: which chunks may go to the one-launch path, on the CPU (no kernel is launched)."""
from types import SimpleNamespace

import pytest
import torch


def _storage(cap=4, block=4, nh=2, hs=8, dtype=torch.bfloat16):
    from landmark_hip.mem_cache import MemLMCacheStorage
    return MemLMCacheStorage(1, cap, block - 1, nh, hs, dtype=dtype, device="cpu")


def _on(device, dtype, *shape):
    """What the store asks a GPU tensor before it hands it to the kernel."""
    return SimpleNamespace(is_cuda=True, device=torch.device("cuda", device), dtype=dtype, shape=torch.Size(shape),
                           dim=lambda: len(shape))


@pytest.mark.parametrize("elsewhere", ["keys", "values", "is_mem", None])
def test_rows_of_another_gpu_do_not_take_the_one_launch_path(elsewhere, monkeypatch):
    from landmark_hip import attention
    monkeypatch.setattr(attention, "_check_is_mem", lambda *a, **k: None)        # the marks are as they must be
    s = _storage()
    s.cache_mem_k = s.cache_mem_v = _on(0, torch.bfloat16, 1, 4, 4, 2, 8)
    at = {name: int(name == elsewhere) for name in ("keys", "values", "is_mem")}
    assert s._continues_the_stream(_on(at["keys"], torch.bfloat16, 1, 2, 4, 8), _on(at["values"], torch.bfloat16, 1, 2, 4, 8),
                                   _on(at["is_mem"], torch.bool, 1, 4), 0, 4) == (elsewhere is None)


@pytest.mark.parametrize("elsewhere", range(8))
def test_the_native_store_refuses_tensors_of_several_devices(elsewhere):
    from landmark_hip import _lib
    s = _storage()
    x = torch.zeros(1, 2, 4, 8, dtype=torch.bfloat16)
    args = [x, x, torch.zeros(1, 4, dtype=torch.bool), s.last_incomplete_k, s.last_incomplete_v, s.last_incomplete_ismem,
            s.cache_mem_k, s.cache_mem_v]
    args[elsewhere] = args[elsewhere].to("meta")
    with pytest.raises(AssertionError, match="on the cache's device"):
        _lib.native().ring_store(*args, 0, 0)
    with pytest.raises(AssertionError, match="GPU"):                               # one device, but the CPU
        _lib.native().ring_store(*(t.to("cpu") if t.is_cpu else torch.zeros(t.shape, dtype=t.dtype) for t in args), 0, 0)


def test_a_refused_store_does_not_leave_its_tail_to_the_path_that_does_not_look_at_it(monkeypatch):
    from landmark_hip import _lib
    s = _storage()
    x = torch.zeros(1, 2, 6, 8, dtype=torch.bfloat16)
    marks = torch.tensor([[False, True, False, True, True, False]])       # a landmark too many; then the tail opens with one
    with pytest.raises(AssertionError):
        s.store_in_cache(x, {"v": x, "is_mem": marks})
    # the chunk by itself continues the stream, as _check_is_mem would find on the GPU
    monkeypatch.setattr(s, "_continues_the_stream", lambda *a: True)
    monkeypatch.setattr(_lib, "native", lambda: pytest.fail("stored without a look at the tail"))
    with pytest.raises(AssertionError, match="every block"):
        s.store_in_cache(x[:, :, :2], {"v": x[:, :, :2], "is_mem": torch.tensor([[False, True]])})
