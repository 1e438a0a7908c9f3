"""``CAREKVCache.reset_sequence`` launches on the cache's device, whatever device
is current (without a device: the library and the guard are stand-ins)."""
from types import SimpleNamespace

import numpy as np
import torch

import care_kv
from care_kv import _lib, cache as cache_mod


def test_launches_on_the_caches_device(monkeypatch):
    entered, launched = [], []

    class Guard:
        def __init__(self, device):
            self.device = device

        def __enter__(self):
            entered.append(self.device)

        def __exit__(self, *exc):
            entered.pop()

    class Lib:
        def carekv_reset_sequence(self, *args):
            launched.append((list(entered), args[10]))
            return 0
    lib = Lib()
    monkeypatch.setattr(torch.cuda, "device", Guard)
    monkeypatch.setattr(_lib, "load", lambda path=None: lib)
    monkeypatch.setattr(_lib, "stream_ptr", lambda device: 0)
    c = cache_mod.CAREKVCache.__new__(cache_mod.CAREKVCache)
    c.cfg = care_kv.CacheConfig(num_layers=1, num_heads=4, num_kv_heads=2, head_dim=64, page_size=16, max_pages=4)
    c.device, c.n_seq, c.ncg, c.nvb, c.kivi_packed = torch.device("cuda"), 3, 2, 4, False
    for n in ("valid", "has_meta", "k_slot", "v_slot", "next_slot"):
        setattr(c, n, SimpleNamespace(device=torch.device("cuda", 1), data_ptr=lambda: 0))
    c._freed, c.streaming_store, c.rescale_open = {}, False, False
    c.next_page = np.ones((1, 2, 3), dtype=np.int64)
    c.valid_host = np.ones((1, 2, 3, 4), dtype=np.int32)
    c._token_start = np.ones((1, 2, 3, 4), dtype=np.int64)
    c.reset_sequence(-1)
    assert launched == [([torch.device("cuda", 1)], 2)]
    assert not c.next_page[:, :, 2].any() and c.next_page[:, :, :2].all()
