"""The host tables of ``CAREKVCache.append`` and ``decode_attention`` without a
device: an entry is made for every row that the kernels are told to read."""
import numpy as np
import pytest
import torch

import care_kv
from care_kv import _lib, cache as cache_mod


class _Lib:
    """carekv_append_rows over host memory: keeps the destinations it is given."""

    def carekv_append_rows(self, arena, k, v, dest, n_rows, stream):
        self.n_rows = n_rows
        return 0


@pytest.fixture
def cache(monkeypatch):
    lib, tables = _Lib(), []
    monkeypatch.setattr(_lib, "load", lambda path=None: lib)
    monkeypatch.setattr(_lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(cache_mod, "to_device", lambda a, device: tables.append(a) or torch.from_numpy(a))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    cfg = care_kv.CacheConfig(num_layers=1, num_heads=4, num_kv_heads=2, head_dim=64, page_size=16, max_pages=4)
    c = cache_mod.CAREKVCache.__new__(cache_mod.CAREKVCache)
    c.cfg, c.device, c.kivi_packed, c.streaming_store = cfg, torch.device("cpu"), False, False
    c.next_page = np.zeros((1, 2, 3), dtype=np.int64)
    c.valid_host = np.zeros((1, 2, 3, 4), dtype=np.int32)
    c._token_start = np.zeros((1, 2, 3, 4), dtype=np.int64)
    c._row_indices, c._dest_tables, c.arena = {}, {}, lambda layer: None
    c.lib, c.tables = lib, tables
    return c


@pytest.mark.parametrize("B,H,seqs", [(2, 2, [0]), (3, 2, [0, 1]), (1, 2, [0, 1]), (2, 2, []), (1, 3, [0]),
                                      (2, 5, [0, 2])])
def test_mismatched_rows_are_refused(cache, B, H, seqs):
    x = torch.zeros(B, H, 64, dtype=torch.float16)
    with pytest.raises(ValueError):
        cache.append(0, x, x, seqs=seqs)
    assert not cache.tables and not cache.next_page.any() and not cache.valid_host.any()


def test_a_destination_for_every_row(cache):
    for B, seqs in ((2, [2, 0]), (1, [1]), (3, None), (2, [2, 0])):
        x = torch.zeros(B, 2, 64, dtype=torch.float16)
        cache.append(0, x, x, seqs=seqs)
        assert cache.lib.n_rows == 2 * B == len(cache.tables[-1])
        assert cache.tables[-1][:, 0].tolist() == [s for s in (seqs or range(B)) for _ in range(2)]
        assert cache.tables[-1][:, 1].tolist() == [0, 1] * B


def test_decode_rows_without_a_slot_are_refused(cache):
    q = torch.zeros(3, 4, 64, dtype=torch.float16)
    for seqs in ([], [0], [0, 2]):
        with pytest.raises(ValueError):
            care_kv.decode_attention(cache, 0, q, seqs=seqs)
