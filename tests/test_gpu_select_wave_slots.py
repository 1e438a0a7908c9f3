"""The wave-per-query select with several slots per page against the
work-group select, bit for bit (outputs, selections): decode rows of 1-256
pages and prompt rows, equal pages whose ties meet the threshold inside a
page and across pages, one kind stored only, budgets past the candidates."""
import pytest
import torch

from test_gpu_select_wave import _both, _need_gpu, _same, paper_env  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # Hq, Hkv, D, lengths, stored (K, V), (read K, read V), policy
    (32, 4, 64, [2303, 40, 1000, 16], (2, 4), (2, 2), "joint"),
    (32, 4, 64, [4096, 15], (1, 3), (64, 64), "joint"),
    (16, 4, 128, [2000, 3001], (4, 2), (16, 24), "separate"),
    (8, 8, 128, [1030, 64], (3, 4), (5000, 5000), "joint"),
    (8, 2, 64, [1500], (0, 2), (8, 8), "joint"),
    (8, 2, 64, [1500], (2, 0), (8, 8), "separate"),
]


def _cache(care_kv, Hq, Hkv, D, pages, stored, read, policy, n_seq):
    cfg = care_kv.CacheConfig(num_layers=1, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16, max_pages=pages,
                              base_bits=3, group_size=32, k_channel_group=32, v_token_block=4, sketch_dim=32,
                              packed_base=True, scale_quant="int8", store_budget_mode="absolute",
                              store_abs_k=stored[0], store_abs_v=stored[1], read_budget_ratio=0.0,
                              read_budget_mode="absolute", read_abs_k=read[0], read_abs_v=read[1], route_policy=policy)
    return care_kv.CAREKVCache(cfg, n_seq=n_seq)


def _prompt(g, Hkv, n, D, ties):
    K = torch.randn(Hkv, n, D, generator=g, device="cuda")
    K[:, :, :2] *= 6.0
    V = torch.randn(Hkv, n, D, generator=g, device="cuda")
    if ties and n >= 96:
        for X in (K, V):
            X[:, 32:48], X[:, 64:80] = X[:, 16:32], X[:, 16:32]   # equal pages
            X[:, 84:88], X[:, 88:92] = X[:, 80:84], X[:, 80:84]   # equal V blocks of a page
    return K.half(), V.half()


@pytest.mark.parametrize("case", CASES, ids=[f"g{c[0] // c[1]}-D{c[2]}-s{c[4][0]}{c[4][1]}-{c[6]}" for c in CASES])
def test_decode(paper_env, case):  # noqa: F811
    import care_kv
    Hq, Hkv, D, lens, stored, read, policy = case
    print(f"wave select slots Hq={Hq} Hkv={Hkv} D={D} lens={lens} stored={stored} read={read} {policy}", flush=True)
    cache = _cache(care_kv, Hq, Hkv, D, max(lens) // 16 + 2, stored, read, policy, len(lens))
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + D)
    for b, n in enumerate(lens):
        cache.write_prefill(0, *_prompt(g, Hkv, n, D, True), seqs=[b])
    q = torch.randn(len(lens), Hq, D, generator=g, device="cuda").half()
    a, b = _both(paper_env, lambda: care_kv.decode_attention(cache, 0, q, diag_cap=1024))
    _same(a, b)
    assert int((a[1] >= 0).sum()) > 0


@pytest.mark.parametrize("Hq,Hkv,D,stored", [(32, 4, 64, (2, 4)), (12, 12, 64, (2, 1)), (8, 2, 128, (4, 3))])
def test_prompt_rows(paper_env, Hq, Hkv, D, stored):  # noqa: F811
    import care_kv
    T = 700
    print(f"wave select slots prompt rows Hq={Hq} Hkv={Hkv} D={D} stored={stored}", flush=True)
    cache = _cache(care_kv, Hq, Hkv, D, T // 16 + 2, stored, (2, 2), "joint", 1)
    g = torch.Generator(device="cuda").manual_seed(T + D)
    K, V = _prompt(g, Hkv, T, D, True)
    cache.write_prefill(0, K, V)
    kh, vh = care_kv.quant_dequant(K, 3), care_kv.quant_dequant(V, 3)
    q = torch.randn(T, Hq, D, generator=g, device="cuda").half()
    _, lse = care_kv.prefill_attention(q.transpose(0, 1), kh, vh, return_lse=True)
    a, b = _both(paper_env, lambda: care_kv.prefill_correction(cache, 0, q, kh, vh, lse, diag_cap=8))
    _same(a, b)
    assert int((a[1] >= 0).sum()) > 0
