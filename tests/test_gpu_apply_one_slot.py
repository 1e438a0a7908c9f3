"""The one-slot apply pass (one K and one V slot a page at most) against the
ranked one, which a larger record capacity selects: the same selections and
the same terms in the same order, so the same output bits.  Decode rows with
more than 4 query heads per kv head or fp16 pages, and prompt rows; pages
whose only slots lie in any channel group or block, ragged last pages."""
import pytest
import torch

from helpers import PAPER_ENV

pytestmark = pytest.mark.gpu


def _cache(care_kv, Hq, Hkv, D, n, lens, base="uniform", scales="int8"):
    cfg = care_kv.CacheConfig(num_layers=1, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16,
                              max_pages=n // 16 + 2, base_bits=3 if base == "uniform" else 2, base_quantizer=base,
                              group_size=32, k_channel_group=32, v_token_block=4, sketch_dim=32, packed_base=True,
                              scale_quant=scales, store_budget_mode="absolute", store_abs_k=1, store_abs_v=1,
                              read_budget_ratio=0.0, read_budget_mode="absolute", read_abs_k=12, read_abs_v=12,
                              route_policy="joint")
    return care_kv.CAREKVCache(cfg, n_seq=lens)


def _prompt(g, Hkv, n, D):
    K, V = (torch.randn(Hkv, n, D, generator=g, device="cuda") for _ in range(2))
    t = torch.arange(n, device="cuda")
    for c in range(D // 32):  # the loud channel group and V block move from page to page
        K[:, (t // 16) % (D // 32) == c, 32 * c + 3] *= 6.0
    V[:, (t // 4) % 4 == (t // 16) % 4] *= 3.0
    return K.half(), V.half()


def _both(cache, call):
    one = call()
    k_cap, cache.k_cap = cache.k_cap, 2
    try:
        ranked = call()
    finally:
        cache.k_cap = k_cap
    assert int((one[1] >= 0).sum()) > 0
    a, b = (torch.sort(x[1].flatten(0, -2), -1).values for x in (one, ranked))
    n = min(a.shape[-1], b.shape[-1])
    assert torch.equal(a[..., -n:], b[..., -n:])
    assert torch.equal(one[0], ranked[0])


@pytest.mark.parametrize("mode", ["exact", "linear"])
@pytest.mark.parametrize("Hq,Hkv,D,base,scales", [(32, 4, 64, "uniform", "int8"), (5, 1, 128, "uniform", "none"),
                                                  (8, 4, 64, "kivi_style", "int8"), (4, 2, 128, "kivi_style", "int8")])
def test_decode(monkeypatch, Hq, Hkv, D, base, scales, mode):
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    for k, v in dict(PAPER_ENV, CAREKV_K_CORRECTION_MODE=mode).items():
        monkeypatch.setenv(k, v)
    lens = [515, 17, 300, 9]
    print(f"one-slot apply Hq={Hq} Hkv={Hkv} D={D} {base} {scales} {mode}", flush=True)
    cache = _cache(care_kv, Hq, Hkv, D, 515, len(lens), base, scales)
    g = torch.Generator(device="cuda").manual_seed(Hq + D)
    for b, n in enumerate(lens):
        cache.write_prefill(0, *_prompt(g, Hkv, n, D), seqs=[b])
    q = torch.randn(len(lens), Hq, D, generator=g, device="cuda").half()
    _both(cache, lambda: care_kv.decode_attention(cache, 0, q, diag_cap=64))


@pytest.mark.parametrize("Hq,Hkv,D,T", [(32, 4, 64, 700), (8, 8, 128, 205), (6, 2, 64, 33)])
def test_prompt_rows(monkeypatch, Hq, Hkv, D, T):
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    for k, v in dict(PAPER_ENV, CAREKV_K_CORRECTION_MODE="exact").items():
        monkeypatch.setenv(k, v)
    print(f"one-slot apply prompt rows Hq={Hq} Hkv={Hkv} D={D} T={T}", flush=True)
    cache = _cache(care_kv, Hq, Hkv, D, T, 1)
    g = torch.Generator(device="cuda").manual_seed(T + D)
    K, V = _prompt(g, Hkv, T, D)
    cache.write_prefill(0, K, V)
    kh, vh = care_kv.quant_dequant(K, 3), care_kv.quant_dequant(V, 3)
    q = torch.randn(T, Hq, D, generator=g, device="cuda").half()
    _, lse = care_kv.prefill_attention(q.transpose(0, 1), kh, vh, return_lse=True)
    _both(cache, lambda: care_kv.prefill_correction(cache, 0, q, kh, vh, lse, diag_cap=64))
