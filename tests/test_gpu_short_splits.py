"""Short splits of the page-per-wave streaming pass: 4, 8 and 12 pages per
work-group give the 16-page split's selections, and outputs within the weights'
rounding (a wave rounds its weights to fp16 against its own pages' running
maximum, so with other splits each differs by up to 2^-10 of itself, and the
output by up to 2^-10 max |V_hat| beside its own rounding), on ragged rows, for 5 and 8 query heads per kv
head and the fp16 (KIVI-style) base; the default split of short rows too."""
import pytest
import torch

from helpers import PAPER_ENV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,D,base", [(32, 4, 64, "uniform"), (5, 1, 128, "uniform"), (8, 4, 128, "kivi_style")])
def test_short_splits(monkeypatch, Hq, Hkv, D, base):
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    from care_kv.attention import default_split_pages
    for k, v in dict(PAPER_ENV, CAREKV_K_CORRECTION_MODE="exact").items():
        monkeypatch.setenv(k, v)
    lens = [512, 17, 300, 16]
    print(f"short splits Hq={Hq} Hkv={Hkv} D={D} {base} lens={lens}", flush=True)
    cfg = care_kv.CacheConfig(num_layers=1, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16, max_pages=36,
                              base_bits=2 if base != "uniform" else 3, base_quantizer=base, group_size=32,
                              k_channel_group=32, v_token_block=4, sketch_dim=32, packed_base=True, scale_quant="int8",
                              store_budget_mode="absolute", store_abs_k=2, store_abs_v=2, read_budget_ratio=0.0,
                              read_budget_mode="absolute", read_abs_k=8, read_abs_v=8, route_policy="joint")
    cache = care_kv.CAREKVCache(cfg, n_seq=len(lens))
    g = torch.Generator(device="cuda").manual_seed(Hq + D)
    vmax = 0.0
    for b, n in enumerate(lens):
        K, V = (torch.randn(Hkv, n, D, generator=g, device="cuda").half() for _ in range(2))
        cache.write_prefill(0, K, V, seqs=[b])
        vmax = max(vmax, 1.5 * float(V.abs().max()))  # V_hat within half a step of V
    q = torch.randn(len(lens), Hq, D, generator=g, device="cuda").half()
    run = lambda sp: care_kv.decode_attention(cache, 0, q, diag_cap=64, split_pages=sp)  # noqa: E731
    ref, sel = run(16)
    assert default_split_pages(32, 4 * Hkv, step=4) < 16
    for sp in (4, 8, 12, None):
        out, s = run(sp)
        assert torch.equal(s, sel), sp
        ulp = torch.maximum(out.abs(), ref.abs()).float().clamp_min(2.0 ** -14).log2().floor().exp2() * 2.0 ** -10
        assert bool(((out.float() - ref.float()).abs() <= 2 * ulp + 2.0 ** -10 * vmax).all()), sp
