"""Operands that stand 2 or 8 bytes off a 16-byte boundary (views into a larger
buffer, a caller's own tables) give the bits of aligned ones."""
import pytest
import torch

from helpers import PAPER_ENV

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")


def _off(x, n):
    """x's values, contiguous, n elements past the start of an allocation."""
    buf = torch.empty(x.numel() + n + 8, dtype=x.dtype, device=x.device)
    y = buf[n:n + x.numel()].view(x.shape)
    y.copy_(x)
    assert y.is_contiguous() and y.data_ptr() % 16 == n * x.element_size()
    return y


@pytest.mark.parametrize("n", [1, 4])
@pytest.mark.parametrize("D,T", [(64, 75), (128, 33)])
def test_prefill(D, T, n):
    import care_kv
    print(f"prompt operands {2 * n} bytes off D={D} T={T}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn(h, T, D, generator=g, device="cuda").half() for h in (4, 2, 2))
    kh, vh = care_kv.quant_dequant(k, 3), care_kv.quant_dequant(v, 3)
    o = care_kv.prefill_attention(q, kh, vh)
    assert torch.equal(care_kv.prefill_attention(*(_off(x, n) for x in (q, kh, vh))), o)
    args = (q, k, v, kh, vh, o)
    ref, sel = care_kv.prefill_eval(*args, ratio=0.2, diag_cap=20)
    got, s2 = care_kv.prefill_eval(*(_off(x, n) for x in args), ratio=0.2, diag_cap=20)
    assert torch.equal(got, ref) and torch.equal(s2, sel)


@pytest.mark.parametrize("sketch_dim", [32, 24, 20])
def test_sketch_table(monkeypatch, sketch_dim):
    import care_kv
    for k, v in dict(PAPER_ENV, CAREKV_KSCORE_LIVE="0").items():
        monkeypatch.setenv(k, v)
    print(f"sketch table 2 bytes off, sketch_dim={sketch_dim}", flush=True)
    N, Hq, Hkv, D = 700, 8, 2, 64
    cfg = care_kv.CacheConfig(num_layers=1, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16, max_pages=N // 16 + 2,
                              base_bits=3, group_size=32, k_channel_group=32, v_token_block=4, sketch_dim=sketch_dim,
                              packed_base=True, scale_quant="int8", store_budget_mode="absolute", store_abs_k=2,
                              store_abs_v=2, read_budget_ratio=0.0, read_budget_mode="absolute", read_abs_k=8, read_abs_v=8,
                              route_policy="separate")
    cache = care_kv.CAREKVCache(cfg)
    g = torch.Generator(device="cuda").manual_seed(3)
    cache.write_prefill(0, *(torch.randn(Hkv, N, D, generator=g, device="cuda").half() for _ in range(2)))
    q = torch.randn(1, Hq, D, generator=g, device="cuda").half()
    ref, sel = care_kv.decode_attention(cache, 0, q, diag_cap=16)
    table = _off(cache.k_sketch, 1)
    cache.arena(0).k_sketch = table.data_ptr()
    got, s2 = care_kv.decode_attention(cache, 0, q, diag_cap=16)
    assert torch.equal(got, ref) and torch.equal(s2, sel)
