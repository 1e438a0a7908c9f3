"""The sketch proxy's distances ||V_hat_t - O_base|| where their expansion loses
bits or is not finite.

O_base sits on one token's V_hat, exactly (the other weights underflow in the
sum), and one token of each page carries the page's mass, so the proxy's page
record is that token's weight and weight times distance."""
import pytest
import torch

from helpers import PAPER_ENV

pytestmark = pytest.mark.gpu


def _cache(care_kv, Hq, Hkv, D, N, **kw):
    args = dict(num_layers=1, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16, max_pages=N // 16 + 1, base_bits=3,
                group_size=32, k_channel_group=32, v_token_block=4, sketch_dim=32, packed_base=True, scale_quant="none",
                store_budget_mode="absolute", store_abs_k=1, store_abs_v=1, read_budget_ratio=0.0,
                read_budget_mode="absolute", read_abs_k=4, read_abs_v=4, route_policy="separate")
    args.update(kw)
    return care_kv.CAREKVCache(care_kv.CacheConfig(**args))


@pytest.mark.parametrize("shift", [0.0, 0.7, 1.0, 2.0, 3.5])
@pytest.mark.parametrize("Hq,Hkv,D", [(5, 1, 128), (10, 2, 64), (12, 1, 128)])
def test_distance_bits(monkeypatch, Hq, Hkv, D, shift):
    """V around `shift` standard deviations: |V|^2 + |O|^2 is 1 + shift^2 times
    |V - O|^2.  A distance from fp32 differences is within a few 2^-24 of itself
    (rms of 32 roundings of a growing sum of squares, halved by the root, and
    those of the record's two sums): bar 2^-23 rms and 2^-21 at most."""
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    for k, v in dict(PAPER_ENV, CAREKV_KSCORE_LIVE="0").items():
        monkeypatch.setenv(k, v)
    N, P, G = 4096, 256, Hq // Hkv
    print(f"proxy distance bits {Hq}/{Hkv} D={D} shift={shift}", flush=True)
    cache = _cache(care_kv, Hq, Hkv, D, N, base_bits=4)
    g = torch.Generator(device="cuda").manual_seed(D + G)
    V = torch.randn(Hkv, N, D, generator=g, device="cuda") + shift * torch.randn(Hkv, 1, D, generator=g, device="cuda").sign()
    q = torch.randn(1, Hq, D, generator=g, device="cuda").abs().half()
    K = torch.zeros(Hkv, N, D, device="cuda")
    K[:, ::16] = 4.0       # one token of each page
    K[:, 37] = 8.0         # and one over all
    K += 0.02 * torch.randn(Hkv, N, D, generator=g, device="cuda")
    K, V = K.half(), V.half()
    cache.write_prefill(0, K, V)
    care_kv.decode_attention(cache, 0, q)
    torch.cuda.synchronize()
    n = Hkv * G * P * 16   # the proxy's records are the workspace's last region
    rec = cache.workspace("decode", 0)[-((n + 255) // 256 * 256):][:n].view(torch.float32).view(Hkv, G, P, 4).double()
    vh = care_kv.quant_dequant(V, 4).double()
    kh = care_kv.quant_dequant(K, 4).double()
    A = (q.double().view(Hkv, G, D) @ kh.transpose(1, 2).contiguous() * D ** -0.5).softmax(-1)
    dist = (vh - vh[:, 37:38]).norm(dim=-1)[:, None]
    page = lambda x: x.reshape(Hkv, G, P, 16).sum(-1)  # noqa: E731
    assert float(A[..., 37].min()) > 1 - 1e-7
    err = (rec[..., 2] / rec[..., 0]) / (page(A * dist) / page(A)) - 1
    err = torch.cat((err[..., :2], err[..., 3:]), -1)  # (page 2 holds token 37, at distance 0)
    print("rms %.2e max %.2e" % (float(err.square().mean().sqrt()), float(err.abs().max())), flush=True)
    assert float(err.square().mean().sqrt()) <= 2.0 ** -23 and float(err.abs().max()) <= 2.0 ** -21


@pytest.mark.parametrize("Hq,Hkv,D", [(5, 1, 128), (8, 1, 64)])
def test_infinite_output(monkeypatch, Hq, Hkv, D):
    """65504 comes back from three bits as infinity: O_base is infinite in that
    channel and every other token infinitely far.  The pages tie, the lowest
    win; the token's own page (inf - inf) is no candidate."""
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    for k, v in dict(PAPER_ENV, CAREKV_KSCORE_LIVE="0", CAREKV_SCORE_NORMALIZE="0").items():
        monkeypatch.setenv(k, v)
    N = 200
    print(f"proxy with an infinite output {Hq}/{Hkv} D={D}", flush=True)
    cache = _cache(care_kv, Hq, Hkv, D, N)
    g = torch.Generator(device="cuda").manual_seed(D)
    K, V = (torch.randn(Hkv, N, D, generator=g, device="cuda").half() for _ in range(2))
    V[:, 5, 7] = 65504.0
    cache.write_prefill(0, K, V)
    q = torch.randn(1, Hq, D, generator=g, device="cuda").half()
    _, diag = care_kv.decode_attention(cache, 0, q, diag_cap=16)
    assert bool(torch.isinf(care_kv.quant_dequant(V, 3)[:, 5, 7]).all())
    for h in range(Hq):
        got = [(int(d) >> 3) & 0x7FFFFFF for d in diag[0, h].tolist() if d >= 0 and int(d) >> 30 == 0]
        assert got == [1, 2, 3, 4], (h, got)
