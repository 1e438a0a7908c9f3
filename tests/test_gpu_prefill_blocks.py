"""The prefill attention's block orders against a plain fp32 product with an
fp64 softmax: head groups of unequal size with a ragged last block, one group,
and a head count that 8 does not divide.

Bars: the output within 2^-10 sum_t a_t |v_t| (two fp16 roundings of a weight)
plus one fp16 ulp; the log-sum-exp within 2^-21 (|lse| + 8)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,T,D,causal", [
    (10, 40, 4, 2050, 128, True),    # ragged blocks; groups of 17, 17 and 16 heads
    (12, 32, 4, 2113, 128, False),   # groups without the causal skip
    (3, 40, 5, 5000, 64, True),      # groups of 8 and 7 heads
    (2, 16, 2, 193, 128, True),      # one group
    (1, 12, 12, 129, 64, True),      # 12 heads: every head at once
])
def test_block_orders(B, Hq, Hkv, T, D, causal):
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    print(f"prefill attention blocks B={B} {Hq}/{Hkv} T={T} D={D} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + Hq)
    q, k, v = (torch.randn(B, h, T, D, generator=g, device="cuda").half() for h in (Hq, Hkv, Hkv))
    out, lse = care_kv.prefill_attention(q, k, v, causal=causal, return_lse=True)
    future = torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)
    for b in range(B):
        for hk in range(Hkv):
            heads = slice(hk * (Hq // Hkv), (hk + 1) * (Hq // Hkv))
            for h in range(heads.start, heads.stop):
                S = (q[b, h].float() @ k[b, hk].float().t().contiguous()).double() / math.sqrt(D)
                if causal:
                    S = S.masked_fill(future, -math.inf)
                z = S.logsumexp(-1)
                A = (S - z[:, None]).exp().float()
                ref, bound = A @ v[b, hk].float(), 2.0 ** -10 * (A @ v[b, hk].float().abs())
                ulp = ref.abs().clamp_min(2.0 ** -14).log2().floor().exp2() * 2.0 ** -10
                assert bool(((out[b, h].float() - ref).abs() <= bound + ulp).all()), (b, h)
                assert bool(((lse[b, h].double() - z).abs() <= 2.0 ** -21 * (z.abs() + 8)).all()), (b, h)
