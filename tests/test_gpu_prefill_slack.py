"""The prefill attention's running maximum, which is reduced only in tiles that
hold a larger score: scores that rise tile by tile, in steps or slowly, one late peak, falling scores, and a first tile that is mostly masked,
against an fp64 evaluation.

Bars: the output within 2^-10 sum_t a_t |v_t| (two fp16 roundings of a weight)
plus one fp16 ulp; the log-sum-exp, whose rounding is relative to the scaled
score and its sum's, within 2^-21 (|lse| + 8)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["rise", "jump", "peak", "fall"])
@pytest.mark.parametrize("D,T,causal", [(64, 31, True), (64, 300, True), (128, 33, True), (128, 260, False), (128, 517, True)])
def test_moving_maximum(shape, D, T, causal):
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    print(f"prefill attention {shape} D={D} T={T} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + D)
    q, k, v = (torch.randn(2, T, D, generator=g, device="cuda") for _ in range(3))
    t = torch.arange(T, device="cuda").float()
    level = {"rise": 0.05 * t, "jump": 9.0 * (t // 64), "peak": 60.0 * (t == T - 2), "fall": -0.1 * t}[shape]
    q[..., 0], k[..., 0] = math.sqrt(D) / 4, 4.0 * level   # score = q.k / sqrt(D) + level
    q, k, v = q.half(), k.half(), v.half()
    out, lse = care_kv.prefill_attention(q, k, v, causal=causal, return_lse=True)
    S = (q.double() @ k.double().transpose(1, 2).contiguous()) / math.sqrt(D)
    if causal:
        S = S.masked_fill(torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1), -math.inf)
    A = S.softmax(-1)
    ref, bound = A @ v.double(), 2.0 ** -10 * (A @ v.double().abs())
    ulp = ref.abs().clamp_min(2.0 ** -14).log2().floor().exp2() * 2.0 ** -10
    assert bool(((out.double() - ref).abs() <= bound + ulp).all())
    z = S.logsumexp(-1)
    assert bool(((lse.double() - z).abs() <= 2.0 ** -21 * (z.abs() + 8)).all())
