"""A prompt row's attention depends on its own scores alone: the same bits
whatever stands in the later rows, beside it in the batch, or behind the prompt."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(B, Hq, Hkv, T, D, seed):
    """Inputs whose running maxima move in many tiles: a level that rises and falls with the token."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(B, h, T, D, generator=g, device="cuda") for h in (Hq, Hkv, Hkv))
    t = torch.arange(T, device="cuda").float()
    q[..., 0], k[..., 0] = math.sqrt(D) / 4, 16.0 * torch.sin(t / 37.0) + 0.02 * t
    return q.half(), k.half(), v.half()


def _same(a, b):
    return all(torch.equal(x.view(torch.int16), y.view(torch.int16)) for x, y in zip(a, b))


@pytest.mark.parametrize("D,T,cut", [(64, 300, 131), (64, 517, 400), (128, 300, 131), (128, 517, 33)])
def test_later_rows(D, T, cut):
    """Other queries, keys and values from `cut` on, and a prompt that ends there."""
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    print(f"prefill attention, later rows D={D} T={T} cut={cut}", flush=True)
    q, k, v = _rows(1, 4, 2, T, D, T + D)
    ref = [x[:, :, :cut] for x in care_kv.prefill_attention(q, k, v, return_lse=True)]
    q2, k2, v2 = (x.clone() for x in (q, k, v))
    q2[:, :, cut:] *= -3.0
    k2[:, :, cut:] *= 2.0
    v2[:, :, cut:] += 1.0
    got = [x[:, :, :cut] for x in care_kv.prefill_attention(q2, k2, v2, return_lse=True)]
    assert _same(got, ref)
    assert _same(care_kv.prefill_attention(*(x[:, :, :cut].contiguous() for x in (q, k, v)), return_lse=True), ref)


def test_batch():
    """One sequence of a large batch, and alone."""
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    B, Hq, Hkv, T, D = 10, 40, 4, 2050, 128
    print(f"prefill attention, batch of {B} and alone T={T}", flush=True)
    q, k, v = _rows(B, Hq, Hkv, T, D, 5)
    out, lse = care_kv.prefill_attention(q, k, v, return_lse=True)
    for b in (0, 7):
        assert _same([out[b], lse[b]], care_kv.prefill_attention(q[b], k[b], v[b], return_lse=True))
