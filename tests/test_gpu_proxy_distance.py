"""The sketch proxy's distances ||V_hat_t - O_base||: expanded on the matrix
cores, taken directly where the expansion cancels.

Selections and outputs against the oracle (epsilon ties of the scores, 1e-4
relative) where a query's output sits on one token's V_hat (the cancelling
case), at small and large magnitudes of V (the operand's scale), with several
slots per page, GQA groups of 1, 4, 5 and 8 queries and a part-filled last
page."""
import numpy as np
import pytest
import torch

from helpers import PAPER_ENV
from oracle.check import (compare_selection, forced_selection, oracle_candidates, oracle_slice_from_device,
                          output_errors)
from oracle import quant as Q
from oracle.attention import base_attention, vectorized_joint_correction

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,D,N,bits,vmag,peak", [(8, 8, 64, 55, 3, 1.0, 0.0), (8, 2, 128, 530, 4, 1.0, 0.0),
                                                     (5, 1, 64, 300, 3, 3e-3, 0.0), (8, 1, 128, 300, 2, 300.0, 0.0),
                                                     (4, 1, 128, 400, 4, 1.0, 60.0), (8, 1, 64, 200, 3, 1.0, 60.0)])
def test_proxy_distances(monkeypatch, Hq, Hkv, D, N, bits, vmag, peak):
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    import care_kv
    for k, v in dict(PAPER_ENV, CAREKV_KSCORE_LIVE="0", CAREKV_K_CORRECTION_MODE="exact").items():
        monkeypatch.setenv(k, v)
    print(f"proxy distances Hq={Hq} Hkv={Hkv} D={D} N={N} INT{bits} vmag={vmag} peak={peak}", flush=True)
    kw = dict(read_budget_mode="absolute", read_abs_k=6, read_abs_v=5, route_policy="joint")
    cfg = care_kv.CacheConfig(num_layers=1, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16,
                              max_pages=N // 16 + 2, base_bits=bits, group_size=32, k_channel_group=32,
                              v_token_block=4, sketch_dim=32, packed_base=True, scale_quant="none",
                              store_budget_mode="absolute", store_abs_k=2, store_abs_v=2, read_budget_ratio=0.0, **kw)
    cache = care_kv.CAREKVCache(cfg)
    g = torch.Generator(device="cuda").manual_seed(N + D)
    K = torch.randn(Hkv, N, D, generator=g, device="cuda")
    V = torch.randn(Hkv, N, D, generator=g, device="cuda") * vmag
    q = torch.randn(1, Hq, D, generator=g, device="cuda")
    if peak:  # the logit of token 37 far above the rest: O_base = V_hat of that token, up to rounding
        q = q.abs()
        K[:, 37] = peak * 8.0 / D
    cache.write_prefill(0, K.half(), V.half())
    out, diag = care_kv.decode_attention(cache, 0, q.half(), diag_cap=64)
    torch.cuda.synchronize()
    grp, qn = Hq // Hkv, q.half().cpu().numpy()[0]
    for h in range(Hkv):
        oc = oracle_slice_from_device(cache, 0, h, num_heads=grp, store_budget_mode="absolute", **kw)
        pids = oc.all_page_ids(0, 0)
        Kc, Ks, Vc, Vs, _ = oc.read_base_concat(0, 0, pids)
        Kh, Vh = (Q.dequantize(c, s, 32).astype(np.float32) for c, s in ((Kc, Ks), (Vc, Vs)))
        Qg = qn[h * grp:(h + 1) * grp]
        S, A, O = base_attention(Kh, Vh, Qg.astype(np.float32))
        args = dict(kind="both", k_corr_scale=0.1, score_normalize=True, kscore_live=False, k_mode="exact")
        d = {}
        vectorized_joint_correction(oc, 0, 0, pids, Qg, S, A, Vh, O, diag=d, **args)
        Kcand, Vcand = oracle_candidates(oc, 0, 0, len(pids))
        rows = diag[0, h * grp:(h + 1) * grp].cpu().numpy()
        _, _, bad = compare_selection(rows, d, Kcand, Vcand, eps=1e-4)
        assert bad == 0, h
        dlt = vectorized_joint_correction(oc, 0, 0, pids, Qg, S, A, Vh, O,
                                          force_sel=forced_selection(rows, Kcand, Vcand), **args)
        got = out[0, h * grp:(h + 1) * grp].cpu().numpy()
        _, rel, _ = output_errors(got, (O + dlt).astype(np.float16))
        assert rel <= 1e-2, (h, rel)
