"""``carekv_prefill_eval`` at the edges of its row blocks and token tiles.

A work-group takes 16, 8 or 4 rows by the prompt's length (at most 2304, 4608
and 8192 tokens) and deals 16-token tiles to 16 waves.  Against the oracle on
sampled rows, under the bars of tests/test_gpu_prefill_eval.py; and a row's
result depends on nothing after the row, bit for bit: not on the prompt's
length, the rows per work-group, or infinities and NaN in later tokens."""
import numpy as np
import pytest
import torch

from oracle.attention import prefill_eval as oracle_eval
from test_gpu_prefill_eval import F16, KNOBS, _bar, _rand_case

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")


def _run(arrays, n, knobs, cap, O=None):
    import care_kv
    d = [torch.from_numpy(np.ascontiguousarray(x[:, :n])).cuda() for x in arrays]
    O = care_kv.prefill_attention(d[0], d[3], d[4]) if O is None else O[:, :n].contiguous()
    out, dg = care_kv.prefill_eval(*d, O, diag_cap=cap, **knobs)
    torch.cuda.synchronize()
    return out, dg, O


@pytest.mark.parametrize("T,D,knob", [(1, 64, "both-norm"), (15, 128, "both-raw"), (17, 64, "k"), (33, 64, "v"),
                                      (257, 128, "both-norm"), (2304, 64, "both-norm"), (2305, 64, "both-raw"),
                                      (2305, 128, "k"), (4608, 64, "both-norm"), (4609, 128, "both-raw")])
def test_rows_and_tiles(T, D, knob):
    print(f"carekv_eval edges T={T} D={D} {knob}", flush=True)
    knobs = KNOBS[knob]
    Qh, K, V, Kh, Vh = arrays = _rand_case(2, 1, D, T, seed=T + D)
    cap = max(3, int(T * knobs["ratio"]) + 1)
    out, dg, O = _run(arrays, T, knobs, cap)
    rows = sorted({0, T // 2, max(0, T - 17), max(0, T - 2), T - 1})
    diag, force, sel = {}, {}, {}
    oracle_eval(Qh, K, V, Kh, Vh, diag=diag, o_base=O.cpu().numpy(), rows=rows, **knobs)
    dgn = dg.cpu().numpy()
    for (h, t), (idx, sc) in diag.items():
        got = dgn[h, t][dgn[h, t] >= 0]
        assert len(got) == len(idx) and np.all(np.diff(got) > 0), (h, t)
        sel[(h, t)] = got
        if not np.array_equal(got, idx):  # tokens whose scores tie to within 1e-5 of the row's top score
            assert abs(float(sc[got].min()) - float(sc[idx].min())) <= 1e-5 * float(np.abs(sc).max()) + 1e-30, (h, t)
            force[(h, t)] = got
    assert len(force) <= 2
    ref = oracle_eval(Qh, K, V, Kh, Vh, force_sel=force, o_base=O.cpu().numpy(), rows=rows, **knobs)
    _bar(out.cpu().numpy().transpose(1, 0, 2), ref, sel, V, Vh, knobs["k_corr_scale"], 2, rows=sorted(sel), max_frac=0.25)
    n = T // 2 + 1  # the same rows in a shorter prompt
    short, sdg, _ = _run(arrays, n, knobs, cap, O=O)
    assert torch.equal(short, out[:, :n]) and torch.equal(sdg, dg[:, :n])


@pytest.mark.parametrize("D", [64, 128])
def test_later_infinities_stay_out(D):
    """Infinities and NaN in token T - 3: every earlier row as without them."""
    print(f"carekv_eval later infinities D={D}", flush=True)
    T, knobs = 75, KNOBS["both-norm"]
    arrays = _rand_case(2, 1, D, T, seed=3)
    out, dg, O = _run(arrays, T, knobs, 4)
    for which in (1, 2, 3, 4):
        bad = [x.copy() for x in arrays]
        bad[which][:, T - 3, 5] = F16(np.inf)
        bad[which][:, T - 3, 9] = F16(np.nan)
        o2, d2, _ = _run(bad, T, knobs, 4, O=O)
        assert torch.equal(o2[:, :T - 3], out[:, :T - 3]) and torch.equal(d2[:, :T - 3], dg[:, :T - 3]), which


def test_value_equal_to_output():
    """One token holds all of a row's weight, so V_hat_j = o up to fp16: the
    distance ||V_hat_j - o|| comes from the difference itself, and a token
    with V_hat_j = o exactly scores 0 as in the oracle."""
    print("carekv_eval value equal to the output", flush=True)
    T, knobs = 40, dict(KNOBS["both-raw"], v_score="output_aware")
    Qh, K, V, Kh, Vh = arrays = _rand_case(2, 1, 64, T, seed=5)
    Kh[:, 3], Qh[:] = 4.0, 4.0  # every row's weight on token 3
    out, dg, O = _run(arrays, T, knobs, 8)
    diag = {}
    oracle_eval(Qh, K, V, Kh, Vh, diag=diag, o_base=O.cpu().numpy(), **knobs)
    dgn, force, sel = dg.cpu().numpy(), {}, {}
    for (h, t), (idx, sc) in diag.items():
        got = dgn[h, t][dgn[h, t] >= 0]
        sel[(h, t)] = force[(h, t)] = got
        if not np.array_equal(got, idx):
            assert abs(float(sc[got].min()) - float(sc[idx].min())) <= 1e-5 * float(np.abs(sc).max()) + 1e-30, (h, t)
    ref = oracle_eval(Qh, K, V, Kh, Vh, force_sel=force, o_base=O.cpu().numpy(), **knobs)
    _bar(out.cpu().numpy().transpose(1, 0, 2), ref, sel, V, Vh, knobs["k_corr_scale"], 2)
