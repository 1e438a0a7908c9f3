"""``carekv_prefill_eval`` with infinities and NaN: rows that do not read such a
token keep their bits, whatever the other rows of their block read; rows that
see one select as the fp32 formulas say."""
import numpy as np
import pytest
import torch

from test_gpu_prefill_eval import F16, KNOBS, _rand_case
from test_gpu_prefill_eval_edges import _need_gpu, _run  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,T,at", [(64, 600, 597), (128, 600, 581), (64, 2400, 2390), (128, 4700, 4698)])
@pytest.mark.parametrize("which", [2, 4])  # V, V_hat
def test_rows_that_do_not_read_it(D, T, at, which):
    """Half of the tokens are read: the wave that holds the token sums many others of each row."""
    print(f"carekv_eval non-finite token D={D} T={T} at={at} which={which}", flush=True)
    knobs = dict(KNOBS["both-raw"], ratio=0.5)
    arrays = _rand_case(2, 1, D, T, seed=T + D)
    cap = T // 2 + 2
    out, dg, O = _run(arrays, T, knobs, cap)
    bad = [x.copy() for x in arrays]
    bad[which][:, at, 5] = F16(np.inf)
    bad[which][:, at, 9] = F16(np.nan)
    o2, d2, _ = _run(bad, T, knobs, cap, O=O)
    assert torch.equal(o2[:, :at], out[:, :at]) and torch.equal(d2[:, :at], dg[:, :at])
    assert not bool(torch.isfinite(o2[:, at:, 9]).any())  # rows that see the token read it


@pytest.mark.parametrize("D", [64, 128])
def test_infinite_distance_with_means(D):
    """V_hat infinite in token 20, o_base finite: the token's scores and both
    means are infinite, every other score over them is 0.  The token (infinity
    over infinity) comes first, then the lowest tokens; its channel is not
    finite, the others are corrected from the tokens read."""
    print(f"carekv_eval infinite distance D={D}", flush=True)
    T, at, knobs = 75, 20, dict(KNOBS["both-norm"], ratio=0.2, v_score="output_aware")
    arrays = _rand_case(2, 1, D, T, seed=3)
    cap = 20
    out, dg, O = _run(arrays, T, knobs, cap)
    bad = [x.copy() for x in arrays]
    bad[4][:, at, 5] = F16(np.inf)
    o2, d2, _ = _run(bad, T, knobs, cap, O=O)
    assert torch.equal(o2[:, :at], out[:, :at]) and torch.equal(d2[:, :at], dg[:, :at])
    for t in range(at, T):
        k = max(knobs.get("min_residuals", 1), int((t + 1) * knobs["ratio"]))
        want = sorted([at] + [j for j in range(t + 1) if j != at][:k - 1])
        for h in range(2):
            assert d2[h, t][d2[h, t] >= 0].tolist() == want, (h, t)
    chan = torch.arange(D, device="cuda") != 5
    assert bool(torch.isfinite(o2[:, :, chan]).all()) and not bool(torch.isfinite(o2[:, at:, 5]).any())


@pytest.mark.parametrize("D", [64, 128])
def test_infinite_score(D):
    """q.K_hat = +infinity in token 20: the softmax of every row that sees it is NaN, as is the row."""
    print(f"carekv_eval infinite score D={D}", flush=True)
    T, at, knobs = 75, 20, KNOBS["both-raw"]
    arrays = _rand_case(2, 1, D, T, seed=4)
    arrays = [np.abs(arrays[0])] + [x.copy() for x in arrays[1:]]
    out, dg, O = _run(arrays, T, knobs, 4)
    arrays[3][:, at] = F16(np.inf)
    o2, d2, _ = _run(arrays, T, knobs, 4, O=O)
    assert torch.equal(o2[:, :at], out[:, :at]) and torch.equal(d2[:, :at], dg[:, :at])
    assert bool(torch.isnan(o2[:, at:]).all())
