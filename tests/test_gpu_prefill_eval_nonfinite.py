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
