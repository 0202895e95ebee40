"""The per-window factorisation (16x16 tiles in LDS) at the sizes where its
tiling can go wrong, against the FP64 oracle: one camera, systems that end on a
tile boundary (the right-hand side then has a tile row of its own), one row
short of it and one past it, the largest window, and rows summed from one to
many chunks."""
import numpy as np
import pytest

from nav24_amd import problems
from nav24_amd.abi import NAV_BA_FP64, workload_options
from oracle import oracle
from parity_util import say

pytestmark = pytest.mark.gpu


def window(n_free, n_pt):
    # two fixed cameras beside the free ones; every point in three views or more
    return problems.workload(3, seed=n_free, n_cam=n_free + 2, n_pt=n_pt, obs_min=3, rot_sigma=0.005,
                             trans_sigma=0.01, point_sigma=0.02)


# 6 n_free unknowns: 6 (less than a tile), 18 and 30 (around 16 and 32), 48, 96 and
# 144 (tile multiples), 174 and 180 (the largest tile rows)
@pytest.mark.parametrize("n_free", [1, 3, 5, 8, 9, 16, 24, 29, 30])
@pytest.mark.parametrize("chunk", [0, 64])
def test_window_sizes_match_oracle(n_free, chunk):
    """Three LM iterations.  The two solves differ by the order of their FP64
    sums only; the scene is well conditioned (three views, a few mrad), where the
    repository's parity bars hold: 1e-9 on costs, 1e-6 on poses."""
    from nav24_amd.ba import GraphOptimHip
    p = window(n_free, 400)
    o = workload_options(3)
    o.precision, o.n_iter = NAV_BA_FP64, 3
    ref = oracle.solve(p, o)
    s = GraphOptimHip(0)
    s.set_schur_chunk(chunk)
    one = s.solve(p, o)
    many = s.solve_batched([p, window(2, 300), p], o)
    s.close()
    for r in (one, many[0], many[2]):
        assert (r.iterations, r.trials, r.stop_reason) == (ref.iterations, ref.trials, ref.stop_reason)
        rel = np.abs(r.cost_history - ref.cost_history).max() / ref.cost_history.max()
        dT = np.abs(r.T_cw - ref.T_cw).max()
        say(f"free cameras {n_free}, chunk {chunk}: cost {rel:.1e}, pose {dT:.1e}")
        assert rel <= 1e-9 and dT <= 1e-6
    assert np.array_equal(many[0].T_cw, many[2].T_cw)
