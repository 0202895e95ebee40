"""A run's launches: the linearisation's two sides in one launch or apart (as stage
timing runs them), and its bursts and what the host reads of them, against the FP64 oracle: no,
one and several iterations, on either side of the window count up to which the
final flags go with every burst, with trials that are rejected."""
import numpy as np
import pytest

from nav24_amd import problems
from nav24_amd.abi import NAV_BA_FP64, NAV_BA_MIXED, workload_options
from oracle import oracle
from parity_util import say

pytestmark = pytest.mark.gpu


def window(seed, far):
    # far: a start from which some trials fail (a tenth of a radian, a metre)
    return problems.workload(3, seed=seed, n_cam=4, n_pt=60, obs_min=3, rot_sigma=0.1 if far else 0.005,
                             trans_sigma=1.0 if far else 0.01, point_sigma=0.3 if far else 0.02)


@pytest.mark.parametrize("n_win", [1, 2, 64, 65])
@pytest.mark.parametrize("n_iter", [0, 1, 6])
def test_bursts_match_oracle(n_win, n_iter):
    """The same counts, and costs to the repository's parity bar (1e-9) while the
    paths agree; three distinct windows, so that the oracle solves three."""
    from nav24_amd.ba import GraphOptimHip
    kinds = [window(1, False), window(2, True), window(3, False)]
    o = workload_options(3)
    o.precision, o.n_iter, o.lambda_init = NAV_BA_FP64, n_iter, 1e-4
    refs = [oracle.solve(p, o) for p in kinds]
    s = GraphOptimHip(0)
    rs = s.solve_batched([kinds[k % 3] for k in range(n_win)], o)
    again = s.solve_batched([kinds[k % 3] for k in range(n_win)], o)
    s.close()
    say(f"{n_win} windows, {n_iter} iterations: trials {[r.trials for r in refs]}")
    for k, (r, a) in enumerate(zip(rs, again)):
        ref = refs[k % 3]
        assert (r.iterations, r.trials, r.stop_reason) == (ref.iterations, ref.trials, ref.stop_reason)
        assert np.abs(r.cost_history - ref.cost_history).max() <= 1e-9 * ref.cost_history.max()
        assert abs(r.final_cost - ref.final_cost) <= 1e-9 * ref.cost_history.max()
        assert np.array_equal(r.outlier, ref.outlier) and r.n_outliers == ref.n_outliers
        assert np.array_equal(r.T_cw, a.T_cw) and np.array_equal(r.cost_history, a.cost_history)


@pytest.mark.parametrize("fisheye", [False, True])
@pytest.mark.parametrize("precision", [NAV_BA_FP64, NAV_BA_MIXED])
@pytest.mark.parametrize("n_pt", [40, 1500])  # a camera in one item, in several
def test_linearisation_together_or_apart(fisheye, precision, n_pt):
    from nav24_amd.ba import GraphOptimHip
    p = problems.workload(3, seed=n_pt, n_cam=6, n_pt=n_pt, obs_min=3, rot_sigma=0.005, trans_sigma=0.01)
    if fisheye:
        p = problems.with_kb8(p, seed=1)
    o = workload_options(3)
    o.precision, o.n_iter = precision, 3
    s = GraphOptimHip(0)
    one = s.solve(p, o)
    s.set_timing(True)
    apart = s.solve(p, o)
    s.close()
    assert np.array_equal(one.T_cw, apart.T_cw) and np.array_equal(one.X, apart.X)
    assert np.array_equal(one.cost_history, apart.cost_history) and one.trials == apart.trials


def test_pending_error_of_the_program_stays():
    """An error that the program's own HIP call left is neither taken by a run and a
    fetch nor taken for theirs."""
    import ctypes as C
    from nav24_amd.ba import GraphOptimHip, lib
    hip = lib()  # the runtime that the library is linked to
    o = workload_options(3)
    o.precision, o.n_iter = NAV_BA_FP64, 2
    s = GraphOptimHip(0)
    s.prepare(window(1, False), o)
    s.run()
    want = s.fetch()
    hip.hipGetLastError()
    assert hip.hipMemcpy(None, None, C.c_size_t(8), C.c_int(2)) != 0  # null arrays: refused on the host
    left = hip.hipPeekAtLastError()
    assert left != 0
    s.run()
    got = s.fetch()
    assert hip.hipPeekAtLastError() == left
    hip.hipGetLastError()
    s.close()
    assert np.array_equal(got.T_cw, want.T_cw) and np.array_equal(got.X, want.X)
