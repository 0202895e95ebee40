"""Results in caller order (fetch): points without observations come back as
the caller gave them, also when a second call with the same structure moved
them; observation counts around the flags' 16-byte steps; empty windows and
poses of a batch; the same bits as a solve of each window alone."""
import numpy as np
import pytest

from nav24_amd import problems
from nav24_amd.abi import NAV_BA_FP64, NAV_BA_STOP_EMPTY, Problem, workload_options

pytestmark = pytest.mark.gpu


def options():
    o = workload_options(3)
    o.precision, o.n_iter = NAV_BA_FP64, 2
    return o


def window(seed, n_obs, unseen):
    """A window of exactly n_obs observations, `unseen` points of which have none."""
    p = problems.workload(3, seed=seed, n_cam=7, n_pt=300, obs_min=3)
    last = np.flatnonzero(p.obs_pt >= p.n_pt - unseen)
    keep = np.ones(p.n_obs, bool)
    keep[last] = False
    keep &= np.cumsum(keep) <= n_obs
    assert keep.sum() == n_obs
    return Problem(T_cw=p.T_cw, X=p.X, obs_cam=p.obs_cam[keep], obs_pt=p.obs_pt[keep], obs_uv=p.obs_uv[keep],
                   fx=p.fx, fy=p.fy, cx=p.cx, cy=p.cy, cam_fixed=p.cam_fixed)


def moved(p, d):
    return Problem(T_cw=p.T_cw, X=p.X + d, obs_cam=p.obs_cam, obs_pt=p.obs_pt, obs_uv=p.obs_uv, fx=p.fx, fy=p.fy,
                   cx=p.cx, cy=p.cy, cam_fixed=p.cam_fixed)


@pytest.mark.parametrize("n_obs", [399, 400, 401])
@pytest.mark.parametrize("unseen", [0, 5])
def test_unobserved_points_and_flags(n_obs, unseen):
    from nav24_amd.ba import GraphOptimHip
    p, o = window(1, n_obs, unseen), options()
    seen = np.bincount(p.obs_pt, minlength=p.n_pt) > 0
    s = GraphOptimHip(0)
    for q in (p, moved(p, 0.01)):  # the second call takes the cached index
        r = s.solve(q, o)
        assert np.array_equal(r.X[~seen], q.X[~seen])
        assert not np.array_equal(r.X[seen], q.X[seen])
        assert r.outlier.shape == (n_obs,) and int(r.outlier.sum()) == r.n_outliers
        R = r.T_cw[:, :9].reshape(-1, 3, 3)
        assert np.abs(R @ R.transpose(0, 2, 1) - np.eye(3)).max() < 1e-14
    assert s.prepare_cached
    s.close()


def test_batch_equals_single_and_empty_windows_are_returned():
    from nav24_amd.ba import GraphOptimHip
    o = options()
    empty = Problem(T_cw=np.tile(np.r_[np.eye(3).ravel(), 1.0, 2.0, 3.0], (2, 1)), X=np.arange(9.0).reshape(3, 3),
                    obs_cam=np.zeros(0), obs_pt=np.zeros(0), obs_uv=np.zeros((0, 2)))
    wins = [window(1, 399, 5), empty, window(2, 407, 0)]
    s = GraphOptimHip(0)
    got = s.solve_batched(wins, o)
    s.set_schur_kernel(2)  # the batch's kernel, for the same order of sums
    for w, g in zip(wins, got):
        if w is empty:
            assert g.stop_reason == NAV_BA_STOP_EMPTY and g.iterations == 0
            assert np.array_equal(g.T_cw, w.T_cw) and np.array_equal(g.X, w.X)
            continue
        r = s.solve(w, o)
        for k in ("T_cw", "X", "outlier", "cost_history"):
            assert np.array_equal(getattr(g, k), getattr(r, k)), k
    s.close()


@pytest.mark.parametrize("n_win", [1, 3, 65])  # a window, few of them, more than the host reads between bursts
def test_results_without_pinned_memory(n_win):
    """Where the results' buffer cannot be pinned, they come through pageable memory."""
    from nav24_amd.ba import GraphOptimHip, lib
    o = options()
    wins = [window(1 + k % 3, 399 + k % 3, 5 * (k % 2)) for k in range(n_win)]
    s = GraphOptimHip(0)
    s.prepare_batched(wins, o)
    got = []
    for pinned in (1, 0, 1):
        assert lib().nav_ba_debug_set_pinned(s._h, pinned) == 0
        s.run()
        got.append(s.fetch_batched())
    s.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            for k in ("T_cw", "X", "outlier", "cost_history"):
                assert np.array_equal(getattr(a, k), getattr(b, k)), k
            assert (a.iterations, a.trials, a.n_outliers, a.final_cost) == (b.iterations, b.trials, b.n_outliers, b.final_cost)
