"""The host-array entry points on both sides of the size up to which a call goes
through the pinned buffer (1 MiB): the same bits from either way in, with the
larger call made so by key points or sets that no result depends on."""
import threading

import numpy as np
import pytest

from nav24_amd.twoview_synth import motion_candidates, synthetic_two_view
from parity_util import say

pytestmark = pytest.mark.gpu

FISHEYE = (380.0, 380.0, 320.0, 240.0, 0.05, -0.01, 0.002, -0.0003)


@pytest.mark.parametrize("n", [1, 131071, 131072, 131073])  # 8 bytes a point: 131072 fill the buffer
def test_undistort_host_equals_device(n):
    torch = pytest.importorskip("torch")
    from nav24_amd.undistort import KannalaBrandt8Hip
    rng = np.random.default_rng(n)
    uv = np.stack([rng.uniform(0, 640, n), rng.uniform(0, 480, n)], 1).astype(np.float32)
    cam = KannalaBrandt8Hip(FISHEYE)
    host, dev = cam.UndistortKeyPoints(uv), cam.undistort_device(torch.from_numpy(uv).cuda()).cpu().numpy()
    say(f"{n} points")
    assert np.array_equal(host.view(np.uint32), dev.view(np.uint32))


@pytest.fixture(scope="module")
def scene():
    from nav24_amd.twoview import TwoViewReconstructionHip
    sc = synthetic_two_view(300, seed=4, planar=False)
    rng = np.random.default_rng(4)
    sets = np.stack([rng.choice(300, 8, replace=False) for _ in range(60)]).astype(np.int32)
    return TwoViewReconstructionHip(), sc, sets


def test_two_view_small_and_large_calls_agree(scene):
    tv, sc, sets = scene
    many = 70_000  # unused key points: 560 KB in each image
    k1 = np.concatenate([sc.kp1, np.zeros((many, 2), np.float32)])
    k2 = np.concatenate([sc.kp2, np.zeros((many, 2), np.float32)])
    small = tv.Hypotheses(sc.kp1, sc.kp2, sc.matches, sets)
    large = tv.Hypotheses(sc.kp1, sc.kp2, sc.matches, np.tile(sets, (150, 1)))  # 1.3 MB of sets and matrices
    for a, b in zip(small, large):
        assert np.array_equal(a.view(np.uint32), b[:len(a)].view(np.uint32))
    H21, H12, F21 = small
    for f, m in ((tv.FindHomographyScores, (H21, H12)), (tv.FindFundamentalScores, (F21,))):
        for a, b in zip(f(sc.kp1, sc.kp2, sc.matches, *m), f(k1, k2, sc.matches, *m)):
            assert np.array_equal(a, b)
    inl = tv.FindFundamentalScores(sc.kp1, sc.kp2, sc.matches, F21)[3]
    motions = motion_candidates(sc, 2, seed=4)
    a = tv.CheckRT(sc.kp1, sc.kp2, sc.matches, inl, sc.K, *motions)
    b = tv.CheckRT(k1, k2, sc.matches, inl, sc.K, *motions)
    n = len(sc.kp1)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[3], b[3])
    assert np.array_equal(a[1], b[1][:, :n]) and np.array_equal(a[2], b[2][:, :n])
    assert not b[2][:, n:].any()


def test_calls_from_several_threads(scene):
    tv, sc, sets = scene
    want = tv.Hypotheses(sc.kp1, sc.kp2, sc.matches, sets)
    bad = []

    def work():
        for _ in range(20):
            got = tv.Hypotheses(sc.kp1, sc.kp2, sc.matches, sets)
            if not all(np.array_equal(a, b) for a, b in zip(got, want)):
                bad.append(1)

    ts = [threading.Thread(target=work) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_null_key_points_are_refused():
    """A count of key points without the array is an error, also where no match
    reads them (n = 0), and 0 key points need none."""
    import ctypes as C
    from nav24_amd import twoview
    L = twoview.lib()
    kp, best, score = (C.c_float * 4)(), C.c_int32(), C.c_float()
    K = (C.c_float * 9)(1, 0, 0, 0, 1, 0, 0, 0, 1)
    t = (C.c_float * 3)()
    ng, par, cs, p3, gd = C.c_int32(), C.c_float(), C.c_float(), (C.c_float * 6)(), (C.c_uint8 * 2)()

    def scored(k1, n1):
        return L.nav_tv_score_homography_host(k1, n1, kp, 2, None, 0, None, None, 0, 1.0, 5.991, None, C.byref(best),
                                              C.byref(score), None, 0)

    def checked(k1, n1):
        return L.nav_tv_check_rt_host(k1, n1, kp, 2, None, None, 0, K, K, t, 1, 4.0, 0.99998, 50, C.byref(ng),
                                      C.byref(par), C.byref(cs), p3, gd, 0)

    for f in (scored, checked):
        assert f(kp, 2) == 0 and f(None, 0) == 0
        assert f(None, 2) != 0
