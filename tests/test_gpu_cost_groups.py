"""The differentiable cost's tiles, groups and camera chunks where they can go
wrong, against the FP64 oracle: points that fill a tile exactly, fall one short of
it or exceed it, points and cameras without observations, a problem without
observations, and each gradient asked for alone."""
import numpy as np
import pytest

from nav24_amd import problems
from nav24_amd.abi import Problem
from oracle import cost_oracle as co
from parity_util import say

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 1e-11  # the repository's bar for this comparison (sums of FP64 terms in another order)


def counted(seed, counts, n_cam=6, idle_cam=False):
    """A problem whose point q has counts[q] observations (repeated from the
    generated ones); with idle_cam its last camera has none."""
    g = problems.params_for(4, seed)
    g.n_pt, g.n_cam = len(counts), n_cam
    p = problems.make(g)
    keep = []
    for q, n in enumerate(counts):
        own = np.flatnonzero((p.obs_pt == q) & ((p.obs_cam != n_cam - 1) | (not idle_cam)))
        keep.append(np.resize(own, n if len(own) else 0))
    keep = np.concatenate(keep).astype(int)
    r = Problem(T_cw=p.T_cw, X=p.X, obs_cam=p.obs_cam[keep], obs_pt=p.obs_pt[keep], obs_uv=p.obs_uv[keep])
    r.fx, r.fy, r.cx, r.cy, r.dist = p.fx, p.fy, p.cx, p.cy, p.dist
    return r


def reference(probs, T, X, intr):
    out, c0, p0 = [], 0, 0
    for p in probs:
        out.append(co.cost_and_grad(T[c0:c0 + len(p.T_cw)], X[p0:p0 + len(p.X)], p.obs_cam, p.obs_pt, p.obs_uv, intr, True))
        c0, p0 = c0 + len(p.T_cw), p0 + len(p.X)
    return (np.array([r[0] for r in out]), np.concatenate([r[1] for r in out]), np.concatenate([r[2] for r in out]),
            sum(r[3] for r in out))


CASES = {
    "one observation": [[1]],
    "a full tile and one more": [[256, 1]],
    "one short, then over": [[255, 257, 3]],
    "a point of several rounds": [[3, 700, 0, 5]],
    "many small points": [[4] * 200],
    "an empty problem between": [[5, 0, 7], [0, 0], [130, 130, 2]],
    "as many tiles as groups": [[256] * 2048],
    "one tile more": [[256] * 2049],
    "groups of three, two problems": [[256] * 2049, [256] * 2050],
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("idle_cam", [False, True])
def test_layouts_match_oracle(name, idle_cam):
    from nav24_amd import diffcost
    probs = [counted(3 + k, c, idle_cam=idle_cam) for k, c in enumerate(CASES[name])]
    T, X = np.concatenate([p.T_cw for p in probs]), np.concatenate([p.X for p in probs])
    q = probs[0]
    intr = np.array([q.fx, q.fy, q.cx, q.cy, *q.dist])
    b = diffcost.CostBatch(probs)
    dT, dX, dI = (torch.tensor(a, device="cuda") for a in (T, X, intr))
    ref = reference(probs, T, X, intr)
    r = b.eval(dT, dX, dI)
    for what, g, want in zip(("cost", "pose", "point", "intr"), (r.cost, r.g_pose, r.g_X, r.g_intr), ref):
        err = np.abs(g.cpu().numpy() - want).max() / max(np.abs(want).max(), 1e-300)
        say(f"{name}, {what}: {err:.1e}")
        assert err <= TOL
    seen = np.bincount(np.concatenate([p.obs_pt + sum(len(o.X) for o in probs[:k]) for k, p in enumerate(probs)]),
                       minlength=len(X)) > 0
    assert torch.count_nonzero(r.g_X[torch.tensor(~seen, device="cuda")]) == 0
    # each gradient alone: the same bits, nothing else written
    lib, stream = diffcost.lib(), torch.cuda.current_stream().cuda_stream
    for k in range(3):
        cost = torch.full_like(r.cost, -1.0)
        got = [torch.full_like(t, -1.0) for t in (r.g_pose, r.g_X, r.g_intr)]
        ptr = [t.data_ptr() if j == k else None for j, t in enumerate(got)]
        b._check(lib.nav_ba_cost_eval(b._h, diffcost.NAV_BA_COST_F64, dT.data_ptr(), dX.data_ptr(), dI.data_ptr(),
                                      cost.data_ptr(), *ptr, stream))
        assert torch.equal(cost, r.cost) and torch.equal(got[k], (r.g_pose, r.g_X, r.g_intr)[k])
        assert all(bool((t == -1.0).all()) for j, t in enumerate(got) if j != k)
    assert torch.equal(b.eval(dT, dX, dI, grad=False).cost, r.cost)
    b.close()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n_cam,n_pt", [(2, 1), (4, 341), (4, 342), (257, 400)])  # 1 024 point entries per workgroup
def test_scaled_gradients_in_one_kernel(dtype, n_cam, n_pt):
    """The backward's one kernel against the product with the pose kernel's result
    and the saved gradients: the same operations, so the same bits; with a graph
    of the backward the products are differentiable in the incoming gradient."""
    from nav24_amd.diffcost import BACost, CostBatch, _tangent_grad
    p = counted(1, [3] * n_pt, n_cam=n_cam)
    T = torch.tensor(p.T_cw, device="cuda", dtype=dtype)
    gen = torch.Generator().manual_seed(n_cam)
    leaves = [(0.05 * torch.randn(n_cam, 6, generator=gen)).to("cuda", dtype), torch.tensor(p.X, device="cuda", dtype=dtype),
              torch.tensor([p.fx, p.fy, p.cx, p.cy, *p.dist], device="cuda", dtype=dtype)]
    b = CostBatch([p])
    r = b._eval_tangent(*leaves, T, True)[2]
    g = torch.tensor(0.37, device="cuda", dtype=dtype)
    want = [g * _tangent_grad(leaves[0], r.g_pose), g * r.g_X, g * r.g_intr]
    leaves = [t.requires_grad_(True) for t in leaves]
    got = torch.autograd.grad(BACost.apply(*leaves, T, b), leaves, g)
    assert all(torch.equal(a, w) for a, w in zip(got, want))
    (one,) = torch.autograd.grad(BACost.apply(leaves[0].detach(), leaves[1], leaves[2].detach(), T, b), leaves[1], g)
    assert torch.equal(one, want[1])
    gr = g.clone().requires_grad_(True)
    again = torch.autograd.grad(BACost.apply(*leaves, T, b), leaves, gr, create_graph=True)
    (dg,) = torch.autograd.grad(again[2].sum(), gr)
    assert all(torch.equal(a, w) for a, w in zip(again, want)) and torch.allclose(dg, r.g_intr.sum())
    b.close()


def test_batch_of_incoming_gradients():
    """torch.autograd.grad's is_grads_batched runs the backward on a batch at once."""
    from nav24_amd.diffcost import BACost, CostBatch
    p = counted(2, [4] * 20, n_cam=4)
    T = torch.tensor(p.T_cw, device="cuda")
    leaves = [torch.full((4, 6), 0.01, device="cuda", dtype=torch.float64), torch.tensor(p.X, device="cuda"),
              torch.tensor([p.fx, p.fy, p.cx, p.cy, *p.dist], device="cuda")]
    leaves = [t.requires_grad_(True) for t in leaves]
    b = CostBatch([p])
    gs = torch.tensor([1.0, -0.5, 3.0], device="cuda", dtype=torch.float64)
    cost = BACost.apply(*leaves, T, b)
    many = torch.autograd.grad(cost, leaves, gs, is_grads_batched=True, retain_graph=True)
    for k, g in enumerate(gs):
        one = torch.autograd.grad(cost, leaves, g, retain_graph=True)
        assert all(torch.equal(m[k], o) for m, o in zip(many, one))
    b.close()
