"""The constraints and Psi4 in one kernel at the sizes where its tiling can go
wrong (see test_gpu_one_pass), against the CPU oracle: every row within 1e-11
of its own maximum in FP64 and 1e-5 in mixed precision (derivatives staged in
FP32), the bounds that hold for whole tiles.  Psi4 has no value on the polar axis
(x = y = 0 leaves the tetrad's angle to the rounding of the coordinates): its
rows leave those points out.  And outputs that share memory with
the inputs, which take the two passes."""
import numpy as np
import pytest

from test_gpu_one_pass import SIZES, _block

pytestmark = pytest.mark.gpu


def _interior(a, sz):
    return a.reshape(a.shape[0], sz[2], sz[1], sz[0])[:, 3:-3, 3:-3, 3:-3].reshape(a.shape[0], -1)


def _rel(got, ref):
    return (np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)).max()


def _off_axis(bl):
    x, y, z = (np.arange(3, s - 3) for s in bl.sz[0])
    on = (np.abs(bl.pmin[0][0] + 0.05 * x)[None, None, :] < 1e-9) & (np.abs(bl.pmin[0][1] + 0.05 * y)[None, :, None] < 1e-9)
    return ~np.broadcast_to(on, (z.size, y.size, x.size)).reshape(-1)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bflag,precision", [(0, "fp64"), (63, "fp64"), (38, "mixed")])
def test_edge_sizes_against_oracle(n, bflag, precision):
    import pyoracle as po
    import torch
    import sympygr_amd as sgr
    bl, u = _block(n, bflag, 5 + n[2])
    plan = sgr.Plan(bl, sgr.params(adv="upwind", precision=precision))
    du = torch.from_numpy(u).cuda()
    out = torch.full((6, u.shape[1]), 5.0, dtype=torch.float64, device="cuda")
    four = torch.full((4, u.shape[1]), 5.0, dtype=torch.float64, device="cuda")
    plan.constraints_psi4(du, out)
    plan.constraints(du, four)
    torch.cuda.synchronize()
    ref = po.constraints_block(u, bl.sz[0], bl.pmin[0], bl.pmax[0], bflag, psi4=True)
    ref = _interior(ref, bl.sz[0])
    got, got4 = out.cpu().numpy(), four.cpu().numpy()
    tol = 1e-11 if precision == "fp64" else 1e-5
    off = _off_axis(bl)
    all6 = _interior(got, bl.sz[0])
    assert _rel(all6[:4], ref[:4]) <= tol
    assert _rel(all6[4:, off], ref[4:, off]) <= tol
    assert _rel(_interior(got4, bl.sz[0]), ref[:4]) <= tol
    ghosts = np.ones(got[0].size, dtype=bool).reshape(bl.sz[0][::-1])
    ghosts[3:-3, 3:-3, 3:-3] = False
    assert (got[:, ghosts.reshape(-1)] == 5.0).all() and (got4[:, ghosts.reshape(-1)] == 5.0).all()


def test_outputs_over_inputs():
    """Over a shift component and the B fields, which no constraint reads."""
    import torch
    import sympygr_amd as sgr
    bl, u = _block((13, 16, 9), 21, 8)
    plan = sgr.Plan(bl, sgr.params(adv="upwind"))
    du = torch.from_numpy(u).cuda()
    sep = torch.zeros((4, u.shape[1]), dtype=torch.float64, device="cuda")
    plan.constraints(du, sep)
    plan.constraints(du, du[8:12])
    torch.cuda.synchronize()
    assert _rel(_interior(du[8:12].cpu().numpy(), bl.sz[0]), _interior(sep.cpu().numpy(), bl.sz[0])) <= 1e-11
