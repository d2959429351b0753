"""The one-pass right-hand side (FP64, BSSN, standard gauge, Kreiss-Oliger) at
the sizes where its tiling can go wrong: blocks smaller than a tile, one tile,
one point more or less, axes of different sizes, flagged faces whose closures
reach into one or two tiles, and more tiles than workgroups; and calls whose
outputs share memory with the inputs, which take the two passes.  Against the
CPU oracle at the FP64 bar, 1e-12 normwise per field (both evaluate the same
stencils bit for bit; the algebra differs in rounding only)."""
import numpy as np
import pytest

from helpers import interior, normwise

pytestmark = pytest.mark.gpu

SIZES = [(7, 7, 7), (7, 9, 16), (8, 8, 8), (9, 8, 7), (15, 16, 17), (13, 33, 8), (10, 11, 12)]


def _block(n, bflag, seed):
    from sympygr_amd import data
    bl = data.BlockList()
    sz = tuple(k + 6 for k in n)
    pmin = (-0.6, -0.5, -0.7)
    bl.add(sz, pmin, tuple(p + 0.05 * (s - 1) for p, s in zip(pmin, sz)), bflag)
    m = max(sz)
    u = data.perturbed_flat_block(seed=seed, n=m, amp=1e-2, pmin=pmin, pmax=tuple(p + 0.05 * (m - 1) for p in pmin))
    u = u.reshape(24, m, m, m)[:, :sz[2], :sz[1], :sz[0]].reshape(24, -1)
    return bl, np.ascontiguousarray(u)


def _oracle(bl, u, adv):
    import pyoracle as po
    return po.rhs_block(u, bl.sz[0], bl.pmin[0], bl.pmax[0], bl.bflag[0],
                        po.make_params(upwind=adv == "upwind", ko_sigma=0.1))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bflag,adv", [(0, "upwind"), (63, "upwind"), (38, "centred")])
def test_edge_sizes_against_oracle(n, bflag, adv):
    import torch
    import sympygr_amd as sgr
    bl, u = _block(n, bflag, 3 + n[0])
    prm = sgr.params(adv=adv, ko_sigma=0.1)
    du = torch.from_numpy(u).cuda()
    ref = interior(_oracle(bl, u, adv), bl.sz[0])
    out = torch.full_like(du, 5.0)
    sgr.Plan(bl, prm).rhs(out, du)
    one = torch.full_like(du, 5.0)
    sgr.rhs_block_noalloc(one, du, 0, bl.pmin[0], bl.pmax[0], bl.sz[0], bflag, prm)
    torch.cuda.synchronize()
    assert torch.equal(one, out)
    got = out.cpu().numpy()
    assert normwise(interior(got, bl.sz[0]), ref).max() <= 1e-12
    ghosts = np.ones(got[0].size, dtype=bool).reshape(bl.sz[0][::-1])
    ghosts[3:-3, 3:-3, 3:-3] = False
    assert (got[:, ghosts.reshape(-1)] == 5.0).all()


def test_outputs_over_inputs():
    """In place: the two-pass kernels, same result to rounding."""
    import torch
    import sympygr_amd as sgr
    bl, u = _block((13, 16, 9), 21, 8)
    plan = sgr.Plan(bl, sgr.params(adv="upwind", ko_sigma=0.1))
    du = torch.from_numpy(u).cuda()
    plan.rhs(du, du)
    torch.cuda.synchronize()
    ref = interior(_oracle(bl, u, "upwind"), bl.sz[0])
    assert normwise(interior(du.cpu().numpy(), bl.sz[0]), ref).max() <= 1e-12


@pytest.mark.parametrize("faces", [False, True])
def test_many_tiles_equal_single_blocks(faces):
    """More tiles than workgroups (several tiles each, fetched ahead across
    tile boundaries, both kinds of tiles in one list, 8^3 and general shapes):
    every block equals the same block evaluated by itself, bit for bit."""
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.BlockList()
    for b in range(80):
        n = (16, 17, 24, 13)[b % 4] + 6
        lo = -1.0 + 0.02 * b
        bl.add((n, n, n), (lo, -0.5, -0.7), (lo + 0.04 * (n - 1), -0.5 + 0.04 * (n - 1), -0.7 + 0.04 * (n - 1)),
               (b * 7) & 63 if faces else 0)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="perturbed", seed=5, amp=1e-2, lo=-1.0, L=2.0)
    prm = sgr.params(adv="upwind", ko_sigma=0.1)
    out = torch.full_like(u, 5.0)
    plan = sgr.Plan(bl, prm)
    assert plan.info().tiles > 512
    plan.rhs(out, u)
    ref = torch.full_like(u, 5.0)
    for b in range(len(bl)):
        sgr.rhs_block(ref, u, bl.offsets[b], bl.pmin[b], bl.pmax[b], bl.sz[b], bl.bflag[b], prm)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bflag,adv", [(0, "upwind"), (63, "upwind"), (38, "centred")])
def test_ccz4_edge_sizes_against_oracle(n, bflag, adv):
    """The CCZ4 form of the kernel (25 fields, the divergence of Gamma-hat added
    to the K and Theta equations after their own fields) at the same sizes and
    bar, and a first RK stage from it: u + dt/2 rhs and rhs dt/6 + u."""
    import pyoracle as po
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    kappa = (0.02, 0.1, 0.5)
    bl, _ = _block(n, bflag, 0)
    m = max(bl.sz[0])
    cube = data.BlockList()
    cube.add((m,) * 3, bl.pmin[0], tuple(p + 0.05 * (m - 1) for p in bl.pmin[0]), 0)
    u = data.fill_blocks(cube, kind="ccz4", seed=4, amp=1e-2, lo=-1.05, L=2.1)
    s = bl.sz[0]
    u = np.ascontiguousarray(u.reshape(25, m, m, m)[:, :s[2], :s[1], :s[0]].reshape(25, -1))
    prm = sgr.params(adv=adv, ko_sigma=0.1, formulation="ccz4", kappa=kappa)
    ref = po.rhs_block(u, s, bl.pmin[0], bl.pmax[0], bflag,
                       po.make_params(upwind=adv == "upwind", ko_sigma=0.1, ccz4=True, kappa=kappa))
    du = torch.from_numpy(u).cuda()
    out = torch.full_like(du, 5.0)
    plan = sgr.Plan(bl, prm)
    plan.rhs(out, du)
    one = torch.full_like(du, 5.0)
    sgr.rhs_block_noalloc(one, du, 0, bl.pmin[0], bl.pmax[0], s, bflag, prm)
    acc, nxt = torch.zeros_like(du), torch.zeros_like(du)
    dt = 0.0625
    plan.rk4_stage(0, dt, du, du, acc, nxt)
    torch.cuda.synchronize()
    assert torch.equal(one, out)
    inner = (slice(None), slice(3, -3), slice(3, -3), slice(3, -3))

    def of(a):
        return np.asarray(a).reshape(25, s[2], s[1], s[0])[inner].reshape(25, -1)
    got, r, u0 = of(out.cpu()), of(ref), of(u)
    scale = np.abs(r).max(axis=1) + 1e-300
    assert (np.abs(got - r).max(axis=1) / scale).max() <= 1e-12
    # one rounding of the product, one of the sum
    eps = 2.0 ** -52
    for a, w in ((nxt, 0.5 * dt), (acc, dt / 6.0)):
        assert (np.abs(of(a.cpu()) - (u0 + w * got)) <= 2 * eps * (np.abs(u0) + np.abs(w * got))).all()
    assert (out.cpu().reshape(25, s[2], s[1], s[0])[:, :3] == 5.0).all()


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("diss,bflag", [("tvb3", 0), ("tvb5", 0), ("tvb3", 63), ("tvb5", 63), ("tvb5", 38)])
def test_tvb_edge_sizes_against_oracle(n, diss, bflag):
    """TVB dissipation, added by a pass of its own over the same tiles (one-sided
    forms at the first and last point, closures at flagged faces), same sizes
    and bar; the second and the last RK stage from it, to a rounding of each
    of their terms."""
    import pyoracle as po
    import torch
    import sympygr_amd as sgr
    bl, u = _block(n, bflag, 9 + n[1])
    plan = sgr.Plan(bl, sgr.params(adv="upwind", ko_sigma=0.1, dissipation=diss))
    du = torch.from_numpy(u).cuda()
    out = torch.full_like(du, 5.0)
    plan.rhs(out, du)
    base, dt = torch.full_like(du, 0.25), 0.0625
    acc, nxt, end = base.clone(), torch.full_like(du, 5.0), torch.full_like(du, 5.0)
    plan.rk4_stage(1, dt, base, du, acc, nxt)
    plan.rk4_stage(3, dt, base, du, base, end)
    torch.cuda.synchronize()
    s = bl.sz[0]
    ref = po.rhs_block(u, s, bl.pmin[0], bl.pmax[0], bflag, po.make_params(upwind=True, ko_sigma=0.1, dissipation=diss))
    got = interior(out.cpu().numpy(), s)
    assert normwise(got, interior(ref, s)).max() <= 1e-12
    eps = 2.0 ** -52
    for a, w in ((acc, dt / 3.0), (nxt, dt / 2.0), (end, dt / 6.0)):
        a = interior(a.cpu().numpy(), s)
        # the right-hand side and the dissipation are added one after the other
        scale = 0.25 + np.abs(w * got).max(axis=(1, 2, 3), keepdims=True)
        assert (np.abs(a - (0.25 + w * got)) <= 4 * eps * scale).all()
    for a in (out, nxt, end):
        a = a.cpu().numpy().reshape(24, s[2], s[1], s[0])
        assert (a[:, :3] == 5.0).all() and (a[:, :, :, -3:] == 5.0).all()


@pytest.mark.parametrize("sizes", [(9, 9, 9), (10, 10, 10), (11, 12, 12), (18, 20, 9), (26, 27, 7), (7, 33, 12)])
def test_shapes_chosen_by_the_tile_count(sizes):
    """Enough blocks that the rule picks larger tiles than 8^3 (a block by itself
    takes 8^3): fewer tiles than 8^3 would make, and the same bits."""
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.BlockList()
    cubes = 1
    for k in sizes:
        cubes *= -(-k // 8)
    count = 256 // cubes + 5
    for b in range(count):
        lo = (-1.0 + 0.02 * b, -0.5, -0.7)
        sz = tuple(k + 6 for k in sizes)
        bl.add(sz, lo, tuple(p + 0.04 * (s - 1) for p, s in zip(lo, sz)), (b * 11) & 63)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="perturbed", seed=5, amp=1e-2, lo=-1.0, L=2.0)
    prm = sgr.params(adv="upwind", ko_sigma=0.1)
    out, ref = torch.full_like(u, 5.0), torch.full_like(u, 5.0)
    plan = sgr.Plan(bl, prm)
    assert plan.info().tiles < cubes * count
    plan.rhs(out, u)
    for b in range(count):
        sgr.rhs_block(ref, u, bl.offsets[b], bl.pmin[b], bl.pmax[b], bl.sz[b], bl.bflag[b], prm)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
