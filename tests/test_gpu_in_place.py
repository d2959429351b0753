"""Outputs over inputs: the two-pass kernels, in launches of whole blocks, since
a block's stencils must read its nodes before any launch overwrites them."""
import pytest

pytestmark = pytest.mark.gpu


def _plan(bl, prm, monkeypatch, pipe=None, gib=None):
    import sympygr_amd as sgr
    for k, v in (("SGR_PIPE_CHUNKS", pipe), ("SGR_WS_GIB", gib)):
        if v is None:
            monkeypatch.delenv(k, raising=False)
        else:
            monkeypatch.setenv(k, v)
    plan = sgr.Plan(bl, prm)
    for k in ("SGR_PIPE_CHUNKS", "SGR_WS_GIB"):
        monkeypatch.delenv(k, raising=False)
    return plan


def _tiling(kind, sizes=(16, 17)):
    """Blocks of two sizes in turn (8^3 tiles and, in two-pass plans, tiles of
    another shape), all faces of half of them flagged."""
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.BlockList()
    for b in range(8):
        n = sizes[b % 2] + 6
        lo = (-1.0 + 0.1 * b, -0.5, -0.7)
        bl.add((n, n, n), lo, tuple(v + 0.04 * (n - 1) for v in lo), 63 if b & 2 else 0)
    kw = dict(adv="upwind", ko_sigma=0.1)
    if kind == "mixed":
        kw["precision"] = "mixed"
    elif kind == "ccz4":
        kw["formulation"] = "ccz4"
    elif kind == "tvb5":
        kw["dissipation"] = "tvb5"
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="ccz4" if kind == "ccz4" else "perturbed", seed=5,
                         amp=1e-2, lo=-1.0, L=2.0)
    return bl, u, sgr.params(**kw)


@pytest.mark.parametrize("kind", ["fp64", "mixed", "ccz4", "tvb5"])
def test_rhs_in_place_in_several_launches(kind, monkeypatch):
    """In place over several workspace chunks, consecutive and pipelined: the
    bits of in place in one launch, and to rounding the right-hand side of
    separate arrays (1e-12 of each field's maximum; mixed precision runs the
    same kernels there: equal).  A workspace that does not hold the largest
    block is refused."""
    import torch
    import sympygr_amd as sgr
    bl, u, prm = _tiling(kind)
    one = _plan(bl, prm, monkeypatch)
    assert one.info().chunks == 1
    ref, sep = u.clone(), u.clone()
    one.rhs(ref, ref)
    one.rhs(sep, u)
    torch.cuda.synchronize()
    if kind == "mixed":
        assert torch.equal(ref, sep)
    for f in range(u.shape[0]):  # (ghost nodes hold the inputs in both)
        inner = sep[f] != u[f]
        assert (ref[f] - sep[f]).abs().max() <= 1e-12 * sep[f][inner].abs().max(), f
    nf = u.shape[0]
    tile = 512 * ((one.info().derivative_slots - nf) * (4 if kind == "mixed" else 8) + nf * 8)  # workspace of a tile
    largest = one.info().tiles // 4 - 8  # four blocks of 16^3 (8 tiles each), four of 17^3
    ran = 0
    for pipe, gib in (("0", "0.01"), (None, "0.01"), ("5", None)):
        plan = _plan(bl, prm, monkeypatch, pipe, gib)
        info = plan.info()
        fits = info.workspace_bytes >= largest * tile
        print(f"{kind}: chunks={info.chunks} pipelined={info.pipelined} fits={fits}", flush=True)
        assert info.chunks > 1
        got = u.clone()
        if not fits:
            with pytest.raises(sgr.SgrError, match="separate output arrays"):
                plan.rhs(got, got)
            continue
        ran += 1
        plan.rhs(got, got)
        torch.cuda.synchronize()
        assert torch.equal(got, ref), (pipe, gib)
    assert ran


def test_rhs_in_place_refused_if_a_block_does_not_fit(monkeypatch):
    """A workspace of fewer tiles than a block has: refused, nothing written;
    the same plan takes separate arrays."""
    import torch
    import sympygr_amd as sgr
    bl, u, prm = _tiling("fp64", sizes=(24, 13))
    plan = _plan(bl, prm, monkeypatch, None, "0.004")
    got = u.clone()
    with pytest.raises(sgr.SgrError, match="separate output arrays"):
        plan.rhs(got, got)
    out, ref = torch.full_like(u, 5.0), torch.full_like(u, 5.0)
    plan.rhs(out, u)
    _plan(bl, prm, monkeypatch).rhs(ref, u)
    torch.cuda.synchronize()
    assert torch.equal(got, u) and torch.equal(out, ref)


def _rows_rel(bl, a, b):
    """max |a - b| over the interior nodes, over each row's max |b|."""
    import torch
    d, m = [], []
    for i in range(len(bl)):
        s = bl.sz[i]
        o = slice(bl.offsets[i], bl.offsets[i] + s[0] * s[1] * s[2])
        x, y = (v[:, o].reshape(-1, s[2], s[1], s[0])[:, 3:-3, 3:-3, 3:-3] for v in (a, b))
        d.append((x - y).abs().amax(dim=(1, 2, 3)))
        m.append(y.abs().amax(dim=(1, 2, 3)))
    return (torch.stack(d).amax(0) / torch.stack(m).amax(0)).max().item()


@pytest.mark.parametrize("kind", ["fp64", "mixed"])
@pytest.mark.parametrize("psi4,row", [(False, 12), (False, 1), (False, 3), (True, 18), (True, 12), (True, 3),
                                       (True, 6)])
def test_constraints_over_inputs(kind, psi4, row, monkeypatch):
    """Over rows that the constraints read (gt, At, chi to Gt) in several
    launches, and over rows that they do not (shift and B): the values of
    separate output arrays, to the bounds that both keep against the oracle,
    1e-11 of a row's maximum and 1e-5 in mixed precision."""
    import torch
    bl, u, prm = _tiling(kind)
    plan = _plan(bl, prm, monkeypatch)
    n = 6 if psi4 else 4
    sep = torch.full((n, u.shape[1]), 5.0, dtype=torch.float64, device="cuda")
    over = u.clone()
    call = plan.constraints_psi4 if psi4 else plan.constraints
    call(u, sep)
    call(over, over[row:row + n])
    torch.cuda.synchronize()
    assert _rows_rel(bl, over[row:row + n], sep) <= (1e-5 if kind == "mixed" else 1e-11)
    rest = [f for f in range(24) if not row <= f < row + n]
    assert torch.equal(over[rest], u[rest])


def test_constraints_over_inputs_refused_if_a_block_does_not_fit(monkeypatch):
    """One block of 27 tiles: its workspace holds the right-hand side's
    derivatives of them, not the constraints'."""
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.BlockList()
    bl.add((30, 30, 30), (-0.7, -0.5, -0.6), (0.46, 0.66, 0.56), 0)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="perturbed", seed=5, amp=1e-2, lo=-1.0, L=2.0)
    plan = sgr.Plan(bl, sgr.params(adv="upwind"))
    over = u.clone()
    with pytest.raises(sgr.SgrError, match="separate output arrays"):
        plan.constraints(over, over[12:16])
    torch.cuda.synchronize()
    assert torch.equal(over, u)
    sep = torch.zeros((4, bl.total), dtype=torch.float64, device="cuda")
    plan.constraints(u, sep)
    plan.constraints(over, over[8:12])
    torch.cuda.synchronize()
    assert _rows_rel(bl, over[8:12], sep) <= 1e-11


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_rochester_rhs_in_place(precision, monkeypatch):
    """The Rochester shift equation reads Gt at the point: before its own
    output is stored over it.  The bits of separate arrays (same kernels)."""
    import torch
    import sympygr_amd as sgr
    bl, u, _ = _tiling("fp64")
    prm = sgr.params(adv="upwind", ko_sigma=0.1, gauge="rochester", xi=(1, 1, 1), precision=precision)
    for pipe in (None, "5"):
        plan = _plan(bl, prm, monkeypatch, pipe)
        sep, got = u.clone(), u.clone()
        plan.rhs(sep, u)
        plan.rhs(got, got)
        torch.cuda.synchronize()
        assert torch.equal(got, sep)
