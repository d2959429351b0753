"""The two-pass kernels where plans run them (mixed precision and the Rochester
gauge): tile queues against one workgroup per tile, chunk schedules against a
single chunk, and the constraint pass in workspace chunks.  Every point is
computed by the same operations in the same order: equal bit for bit."""
import pytest

pytestmark = pytest.mark.gpu

ENV = ("SGR_STENCIL_QUEUE", "SGR_WS_GIB", "SGR_PIPE_CHUNKS")
KINDS = {"mixed": dict(precision="mixed"), "mixed tvb5": dict(precision="mixed", dissipation="tvb5"),
         "mixed ccz4": dict(precision="mixed", formulation="ccz4"), "rochester": dict(gauge="rochester", xi=(1, 1, 1))}


def _set(n, kind):
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.uniform_tiling(nb=3, n=n, lo=-1.0, hi=1.0, stagger=0.5, faces=True)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="ccz4" if "ccz4" in kind else "perturbed", seed=8,
                         amp=1e-2, lo=-1.0, L=2.0)
    return bl, u, sgr.params(adv="upwind", ko_sigma=0.1, **KINDS[kind])


def _plan(bl, prm, monkeypatch, *values):
    import sympygr_amd as sgr
    for k, v in zip(ENV, values):
        if v is not None:
            monkeypatch.setenv(k, v)
    plan = sgr.Plan(bl, prm)
    for k in ENV:
        monkeypatch.delenv(k, raising=False)
    return plan


# 16^3: 8^3 tiles; 13^3: the tile table's shape
@pytest.mark.parametrize("n", [16, 13])
@pytest.mark.parametrize("kind", list(KINDS))
def test_queues_and_chunks_equal_one_launch(kind, n, monkeypatch):
    import torch
    bl, u, prm = _set(n, kind)
    first = None
    for values in (("0", None, None), ("1", None, None), ("1", "0.01", "0"), ("0", "0.01", "0"), ("1", None, "5"),
                   ("0", None, "5")):
        plan = _plan(bl, prm, monkeypatch, *values)
        info = plan.info()
        assert info.tile_queue == int(values[0]) and (info.chunks > 1) == (values[1:] != (None, None))
        assert info.pipelined == (values[2] == "5")
        out, acc, nxt = torch.full_like(u, 5.0), torch.full_like(u, 3.0), torch.zeros_like(u)
        plan.rhs(out, u)
        plan.rk4_stage(2, 0.01, u, u, acc, nxt)
        torch.cuda.synchronize()
        first = first or (out, acc, nxt)
        assert all(torch.equal(a, b) for a, b in zip(first, (out, acc, nxt))), values


@pytest.mark.parametrize("kind", ["mixed", "rochester"])
def test_constraint_pass_in_chunks(kind, monkeypatch):
    """A two-pass plan with a block of 7 points an axis stages the derivatives
    of the constraints and Psi4 in its workspace."""
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.BlockList()
    for k, n in enumerate((7, 16, 9, 24)):
        lo = (-1.0 + 0.3 * k, -0.51, -0.7)
        bl.add((n + 6,) * 3, lo, tuple(v + 0.04 * (n + 5) for v in lo), (5 * k) & 63)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="perturbed", seed=8, amp=1e-2, lo=-1.0, L=2.0)
    prm = sgr.params(adv="upwind", **KINDS[kind])
    first = None
    for gib in (None, "0.002"):
        out = torch.full((6, bl.total), 5.0, dtype=torch.float64, device="cuda")
        _plan(bl, prm, monkeypatch, None, gib, None).constraints_psi4(u, out)
        torch.cuda.synchronize()
        first = out if first is None else first
        assert torch.equal(out, first)
    # against the one-kernel form on the blocks without the small one, to the
    # bounds that both keep against the oracle
    sub = data.BlockList()
    for b in range(1, len(bl)):
        sub.add(bl.sz[b], bl.pmin[b], bl.pmax[b], bl.bflag[b])
    us = u[:, bl.offsets[1]:].contiguous()
    one = torch.full((6, sub.total), 5.0, dtype=torch.float64, device="cuda")
    sgr.Plan(sub, prm).constraints_psi4(us, one)
    torch.cuda.synchronize()
    for b in range(len(sub)):
        s = sub.sz[b]
        o = slice(sub.offsets[b], sub.offsets[b] + s[0] * s[1] * s[2])
        x, y = (v[:, o].reshape(6, s[2], s[1], s[0])[:, 3:-3, 3:-3, 3:-3].reshape(6, -1)
                for v in (first[:, bl.offsets[1]:], one))
        d = (x - y).abs().amax(1) / y.abs().amax(1)
        assert d.max() <= (1e-5 if kind == "mixed" else 1e-11), b
