"""The per-block entries (sgr_rhs_block, sgr_bssnrhs_host): every host thread
keeps one plan and reuses it for the next block of the same size, so what one
call leaves behind must not reach the next one's result.  Against the CPU
oracle at the FP64 bar, 1e-12 normwise per field."""
import threading

import numpy as np
import pytest

from helpers import interior, normwise

pytestmark = pytest.mark.gpu


def _block(n, seed):
    from sympygr_amd import data
    pmin = (-0.7, -0.4, -0.9)
    pmax = tuple(p + h * (n + 5) for p, h in zip(pmin, (0.07, 0.06, 0.08)))
    return data.perturbed_flat_block(seed=seed, n=n + 6, amp=1e-2, pmin=pmin, pmax=pmax), (n + 6,) * 3, pmin, pmax


def _in_new_thread(fn):
    """fn() in a thread of its own, which starts without a plan."""
    failed = []

    def run():
        try:
            fn()
        except BaseException as e:  # noqa: BLE001 - handed to the test
            failed.append(e)
    t = threading.Thread(target=run)
    t.start()
    t.join()
    if failed:
        raise failed[0]


@pytest.mark.parametrize("host", [False, True])
@pytest.mark.parametrize("n,gib", [(7, None), (16, None), (16, "0.001")])
def test_gauge_changes_between_blocks_of_one_size(n, gib, host, monkeypatch):
    """Rochester, standard, Rochester, standard: the two gauges run other
    kernels over other tile lists (and, at 7 points, other tiles); with a
    workspace of a few tiles, in several launches."""
    import pyoracle as po
    import torch
    import sympygr_amd as sgr
    if gib:
        monkeypatch.setenv("SGR_WS_GIB", gib)

    def calls():
        for k, gauge in enumerate(("rochester", "standard", "rochester", "standard")):
            u, sz, pmin, pmax = _block(n, 20 + k)
            kw = dict(gauge=gauge, xi=(1, 1, 1), ko_sigma=0.1)
            prm = sgr.params(adv="upwind", **kw)
            if host:
                got = np.full_like(u, 5.0)
                sgr.bssnrhs(got, u, 0, pmin, pmax, sz, 63, prm)
            else:
                du = torch.from_numpy(u).cuda()
                out = torch.full_like(du, 5.0)
                torch.cuda.synchronize()
                sgr.rhs_block(out, du, 0, pmin, pmax, sz, 63, prm)
                got = out.cpu().numpy()
            ref = po.rhs_block(u, sz, pmin, pmax, 63, po.make_params(upwind=True, **kw))
            assert normwise(interior(got, sz), interior(ref, sz)).max() <= 1e-12, (k, gauge)
    _in_new_thread(calls)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("diss", ["tvb3", "tvb5"])
def test_tvb_blocks_at_growing_offsets(diss, precision):
    """Equal-sized blocks one after another out of one set of arrays, as a
    block loop calls them: each reads the characteristic speeds of its own
    nodes, so all equal the plan over the whole set bit for bit."""
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.uniform_tiling(nb=2, n=16, lo=-1.0, hi=1.0, stagger=0.5, faces=True)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="perturbed", seed=8, amp=1e-2, lo=-1.0, L=2.0)
    prm = sgr.params(adv="upwind", ko_sigma=0.1, dissipation=diss, precision=precision)
    out, ref = torch.full_like(u, 5.0), torch.full_like(u, 5.0)
    sgr.Plan(bl, prm).rhs(ref, u)
    torch.cuda.synchronize()

    def calls():
        for b in range(len(bl)):
            sgr.rhs_block(out, u, bl.offsets[b], bl.pmin[b], bl.pmax[b], bl.sz[b], bl.bflag[b], prm)
    _in_new_thread(calls)
    assert torch.equal(out, ref)


def test_ccz4_block_takes_25_fields():
    """A CCZ4 block has a 25th array: 24 are refused before the library would
    read a pointer that is not there."""
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    bl = data.BlockList()
    bl.add((22, 22, 22), (-1.05,) * 3, (1.05,) * 3, 63)
    u = data.fill_blocks(bl, backend="torch", device="cuda", kind="ccz4", seed=4, amp=1e-2, lo=-1.05, L=2.1)
    prm = sgr.params(adv="upwind", formulation="ccz4")
    ref, got = torch.full_like(u, 5.0), torch.full_like(u, 5.0)
    sgr.Plan(bl, prm).rhs(ref, u)
    torch.cuda.synchronize()
    sgr.rhs_block(got, u, 0, bl.pmin[0], bl.pmax[0], bl.sz[0], 63, prm)
    assert torch.equal(got, ref)
    with pytest.raises(ValueError, match="25"):
        sgr.rhs_block(got[:24], u[:24], 0, bl.pmin[0], bl.pmax[0], bl.sz[0], 63, prm)
