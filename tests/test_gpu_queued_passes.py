"""Evaluations that launch one work list several times (the density stage per
matrix, B^T Z per spin component) under persistent queues, against one
workgroup per item; on single point blocks and on pairs of them.  Another
density goes through the same buffers first, so that a pass that does nothing
leaves wrong values behind."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def system(gx, gpu):
    mol, bs, _, cfg = gx.workloads.make_config("c1", seed=2, n_water=4)
    lb = gx.workloads.build_tasks(mol, bs, grid="GM3")
    gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
    t = lb.get_tasks()
    assert t["nbe"].max() > 128 and t["npts"].max() > 128
    n = bs.nbf()
    rng = np.random.default_rng(4)
    C, _ = np.linalg.qr(rng.normal(size=(n, 20)))
    U = rng.normal(size=(2, n, n)) / n
    mats = [C @ C.T + C[:, :17] @ C[:, :17].T, C[:, 17:] @ C[:, 17:].T,
            U[0] + U[0].T, 0.3 * (U[1] + U[1].T)]
    return bs, t, cfg["xyz"], mats


def _evaluate(ctx, what, func, xyz, mats):
    Ps, Pz, tPs, tPz = mats
    ctx.upload_density(Ps)
    if what in ("uks", "fxc_uks", "grad_uks"):
        ctx.upload_density_z(Pz)
    if what in ("fxc", "fxc_uks"):
        ctx.upload_trial_density(tPs)
    if what == "fxc_uks":
        ctx.upload_trial_density_z(tPz)
    if what == "rks":
        ctx.exc_vxc(func, "fp64", True)
        return ctx.results()
    if what == "uks":
        ctx.exc_vxc_uks(func)
        return ctx.results_uks()
    if what == "fxc":
        ctx.fxc_contraction(func)
        return ctx.results_fxc()
    if what == "fxc_uks":
        ctx.fxc_contraction_uks(func)
        return ctx.results_fxc_uks()
    ctx.exc_grad(func, xyz, uks=what == "grad_uks")
    return ctx.results_grad()


@pytest.mark.parametrize("func", ["PBE", "SVWN5"])
@pytest.mark.parametrize("what", ["rks", "uks", "fxc", "fxc_uks", "grad", "grad_uks"])
def test_queued_passes_match_direct(gx, system, what, func):
    bs, t, xyz, mats = system
    other = [0.5 * m for m in mats]
    ref = None
    for arena in (0, 48 << 20):  # one chunk, and several
        ctx = gx.DeviceContext(0, arena)
        ctx.upload_basis(bs.xcq_shells())
        ctx.upload_tasks(t)
        for wide in (1 << 30, 65):
            ctx.set_density_wide(wide)
            direct = None
            for nq in (0, 300, 7):
                print(f"{what} {func} arena {arena} pairs from {wide} queues {nq}", flush=True)
                ctx.set_schedule(0)
                _evaluate(ctx, what, func, xyz, other)
                ctx.set_schedule(nq)
                out = _evaluate(ctx, what, func, xyz, mats)
                if direct is None:
                    direct = out
                if ref is None:
                    ref = out
                for a, b, r in zip(out, direct, ref):
                    # Sums of up to 1e5 terms in another order, each a rounding
                    # of 1.1e-16, with a factor of ten for the functional's
                    # derivatives where densities cancel.
                    bar = 1e-10 * max(1.0, np.abs(r).max())
                    assert np.abs(np.asarray(a) - r).max() <= bar
                    if np.ndim(a) == 0:  # the blocks' sums are added in order
                        assert a == b
