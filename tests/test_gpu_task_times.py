"""Task times come from the lists the last evaluation ran, whatever the
settings were or have become: tasks on pairs of point blocks have a density
time after evaluations in the stages, those on single blocks after one on
stored planes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_times_follow_the_evaluation(gx, gpu):
    mol, bs, P, cfg = gx.workloads.make_config("c1", seed=2, n_water=4)
    lb = gx.workloads.build_tasks(mol, bs, grid="GM3")
    t = lb.get_tasks()
    pairs = (t["nbe"] >= 65) & (t["npts"] > 64)
    assert pairs.any()
    ctx = gx.DeviceContext(0)
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(t)
    ctx.upload_density(P)
    ctx.upload_density_z(0.1 * P)
    ctx.set_density_wide(65)

    def times(what, run, after=None):
        print(what, flush=True)
        ctx.enable_task_timing(True)  # all stamps zero
        run()
        if after is not None:
            ctx.set_density_basis_eval(after)
        d, _ = ctx.task_times()
        assert np.all(d > 0), what

    times("in the stages", lambda: ctx.exc_vxc("PBE", "fp64"))
    times("in the stages, then set to stored planes", lambda: ctx.exc_vxc("PBE", "fp64"), 0)
    times("stored planes", lambda: ctx.exc_vxc("PBE", "fp64"))
    times("UKS, set to stored planes", lambda: ctx.exc_vxc_uks("PBE"))
    times("gradient, set to stored planes", lambda: ctx.exc_grad("PBE", cfg["xyz"]))
    times("stored planes, then set to the stages", lambda: ctx.exc_vxc("PBE", "fp64"), 3)
    times("mixed", lambda: ctx.exc_vxc("PBE", "mixed"))
