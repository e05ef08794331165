"""Which basis evaluation mode a context with g functions reports and keeps:
mixed precision always runs on stored planes (0), FP64 as set."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx(gx, gpu):
    xyz = np.array([[0.0, 0.0, 0.0], [0.3, -0.2, 1.8]])
    l = [0, 1, 2, 3, 4] * 2
    bs = gx.BasisSet(l, [x > 1 for x in l], [[0.8 + 0.3 * x] for x in l], [[1.0]] * 10,
                     [r for r in xyz for _ in range(5)], normalize=True, shell_tolerance=1e-10)
    lb = gx.workloads.build_tasks(gx.Molecule([8, 1], xyz), bs, grid="GM3")
    ctx = gx.DeviceContext(0)
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(lb.get_tasks())
    ctx.upload_density(gx.workloads.density(bs.nbf(), 4, 7))
    return ctx


def test_mode_in_effect_with_g_functions(ctx):
    for mode in (3, 1, 0):
        print(f"mode {mode}", flush=True)
        ctx.set_density_basis_eval(mode)
        ctx.exc_vxc("PBE", "mixed")
        assert ctx.density_basis_eval() == 0
        ctx.exc_vxc("PBE", "fp64")
        assert ctx.density_basis_eval() == mode


def test_mixed_autotune_leaves_the_mode_of_fp64(ctx):
    for mode in (3, 1, 0):
        print(f"mixed autotuner, mode {mode}", flush=True)
        ctx.set_density_basis_eval(mode)
        ctx.autotune("PBE", "mixed")
        ctx.exc_vxc("PBE", "fp64")
        assert ctx.density_basis_eval() == mode
