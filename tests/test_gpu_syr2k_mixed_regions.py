"""Mixed-precision B^T Z contraction at the sizes where its division into
regions changes: a task of up to 7 blocks of 16 functions (112) is one region,
one of 8 (113 to 128) two row and two column groups, one of 11 (161 to 176)
three column groups, one of 13 (193) three row groups.  Against the FP64 path;
one task of 3,850 points in several slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfun", [113, 128, 160, 176, 192, 193])
def test_mixed_vxc_where_regions_divide(gx, gpu, nfun):
    bs = gx.BasisSet([0] * nfun, [False] * nfun, [[0.02 * 1.02 ** k] for k in range(nfun)],
                     [[1.0]] * nfun, [np.zeros(3)] * nfun, normalize=True,
                     shell_tolerance=1e-200)
    lb = gx.workloads.build_tasks(gx.Molecule([2], np.zeros((1, 3))), bs, grid="GM3")
    gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
    t = lb.get_tasks()
    assert t["nbe"].max() == nfun and t["npts"].max() > 1024
    ctx = gx.DeviceContext(0)
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(t)
    ctx.upload_density(gx.workloads.density(nfun, 5, 3))
    print(f"mixed regions, {nfun} functions", flush=True)
    vxc = {}
    for prec in ("fp64", "mixed"):
        ctx.exc_vxc("PBE", prec, True)
        vxc[prec] = ctx.results()[2]
    # FP32 roundings (2^-24) of P, B, X and Z in each element's terms.
    bar = 4 * 2.0**-24 * max(1.0, np.abs(vxc["fp64"]).max())
    assert np.abs(vxc["mixed"] - vxc["fp64"]).max() <= bar
