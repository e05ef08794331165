"""Mixed-precision B^T Z contraction at the edges of its regions (16-function
blocks in row pairs; a task of up to 96 functions is one region, larger ones
are divided into up to three row pairs and five columns) and with a task of
many points cut into slices, against the FP64 path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfun", [1, 16, 17, 32, 33, 96, 97, 112, 144, 161, 209, 337])
def test_mixed_vxc_at_region_edges(gx, gpu, nfun):
    # One atom with nfun s functions: one task of 3,850 points (several
    # slices), or a few at the largest nfun.
    mol = gx.Molecule([2], np.zeros((1, 3)))
    alpha = [[0.02 * 1.02 ** k] for k in range(nfun)]
    bs = gx.BasisSet([0] * nfun, [False] * nfun, alpha, [[1.0]] * nfun, [np.zeros(3)] * nfun,
                     normalize=True, shell_tolerance=1e-200)
    P = gx.workloads.density(nfun, min(nfun, 5), 3)
    lb = gx.workloads.build_tasks(mol, bs, grid="GM3")
    t = lb.get_tasks()
    assert t["nbe"].max() == nfun and t["npts"].max() > 1024
    gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
    ctx = gx.DeviceContext(0)
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(lb.get_tasks())
    ctx.upload_density(P)
    print(f"mixed region edges, {nfun} functions", flush=True)
    ctx.exc_vxc("PBE", "fp64", True)
    v64 = ctx.results()[2]
    ctx.exc_vxc("PBE", "mixed", True)
    vmx = ctx.results()[2]
    # FP32 roundings (2^-24) of P, B, X and Z in each element's terms.
    err = np.abs(vmx - v64)
    bar = 4 * 2.0**-24 * max(1.0, np.abs(v64).max())
    if err.max() > bar:
        for i in range(0, nfun, 16):
            print(" ".join("%.0e" % err[i:i + 16, j:j + 16].max() for j in range(0, nfun, 16)))
    print(f"max|dVXC|={err.max():.2e} bar {bar:.1e}", flush=True)
    assert err.max() <= bar
