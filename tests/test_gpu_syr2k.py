"""FP64 B^T Z contraction at the edges of its regions (16-function blocks; a
task of up to 128 functions is one region, larger ones are divided) and with
a task of many points cut into slices, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfun", [1, 16, 17, 112, 128, 129, 145, 208, 209, 337])
def test_vxc_at_region_edges(gx, orc, gpu, nfun):
    # One atom with nfun s functions: one task of 3,850 points (several
    # slices), or a few at the largest nfun, whose tightest functions do not
    # reach every point.
    mol = gx.Molecule([2], np.zeros((1, 3)))
    alpha = [[0.02 * 1.02 ** k] for k in range(nfun)]
    bs = gx.BasisSet([0] * nfun, [False] * nfun, alpha, [[1.0]] * nfun, [np.zeros(3)] * nfun,
                     normalize=True, shell_tolerance=1e-200)
    P = gx.workloads.density(nfun, min(nfun, 5), 3)
    lb = gx.workloads.build_tasks(mol, bs, grid="GM3")
    t = lb.get_tasks()
    assert t["nbe"].max() == nfun and t["npts"].max() > 1024
    w = orc.ssf_weights(np.zeros((1, 3)), t)
    exc_o, _, vxc_o = orc.exc_vxc("PBE", nfun, orc.shells_from(bs.xcq_shells()), P, t, weights=w)
    gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
    integ = gx.XCIntegratorFactory("Device", "Replicated").get_instance(gx.Functional("PBE"), lb)
    print(f"region edges, {nfun} functions", flush=True)
    exc, vxc = integ.eval_exc_vxc(P)
    # Sums of 3,850 terms of one sign pattern: a few thousand roundings of
    # 1.1e-16 of the largest partial sum.
    assert abs(exc - exc_o) <= 1e-11 * abs(exc_o)
    assert np.abs(vxc - vxc_o).max() <= 1e-11 * max(1.0, np.abs(vxc_o).max())
    # One task's sums do not depend on the order its parts finish in.
    exc2, vxc2 = integ.eval_exc_vxc(P)
    assert exc2 == exc and (len(t["npts"]) > 1 or np.array_equal(vxc2, vxc))
