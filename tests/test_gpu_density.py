"""FP64 density kernels at the edges of their tiles (16-function blocks;
64-function tiles on single point blocks, 128-function tiles on pairs of
them, the last of which may be a single one), against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", ["GM3", "FineGrid"])
@pytest.mark.parametrize("nfun", [65, 80, 127, 128, 129, 144, 193, 257])
def test_density_at_tile_edges(gx, orc, gpu, nfun, grid):
    # One atom with nfun functions, s shells but for one f shell: tiles whose
    # bounds fall inside that shell, and tiles of as many shells as functions.
    ns = nfun - 7
    l = [0] * (ns // 2) + [3] + [0] * (ns - ns // 2)
    alpha = [[0.02 * 1.02 ** k] for k in range(len(l))]
    mol = gx.Molecule([2], np.zeros((1, 3)))
    bs = gx.BasisSet(l, [x >= 2 for x in l], alpha, [[1.0]] * len(l), [np.zeros(3)] * len(l),
                     normalize=True, shell_tolerance=1e-200)
    assert bs.nbf() == nfun
    P = gx.workloads.density(nfun, 5, 3)
    t = gx.workloads.build_tasks(mol, bs, grid=grid).get_tasks()
    w = orc.ssf_weights(np.zeros((1, 3)), t)
    t["weights"] = w
    exc_o, nel_o, vxc_o = orc.exc_vxc("PBE", nfun, orc.shells_from(bs.xcq_shells()), P, t,
                                      weights=w)
    ctx = gx.DeviceContext()
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(t)
    ctx.upload_density(P)
    for wide in (1 << 30, 65):
        ctx.set_density_wide(wide)
        print(f"density edges, {nfun} functions, {grid}, wide from {wide}", flush=True)
        ctx.exc_vxc("PBE", "fp64")
        exc, nel, vxc = ctx.results()
        # Some 1e4 roundings of 1.1e-16 of the largest partial sums.
        assert abs(exc - exc_o) <= 1e-11 * abs(exc_o)
        assert abs(nel - nel_o) <= 1e-11 * abs(nel_o)
        assert np.abs(vxc - vxc_o).max() <= 1e-11 * max(1.0, np.abs(vxc_o).max())
