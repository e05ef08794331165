"""FP64 evaluation of g functions in the stages against the stored planes:
Cartesian and spherical shells of every angular momentum, a contracted one, a
last block that is not full, and (at the size of a set knob) the kernel of
block pairs; EXC, NEL and VXC.  The knob accepts what it did, and mixed
precision with g functions stays on stored planes whatever it says."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("func", ["SVWN5", "PBE"])
@pytest.mark.parametrize("copies", [1, 3])
def test_g_functions_in_the_stages(gx, gpu, copies, func):
    xyz = np.array([[0.0, 0.0, 0.0], [0.3, -0.2, 1.8]])
    l, pure, alpha, coeff, origin = [], [], [], [], []
    for r in xyz:
        for am in range(5):
            for p in ([False] if am < 2 else [True, False]):
                for k in range(copies):
                    l.append(am)
                    pure.append(p)
                    alpha.append([1.7 / (am + 1 + k), 0.45 / (1 + k)])
                    coeff.append([0.6, 0.8])
                    origin.append(r)
    bs = gx.BasisSet(l, pure, alpha, coeff, origin, normalize=True, shell_tolerance=1e-10)
    P = gx.workloads.density(bs.nbf(), 4, 7)
    lb = gx.workloads.build_tasks(gx.Molecule([8, 1], xyz), bs, grid="GM3")
    gx.MolecularWeightsFactory("Device", "Default").get_instance().modify_weights(lb)
    ctx = gx.DeviceContext(0)
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(lb.get_tasks())
    ctx.upload_density(P)
    out = {}
    for prec in ("fp64", "mixed"):
        for mode in (0, 3):
            for wide in ((1 << 30,) if mode == 0 else (1 << 30, 65)):
                print(f"{func} {prec} mode {mode} wide {wide}", flush=True)
                ctx.set_density_basis_eval(mode)
                ctx.set_density_wide(wide)
                ctx.exc_vxc(func, prec, True)
                out[prec, mode, wide] = ctx.results()
    ref = out["fp64", 0, 1 << 30]
    for wide in (1 << 30, 65):
        exc, nel, vxc = out["fp64", 3, wide]
        # Sums of some 10^4 terms, each a few roundings of 1.1e-16.
        assert abs(exc - ref[0]) <= 1e-12 * abs(ref[0]) and abs(nel - ref[1]) <= 1e-12 * ref[1]
        assert np.abs(vxc - ref[2]).max() <= 1e-12 * max(1.0, np.abs(ref[2]).max())
        # The same launches: sums in VXC differ by the order of additions.
        a, b = out["mixed", 3, wide], out["mixed", 0, 1 << 30]
        assert a[0] == pytest.approx(b[0], rel=1e-14)
        assert np.abs(a[2] - b[2]).max() <= 1e-13 * max(1.0, np.abs(b[2]).max())
