"""EXC nuclear gradient of rings of hydrogen atoms against the oracle: near the
centre every atom's cell function is of one size, so the weight part meets more
of them than it keeps (12) and forms the rest again; 22 atoms with three shells
each are more shells than one staging of the basis-function part holds (64),
and the six-primitive shell has more primitives than are staged (4)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRAD_BAR = 1e-9  # the gradient tests' bound


@pytest.mark.parametrize("natoms", [2, 5, 13, 14, 22])
def test_exc_grad_ring_matches_oracle(gx, orc, gpu, natoms):
    ang = 2 * np.pi * np.arange(natoms) / natoms
    xyz = np.stack([2.5 * np.cos(ang), 2.5 * np.sin(ang), 0.1 * np.cos(3 * ang + 0.3)], axis=1)
    l, pure, alpha, coeff, origin = [], [], [], [], []
    for r in xyz:
        for am, a, c in ((0, [30.0, 9.0, 3.0, 1.0, 0.35, 0.12], [0.05, 0.15, 0.3, 0.4, 0.3, 0.1]),
                         (0, [0.4], [1.0]), (1, [0.9], [1.0])):
            l.append(am)
            pure.append(False)
            alpha.append(a)
            coeff.append(c)
            origin.append(r)
    bs = gx.BasisSet(l, pure, alpha, coeff, origin, normalize=True, shell_tolerance=1e-10)
    P = gx.workloads.density(bs.nbf(), max(1, natoms // 2), 5)
    lb = gx.workloads.build_tasks(gx.Molecule([1] * natoms, xyz), bs, grid="GM3")
    t = lb.get_tasks()
    w = orc.ssf_weights(xyz, t)
    sh = orc.shells_from(bs.xcq_shells())
    t2 = dict(t)
    t2["weights"] = w
    ctx = gx.DeviceContext(0)
    ctx.upload_basis(bs.xcq_shells())
    ctx.upload_tasks(t2)
    ctx.upload_density(P)
    for func in ("SVWN5", "PBE"):
        for wd in (True, False):
            g_o = orc.exc_grad(func, bs.nbf(), sh, xyz, P, t, weights=w, weight_derivs=wd)
            bar = GRAD_BAR * max(1.0, np.abs(g_o).max())
            for lists in (True, False):
                print(f"ring of {natoms} {func} weight derivatives {wd} lists {lists}", flush=True)
                ctx.set_ssf_neighbour_lists(lists)
                ctx.exc_grad(func, xyz, weight_derivs=wd)
                g = ctx.results_grad()[2]
                err = np.abs(g - g_o).max()
                print(f"max|dG|={err:.3e} bar {bar:.1e}", flush=True)
                assert err <= bar
