"""SSF weights of points whose parents change within a wave of 64: one, two
(taken in turn) and many (each lane's own lists), against the partition formed
in extended precision (the oracle leaves out terms of 1e-13); and a last wave
that is not full."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _weights(xyz, pts, parent, w0):
    """w0 P_parent / sum_A P_A; points near their parent keep w0."""
    f80 = np.longdouble
    x, r, a = xyz.astype(f80), pts.astype(f80), f80(0.64)
    d = np.sqrt(((r[:, None] - x[None]) ** 2).sum(axis=2))
    rab = np.sqrt(((x[:, None] - x[None]) ** 2).sum(axis=2))
    cell = np.ones_like(d)
    for A in range(len(x)):
        for B in range(len(x)):
            if A == B:
                continue
            v = np.clip((d[:, A] - d[:, B]) / (a * rab[A, B]), -1, 1)
            v2 = v * v
            cell[:, A] *= (1 - v * (35 + v2 * (-35 + v2 * (21 - 5 * v2))) / 16) / 2
    near = (rab + np.diag(np.full(len(x), f80(np.inf)))).min(axis=1)
    k = np.arange(len(r))
    keep = d[k, parent] < 0.5 * (1 - a) * near[parent]
    return np.where(keep, w0, w0 * cell[k, parent] / cell.sum(axis=1))


@pytest.mark.parametrize("run", [1000, 64, 40, 21, 1])
@pytest.mark.parametrize("nw", [1, 9])
def test_weights_with_mixed_parents(gx, gpu, nw, run):
    from gauxc_amd import _native
    lib = _native.device_lib()
    Z, xyz = gx.workloads.water_cluster(nw, 2.8 * nw ** (1 / 3), 3)
    xyz = np.ascontiguousarray(xyz, dtype=np.float64)
    rng = np.random.default_rng(run)
    n = 4099
    parent = ((np.arange(n) // run) % len(Z)).astype(np.int32)
    pts = np.ascontiguousarray(xyz[parent] + rng.normal(size=(n, 3)) * rng.choice([0.5, 2.0, 5.0],
                                                                                  size=(n, 1)))
    w0 = rng.uniform(0.5, 1.5, size=n)
    ref = _weights(xyz, pts, parent, w0)
    w = w0.copy()
    print(f"{nw} waters, runs of {run}", flush=True)
    assert lib.xcq_ssf_weights(0, len(Z), xyz.ctypes.data, n, pts.ctypes.data, parent.ctypes.data,
                               w.ctypes.data) == 0, lib.xcq_last_error()
    # Products of up to 26 factors and a sum, each a few roundings of the
    # switching polynomial (of size 1 - v: absolute, not relative).
    assert np.abs(w - ref).max() <= 1e-13
