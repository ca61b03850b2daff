"""GPU test of the reciprocal forces of a thin slab of atoms: the planes through it are touched by more atoms
than twice the mean, which the plane kernels keep no records for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,n,thick", [((100, 90, 96), 6000, 0.9), ((100, 90, 96), 4600, 2.5), ((60, 24, 20), 5000, 1.5),
                                          ((100, 135, 12), 6000, 0.9)])
def test_slab_against_float64(grid, n, thick):
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    from mdpy_amd.unit import ONE_OVER_4PI_EPS0
    from oracle import ewald as EW
    print("case: %d atoms in a slab of %.1f A, grid %s" % (n, thick, grid), flush=True)
    rng = np.random.default_rng(n)
    box = np.array([100.0, 90.0, 96.0])
    x = rng.uniform(-0.5, 0.5, (n, 3)) * np.array([thick, box[1], box[2]])
    x[:, 0] += 0.37 * box[0]
    q = rng.uniform(-1, 1, n)
    q[::9] = 0.0
    e = Engine.bare(n, box, positions=x)
    e.set_masses(np.ones(n))
    e.set_charges(q)
    e.set_lj(np.tile([0.0, 1.0, 0.0, 1.0], (n, 1)))
    e.set_exclusions(np.zeros(n + 1, int), [])
    e.set_scaling(np.zeros(n + 1, int), [])
    e.configure_nonbonded(3.0, skin=0.5)  # short: the list rows have room for a uniform box
    e.configure_pme(grid, 0.36)
    got = []
    for fused in (False, True):
        e.set_pme_fused(fused)
        F, en = e.compute(L.TERM_COUL_RECIP)
        got.append(F.cpu().numpy().copy())
        assert e.status() == 0
    e.close()
    Fr = EW.spme_reciprocal(x, q, box, grid, 4, 0.36, ONE_OVER_4PI_EPS0)[0]
    # float32 grid arithmetic: a few roundings per transform pass and 64 gathered points an atom
    assert np.linalg.norm(got[0] - Fr) <= 5e-6 * np.linalg.norm(Fr)
    assert np.array_equal(got[0], got[1])
