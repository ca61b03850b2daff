"""GPU tests of the pair kernel's two kinds of waves (atoms with and without LJ parameters) and of
its box-fraction positions, against a float64 double loop."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def loop(x, box, q, lj, rc, beta, ke):
    """Forces, energies and per-component sums of |pair force| of LJ and erfc Coulomb."""
    from scipy.special import erfc
    n = len(x)
    F, size, e = np.zeros((n, 3)), np.zeros((n, 3)), [0.0, 0.0]
    for i in range(n):
        d = np.delete(x, i, 0) - x[i]
        d -= box * np.round(d / box)
        r = np.sqrt((d * d).sum(1))
        m = r <= rc
        a, b = lj[i], np.delete(lj, i, 0)[m]
        d, r, qq = d[m], r[m], ke * q[i] * np.delete(q, i)[m]
        eps, s6 = np.sqrt(a[0] * b[:, 0]), (0.5 * (a[1] + b[:, 1]) / r) ** 6
        ec, ex = erfc(beta * r), np.exp(-(beta * r) ** 2)
        flj = 24 * eps * (2 * s6 * s6 - s6) / r ** 2
        fc = qq * (ec / r + 2 * beta / math.sqrt(math.pi) * ex) / r ** 2
        F[i] = -((flj + fc)[:, None] * d).sum(0)
        # sizes of the pieces that float32 rounds: s^12, s^6 and, in the tabulated form, 1/r^3
        size[i] = ((24 * eps * (2 * s6 * s6 + s6) / r ** 2 + np.abs(qq) / r ** 3)[:, None] * np.abs(d)).sum(0)
        e[0] += 0.5 * (4 * eps * (s6 * s6 - s6)).sum()
        e[1] += 0.5 * (qq * ec / r).sum()
    return F, size, e


@pytest.mark.parametrize("n,bare", [(2, 0.5), (5, 1.0), (65, 0.0), (130, 0.5), (700, 0.67)])
def test_mixed_lj_kinds_against_float64(n, bare):
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    from mdpy_amd.unit import KCAL_PER_MOL, ONE_OVER_4PI_EPS0
    print("case: %d atoms, %.0f %% without LJ" % (n, 100 * bare), flush=True)
    rng = np.random.default_rng(n)
    box = np.array([24.0, 26.5, 21.25])
    m = math.ceil(n ** (1 / 3))  # jittered lattice: no pair closer than 1.2 A
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g + 0.5) * box / m + rng.uniform(-0.5, 0.5, (n, 3)) - 0.5 * box
    q = rng.uniform(-1, 1, n)
    lj = np.stack([rng.uniform(0.05, 0.2, n) * KCAL_PER_MOL, rng.uniform(1.5, 2.5, n)] * 2, 1)
    lj[rng.random(n) < bare, 0::2] = 0.0
    got = []
    for shift in (0, 1):
        e = Engine.bare(n, box, positions=x + shift * box * rng.integers(-1, 2, (n, 3)))
        e.set_masses(np.ones(n))
        e.set_charges(q)
        e.set_lj(lj)
        e.set_exclusions(np.zeros(n + 1, int), [])
        e.set_scaling(np.zeros(n + 1, int), [])
        e.configure_nonbonded(9.0, skin=1.0)
        e.configure_pme((24, 24, 24), 0.36)
        F, en = e.compute(L.TERM_LJ | L.TERM_COUL_DIRECT)
        got.append((F.cpu().numpy().copy(), e.compute_forces_only(L.TERM_LJ | L.TERM_COUL_DIRECT).cpu().numpy().copy(), en))
        e.close()
    F, size, en = loop(x, box, q, lj, 9.0, 0.36, ONE_OVER_4PI_EPS0)
    for k in (0, 1):  # evaluation with energies, forces only
        # ~12 float32 roundings per pair term (r^-14 amplifies the distance's), partial sums of the row
        assert np.all(np.abs(got[0][k] - F) <= 2.0 ** -40 + 40 * 2.0 ** -24 * size + 1e-6 * np.abs(F).max())
        # whole box edges change a coordinate's box fraction by its last bit at most
        assert np.all(np.abs(got[1][k] - got[0][k]) <= 2.0 ** -39 + 8 * 2.0 ** -24 * size)
    assert abs(got[0][2]["lj"] - en[0]) <= 1e-5 * abs(en[0]) + 1e-9
    assert abs(got[0][2]["coulomb_direct"] - en[1]) <= 1e-5 * np.abs(size).max() + 1e-9


@pytest.mark.parametrize("grid", [(4, 5, 6), (25, 24, 27), (20, 64, 45), (16, 128, 125), (100, 9, 128), (32, 135, 12),
                                  (30, 40, 150)])
def test_pme_grids_against_float64(grid):
    """Reciprocal forces and energy of odd, even, uneven and large grids (the plane kernels hold up
    to 128 x 128 points; larger planes take the global-grid path) against the float64 oracle."""
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    from mdpy_amd.unit import ONE_OVER_4PI_EPS0
    from oracle import ewald as EW
    print("case: PME grid", grid, flush=True)
    rng = np.random.default_rng(sum(grid))
    n, box = 150, np.array([24.0, 26.5, 21.25])
    x = rng.uniform(-0.5, 0.5, (n, 3)) * box
    q = rng.uniform(-1, 1, n)
    q[::7] = 0.0
    e = Engine.bare(n, box, positions=x)
    e.set_masses(np.ones(n))
    e.set_charges(q)
    e.set_lj(np.tile([0.0, 1.0, 0.0, 1.0], (n, 1)))
    e.set_exclusions(np.zeros(n + 1, int), [])
    e.set_scaling(np.zeros(n + 1, int), [])
    e.configure_nonbonded(9.0, skin=1.0)
    e.configure_pme(grid, 0.36)
    F, en = e.compute(L.TERM_COUL_RECIP)
    F = F.cpu().numpy()
    assert e.status() == 0
    e.close()
    ref = EW.spme_reciprocal(x, q, box, grid, 4, 0.36, ONE_OVER_4PI_EPS0)
    Fr, Er = ref[0], ref[1]
    # float32 grid arithmetic: a few roundings per transform pass and 64 gathered points an atom
    assert np.linalg.norm(F - Fr) <= 5e-6 * np.linalg.norm(Fr)
    self_e = -ONE_OVER_4PI_EPS0 * 0.36 / math.sqrt(math.pi) * (q * q).sum()
    back = -ONE_OVER_4PI_EPS0 * math.pi * q.sum() ** 2 / (2 * 0.36 ** 2 * box.prod())
    assert abs(en["coulomb_reciprocal"] - (Er + self_e + back)) <= 1e-5 * (abs(Er) + abs(self_e))


@pytest.mark.parametrize("n", [24576, 24577, 24700])
def test_resident_workgroups_by_size(n):
    """Both sides of the default's limit (at 16 lanes 1,536 units of work on 256 compute units) give
    the bits of every explicit choice: forces are exact integer sums, in any order."""
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    print("case: %d atoms" % n, flush=True)
    rng = np.random.default_rng(n)
    box, m = np.array([93.0, 96.0, 99.0]), 30
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    e = Engine.bare(n, box, positions=(g + 0.5) * box / m + rng.uniform(-0.4, 0.4, (n, 3)) - 0.5 * box)
    e.set_masses(np.ones(n))
    e.set_charges(rng.uniform(-1, 1, n))
    e.set_lj(np.tile([0.1, 2.0, 0.1, 2.0], (n, 1)))
    e.set_exclusions(np.zeros(n + 1, int), [])
    e.set_scaling(np.zeros(n + 1, int), [])
    e.configure_nonbonded(9.0, skin=1.0)
    e.configure_pme((24, 24, 24), 0.36)
    F = e.compute_forces_only(L.TERM_LJ | L.TERM_COUL_DIRECT).cpu().numpy().copy()
    assert e.status() == 0 and np.abs(F).max() > 0
    for per_cu in (0, 2, 3):
        e.set_nonbonded_persist(per_cu)
        assert np.array_equal(F, e.compute_forces_only(L.TERM_LJ | L.TERM_COUL_DIRECT).cpu().numpy()), per_cu
    e.close()
