"""GPU test of the reciprocal forces' rounding error where long waves are large: water boxes whose lattice has
vacancies on one side, against the float64 oracle."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,cutoff,grid", [(1200, 12.0, 36), (1200, 9.0, 36), (2400, 12.0, 45), (2400, 12.0, 48)])
def test_long_waves_against_float64(waters, cutoff, grid):
    from mdpy_amd import _lib as L, systems
    from mdpy_amd.engine import Engine
    from mdpy_amd.unit import ONE_OVER_4PI_EPS0
    from oracle import ewald as EW
    print("case: %d waters, r_c %.0f A, grid %d" % (waters, cutoff, grid), flush=True)
    m = math.ceil(waters ** (1 / 3))
    edge = (waters / 0.0334) ** (1 / 3)
    s = systems.water_box(m, edge / m, n_waters=waters, seed=waters, cutoff=cutoff, pme_grid=(grid,) * 3)
    e = Engine(s)
    e.set_positions(s.positions)
    x = e.positions()
    F = e.compute(L.TERM_COUL_RECIP)[0].cpu().numpy()
    ex = np.asarray(EW.spme_reciprocal(x, s.charges, s.box, s.pme_grid, 4, e.beta, ONE_OVER_4PI_EPS0)[0])
    e.close()
    # exclusion corrections come with the term; they act within a molecule and leave its sum
    mol = lambda a: a.reshape(waters, 3, 3).sum(1)
    err = np.linalg.norm(mol(F) - mol(ex), axis=0) / np.linalg.norm(mol(ex))
    print("  relative error by axis", err, flush=True)
    # some 50 float32 roundings (12 transform passes, spread, gather, the long waves being the larger part of
    # the potential); pairs of rows along y share a transform, which must not show in the y component:
    # with the imaginary rounding of real coefficients it was 3 to 5 times the x component's
    assert np.all(err <= 50 * 2.0 ** -24) and err[1] <= 1.5 * err[0], err


def test_reciprocal_energy_against_float64():
    """The spread conserves charge (an error in a spread charge's sum is a long wave, to which the energy is
    most sensitive): root mean square error over boxes whose lattice has vacancies."""
    from mdpy_amd import _lib as L, systems
    from mdpy_amd.engine import Engine, beta_from_tolerance
    from mdpy_amd.unit import ONE_OVER_4PI_EPS0
    from oracle import ewald as EW
    waters, grid, err, size = 2000, (40, 40, 40), [], []
    edge = (waters / 0.0334) ** (1 / 3)
    beta = beta_from_tolerance(12.0, 1e-5)
    for seed in range(4):
        s = systems.water_box(13, edge / 13, n_waters=waters, seed=seed, cutoff=12.0, pme_grid=grid)
        n, q = s.num_atoms, np.asarray(s.charges)
        e = Engine.bare(n, s.box, positions=s.positions)
        e.set_masses(s.masses)
        e.set_charges(q)
        e.set_lj(s.lj)
        e.set_exclusions(np.zeros(n + 1, int), [])
        e.set_scaling(np.zeros(n + 1, int), [])
        e.configure_nonbonded(9.0, skin=1.0)
        e.configure_pme(grid, beta)
        got = e.compute(L.TERM_COUL_RECIP)[1]["coulomb_reciprocal"]
        e.close()
        Er = EW.spme_reciprocal(s.positions, q, s.box, grid, 4, beta, ONE_OVER_4PI_EPS0)[1]
        self_e = -ONE_OVER_4PI_EPS0 * beta / math.sqrt(math.pi) * (q * q).sum()
        err.append(got - (Er + self_e))
        size.append(Er)
    rel = math.sqrt(np.mean(np.square(err)) / np.mean(np.square(size)))
    print("case: energy of 2,000 waters, relative error %.2e" % rel, flush=True)
    # the energy is quadratic in the spread charges, whose float32 roundings (2^-24) otherwise average out
    # over the atoms; weights whose sum is off by their own roundings gave 2.6e-7
    assert rel <= 2 * 2.0 ** -24


@pytest.mark.parametrize("grid", [(1080, 4, 5), (1152, 6, 5), (1600, 5, 4), (2187, 4, 4)])
def test_grids_elongated_along_x(grid):
    """Lines so long that a workgroup of the x-axis pass holds fewer of them."""
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    from mdpy_amd.unit import ONE_OVER_4PI_EPS0
    from oracle import ewald as EW
    print("case: PME grid", grid, flush=True)
    rng = np.random.default_rng(grid[0])
    n, box = 60, np.array([24.0, 26.5, 21.25])
    x = rng.uniform(-0.5, 0.5, (n, 3)) * box
    q = rng.uniform(-1, 1, n)
    e = Engine.bare(n, box, positions=x)
    e.set_masses(np.ones(n))
    e.set_charges(q)
    e.set_lj(np.tile([0.0, 1.0, 0.0, 1.0], (n, 1)))
    e.set_exclusions(np.zeros(n + 1, int), [])
    e.set_scaling(np.zeros(n + 1, int), [])
    e.configure_nonbonded(9.0, skin=1.0)
    e.configure_pme(grid, 0.36)
    F = e.compute(L.TERM_COUL_RECIP)[0].cpu().numpy()
    assert e.status() == 0
    e.close()
    Fr = EW.spme_reciprocal(x, q, box, grid, 4, 0.36, ONE_OVER_4PI_EPS0)[0]
    # float32 roundings of up to 7 passes each way, on a derivative along x of K_x/L_x points per A
    assert np.linalg.norm(F - Fr) <= 2.0 ** -24 * 50 * max(1.0, 0.02 * grid[0]) * np.linalg.norm(Fr)
