"""GPU tests of the float32 to fixed-point conversion that pair forces, charge spreading and the
surrogate's partner forces go through: to 2^-40 for both signs, at every magnitude."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bare(n, box, x, q, lj):
    from mdpy_amd.engine import Engine
    e = Engine.bare(n, box, positions=x)
    e.set_masses(np.ones(n))
    e.set_charges(q)
    e.set_lj(lj)
    e.set_exclusions(np.zeros(n + 1, int), [])
    e.set_scaling(np.zeros(n + 1, int), [])
    e.configure_nonbonded(9.0, skin=1.0)
    return e


@pytest.mark.parametrize("lo,hi", [(-12, -8), (-8, -4), (-4, 0), (0, 4)])
def test_pair_forces_of_both_signs(lo, hi):
    """Isolated LJ pairs whose forces span 10^lo to 10^hi: the two atoms' forces are opposite to the last
    bit and within the float32 arithmetic of the float64 value."""
    from mdpy_amd import _lib as L
    print("case: pair forces 1e%d .. 1e%d" % (lo, hi), flush=True)
    rng = np.random.default_rng(20 + lo)
    m, a = 8, 25.0
    box = np.full(3, m * a)
    site = (np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * a - 0.5 * box
    P = len(site)
    d = rng.standard_normal((P, 3))
    d *= (rng.uniform(2.5, 8.0, P) / np.linalg.norm(d, axis=1))[:, None]
    x = np.empty((2 * P, 3))
    x[0::2], x[1::2] = site - 0.5 * d, site + 0.5 * d
    r, sigma = np.linalg.norm(d, axis=1), 2.0
    s6 = (sigma / r) ** 6
    per_eps = 24 * (2 * s6 * s6 - s6) / r  # force along d for eps = 1
    eps = 10.0 ** rng.uniform(lo, hi, P) / np.abs(per_eps)
    lj = np.zeros((2 * P, 4))
    lj[:, 0] = lj[:, 2] = np.repeat(eps, 2)
    lj[:, 1] = lj[:, 3] = sigma
    e = bare(2 * P, box, x, np.zeros(2 * P), lj)
    F = e.compute_forces_only(L.TERM_LJ).cpu().numpy()
    assert e.status() == 0
    e.close()
    assert np.array_equal(F[0::2], -F[1::2])
    want = -(eps * per_eps / r)[:, None] * d
    # the pair's float32 terms (s^12 and s^6 cancel); the box fractions, which hold a coordinate to 2^-32
    # of the edge (r^-14 amplifies the distance's error); one rounding to 2^-40
    size = (eps * 24 * (2 * s6 * s6 + s6) / r ** 2)[:, None]
    bound = 0.5 * 2.0 ** -40 + size * (40 * 2.0 ** -24 * np.abs(d) + 2.0 ** -32 * box[0] * (1 + 14 * np.abs(d) / r[:, None]))
    assert np.all(np.abs(F[0::2] - want) <= bound)


def test_spread_charges_of_both_signs():
    """All charges negated: the same reciprocal forces and energy, to the last bit."""
    from mdpy_amd import _lib as L
    print("case: reciprocal forces of q and -q", flush=True)
    rng = np.random.default_rng(5)
    n, box = 300, np.array([24.0, 26.5, 21.25])
    x = rng.uniform(-0.5, 0.5, (n, 3)) * box
    q = 10.0 ** rng.uniform(-8, 0, n) * rng.choice([-1.0, 1.0], n)
    for grid in ((24, 27, 20), (20, 135, 12)):  # plane kernels, global grid
        out = []
        for sign in (1, -1):
            e = bare(n, box, x, sign * q, np.tile([0.0, 1.0, 0.0, 1.0], (n, 1)))
            e.configure_pme(grid, 0.36)
            F, en = e.compute(L.TERM_COUL_RECIP)
            out.append((F.cpu().numpy().copy(), en["coulomb_reciprocal"]))
            assert e.status() == 0
            e.close()
        assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1], grid
