"""GPU tests of an atom whose position is not a number: it is flagged, and until the flag is read the pair terms
of the other atoms are those without it, wherever they are and whether or not the list was due."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FLAG_NONFINITE = 4
BOX = np.array([24.0, 26.5, 21.25])
N = 343


def system(bare_atom=None):
    """A jittered lattice with an atom (N // 2) near the origin of the box; that atom's parameters zero
    where bare_atom is it."""
    rng = np.random.default_rng(3)
    m = math.ceil(N ** (1 / 3))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N]
    x = (g + 0.5) * BOX / m + rng.uniform(-0.5, 0.5, (N, 3)) - 0.5 * BOX
    q = rng.uniform(-1, 1, N)
    lj = np.tile([0.1, 2.0, 0.1, 2.0], (N, 1))
    lj[rng.random(N) < 0.5, 0::2] = 0.0
    lj[N // 2, 0::2] = 0.1
    if bare_atom is not None:
        q[bare_atom] = 0.0
        lj[bare_atom, 0::2] = 0.0
    return x, q, lj


def engine(x, q, lj, skin):
    from mdpy_amd.engine import Engine
    e = Engine.bare(N, BOX, positions=x)
    e.set_masses(np.full(N, 12.0))
    e.set_charges(q)
    e.set_lj(lj)
    e.set_exclusions(np.zeros(N + 1, int), [])
    e.set_scaling(np.zeros(N + 1, int), [])
    e.configure_nonbonded(9.0, skin=skin)
    e.configure_pme((24, 24, 24), 0.36)
    return e


@pytest.mark.parametrize("skin", [1.0, 0.0])
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("listed_before", [False, True])
def test_other_atoms_do_not_see_it(skin, value, listed_before):
    from mdpy_amd import _lib as L
    terms, k = L.TERM_LJ | L.TERM_COUL_DIRECT, N // 2
    print("case: skin %.0f, %s, list %s" % (skin, value, "kept" if listed_before else "new"), flush=True)
    x, q, lj = system()
    e = engine(x, *system(k)[1:], skin)
    want, en_want = e.compute(terms)
    want = want.cpu().numpy().copy()
    e.close()
    others = np.arange(N) != k
    bad = x.copy()
    bad[k, 1] = value
    e = engine(x if listed_before else bad, q, lj, skin)
    if listed_before:
        e.compute(terms)
        e.set_positions(bad, wrap=False)
    F, en = e.compute(terms)
    F = F.cpu().numpy().copy()
    Ff = e.compute_forces_only(terms).cpu().numpy().copy()
    assert e.status() == FLAG_NONFINITE
    scale = np.abs(want).max()
    for f in (F, Ff):
        assert np.all(np.abs(f[others] - want[others]) <= 2e-5 * scale) and np.all(f[k] == 0.0)
    for name in ("lj", "coulomb_direct"):
        assert abs(en[name] - en_want[name]) <= 1e-4 * abs(en_want[name]) + 1e-6, name
    # valid again, in place: the list has the atom back
    e.set_positions(x, wrap=False)
    F = e.compute(terms)[0].cpu().numpy().copy()
    e.set_positions(x)
    assert np.allclose(F, e.compute(terms)[0].cpu().numpy(), rtol=0, atol=2e-5 * scale) and np.any(F[k] != 0.0)
    assert e.status() == 0
    e.close()


def test_other_atoms_move_without_it():
    """Velocity-Verlet steps (the fused prologue decides the rebuild) with and without the atom's terms."""
    from mdpy_amd import _lib as L
    terms, k = L.TERM_LJ | L.TERM_COUL_DIRECT, N // 2
    print("case: integrator steps", flush=True)
    x, q, lj = system()
    got = []
    for lost in (False, True):
        e = engine(x, *(system()[1:] if lost else system(k)[1:]), 1.0)
        e.configure_integrator(L.INT_VELOCITY_VERLET, dt=0.5)
        if lost:
            e.compute(terms)  # the list is there before
            bad = x.copy()
            bad[k] = np.nan
            e.set_positions(bad, wrap=False)
        e.integrate(terms, 5, use_graph=True, energy_every=5)
        e.synchronize()
        assert e.status() == (FLAG_NONFINITE if lost else 0)
        got.append(e.positions())
        e.close()
    others = np.arange(N) != k
    moved = np.abs(got[0] - x)[others].max()
    assert np.abs(got[1] - got[0])[others].max() <= 1e-4 * moved


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("charged", [True, False])
def test_plain_coulomb(value, charged):
    """All pairs: a charged atom without a position leaves no sum with a value (nothing is added, where a
    clamped distance added the largest numbers there are), one without charge changes nothing."""
    from mdpy_amd import _lib as L
    k = N // 2
    print("case: plain Coulomb, %s, %s" % (value, "charged" if charged else "no charge"), flush=True)
    x, q, lj = system(None if charged else k)
    bad = x.copy()
    bad[k, 1] = value
    out = []
    for p in (x, bad):
        e = engine(p, q, lj, 1.0)
        F, en = e.compute(L.TERM_COUL_PLAIN)
        out.append((F.cpu().numpy().copy(), en["coulomb_plain"]))
        e.close()
    if charged:
        assert not out[1][0].any() and out[1][1] == 0.0
    else:
        assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
