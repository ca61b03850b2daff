"""GPU test of a context that is bound to another number of atoms: parameters, exclusions and terms of the old
system are gone (their arrays are too short for the new one), and the new ones give a fresh context's bits."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOX = np.array([24.0, 26.5, 21.25])


def system(n, seed):
    rng = np.random.default_rng(seed)
    m = 7
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g + 0.5) * BOX / m + rng.uniform(-0.5, 0.5, (n, 3)) - 0.5 * BOX
    return x, rng.uniform(-1, 1, n), np.tile([0.1, 2.0, 0.1, 2.0], (n, 1))


def partners(n):
    """Every atom excludes the next one, CSR."""
    rows = [[j for j in (i - 1, i + 1) if 0 <= j < n] for i in range(n)]
    return np.concatenate([[0], np.cumsum([len(r) for r in rows])]), [j for r in rows for j in r]


def parameters(e, n, q, lj, excluded):
    e.set_masses(np.ones(n))
    e.set_charges(q)
    e.set_lj(lj)
    if excluded:
        e.set_exclusions(*partners(n))
        e.set_scaling(np.zeros(n + 1, int), [])
        e.set_bonds(np.stack([np.arange(n - 1), np.arange(1, n)], 1), np.tile([1.0, 2.0], (n - 1, 1)))


@pytest.mark.parametrize("n,other", [(100, 343), (343, 100)])
@pytest.mark.parametrize("excluded", [False, True])
def test_another_number_of_atoms(n, other, excluded):
    import torch
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    print("case: %d atoms, then %d, %s exclusions" % (n, other, "new" if excluded else "no"), flush=True)
    terms = L.TERM_LJ | L.TERM_COUL_DIRECT | L.TERM_BOND
    x, q, lj = system(n, 1)
    e = Engine.bare(n, BOX, positions=x)
    parameters(e, n, q, lj, True)
    e.configure_nonbonded(9.0, skin=1.0)
    e.configure_pme((24, 24, 24), 0.36)
    e.configure_integrator(L.INT_VELOCITY_VERLET, dt=0.5)
    e.compute(terms)
    x, q, lj = system(other, 2)
    e.n = other
    e.pos = torch.tensor(x, device=e.device)
    e.vel = torch.zeros_like(e.pos)
    e.force_buf = torch.zeros_like(e.pos)
    L.call("mdx_system_set", e.ctx, other, ctypes.c_void_p(e.pos.data_ptr()), ctypes.c_void_p(e.vel.data_ptr()),
           (ctypes.c_double * 3)(*BOX))
    e.configure_nonbonded(9.0, skin=1.0)
    e.configure_pme((24, 24, 24), 0.36)
    for term, what in ((L.TERM_LJ, "LJ"), (L.TERM_COUL_DIRECT, "charges|PME"), (L.TERM_COUL_PLAIN, "charges")):
        with pytest.raises(Exception, match=what):
            e.compute(term)
    with pytest.raises(Exception, match="not configured"):
        e.integrate(terms, 1)
    fresh = Engine.bare(other, BOX, positions=x)
    out = []
    for c in (e, fresh):
        parameters(c, other, q, lj, excluded)
        c.configure_nonbonded(9.0, skin=1.0)
        c.configure_pme((24, 24, 24), 0.36)
        F, en = c.compute(terms | L.TERM_COUL_PLAIN)
        out.append((F.cpu().numpy().copy(), en))
        assert c.status() == 0
        c.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
