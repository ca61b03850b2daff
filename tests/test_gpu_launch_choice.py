"""GPU test that a context finds back to the nonbonded launch shape chosen by system size: lanes per atom order the
float32 sums of a row, so equal forces mean equal lanes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,lanes", [(216, 64), (1100, 32), (2800, 16)])
def test_back_to_the_choice_by_size(waters, lanes):
    from mdpy_amd import _lib as L, systems
    from mdpy_amd.engine import Engine
    print("case: %d waters" % waters, flush=True)
    terms = L.TERM_LJ | L.TERM_COUL_DIRECT
    m = int(np.ceil(waters ** (1 / 3)))
    s = systems.water_box(m, 3.1, n_waters=waters, seed=1, cutoff=9.0, pme_grid=(24, 24, 24))
    e = Engine(s)
    e.set_positions(s.positions)
    forces = lambda: e.compute_forces_only(terms).cpu().numpy().copy()
    F = forces()
    # a tuning run that fails leaves the choice as it was
    with pytest.raises(Exception, match="nonbonded timing needs"):
        e.tune_nonbonded(L.TERM_BOND, 0)
    assert np.array_equal(F, forces())
    other = 16 if lanes == 64 else 64
    assert e.tune_nonbonded(terms, other) == other and not np.array_equal(F, forces())
    assert e.tune_nonbonded(terms, -1) == lanes and np.array_equal(F, forces())
    assert e.tune_nonbonded(terms, lanes) == lanes and np.array_equal(F, forces())
    for per_cu in (2, -1):
        e.set_nonbonded_persist(per_cu)
        assert np.array_equal(F, forces())
    for bad in (lambda: e.tune_nonbonded(terms, 8), lambda: e.set_nonbonded_persist(-2)):
        with pytest.raises(Exception):
            bad()
    e.close()
