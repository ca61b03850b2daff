"""The analysers' two selections on the CPU (the pair histograms replaced by a numpy double loop): conditions
whose values are arrays, equal and unequal, in the same object or in two."""
import numpy as np
import pytest


def frames():
    """Four waters in two frames."""
    from mdpy_amd import systems
    from mdpy_amd.core import Topology, Trajectory
    s = systems.water_box(2, 3.1, n_waters=4, seed=1, cutoff=3.0, pme_grid=(8, 8, 8))
    t = Trajectory(Topology.from_system(s))
    t.set_pbc_matrix(s.pbc_matrix)
    t.append(s.positions)
    t.append(s.positions + 0.1)
    return t


def histograms(trajectory, ids1, ids2, cutoff_radius, num_bins, device=0):
    edges = np.linspace(0, cutoff_radius, num_bins + 1)
    box = np.diag(np.asarray(trajectory.pbc_matrix, dtype=np.float64))
    counts = np.zeros((len(ids1), num_bins), dtype=np.int64)
    for x in np.asarray(trajectory.positions, dtype=np.float64):
        for a, i in enumerate(ids1):
            d = x[i] - x[ids2]
            d -= box * np.round(d / box)
            counts[a] += np.histogram(np.sqrt((d * d).sum(1)), edges)[0]
    return counts, edges


def conditions():
    """Pairs of conditions and the matrix ids that each selects."""
    a, b = np.array([0, 3, 6]), np.array([0, 3, 6])
    shared = [{"particle id": [a]}]
    return [([{"particle id": [a]}], [{"particle id": [b]}], [0, 3, 6], [0, 3, 6]),
            ([{"particle id": [a]}], [{"particle id": [np.array([1, 2, 4, 5])]}], [0, 3, 6], [1, 2, 4, 5]),
            ([{"particle id": [a]}], [{"particle id": [np.array([3])]}], [0, 3, 6], [3]),
            ([{"particle id": [a]}], [{"particle id": [[0, 3, 6]]}], [0, 3, 6], [0, 3, 6]),
            (shared, shared, [0, 3, 6], [0, 3, 6]),
            ([{"particle type": [np.array(["OT"])]}], [{"particle type": [["HT"]]}], [0, 3, 6, 9],
             [1, 2, 4, 5, 7, 8, 10, 11])]


@pytest.mark.parametrize("k", range(6))
@pytest.mark.parametrize("name", ["RDFAnalyser", "CoordinationNumberAnalyser"])
def test_conditions_with_arrays(monkeypatch, name, k):
    from mdpy_amd import analyser
    module = __import__("mdpy_amd.analyser." + {"RDFAnalyser": "rdf_analyser",
                                                "CoordinationNumberAnalyser": "coordination_number_analyser"}[name],
                        fromlist=["pair_histograms"])
    seen = []

    def recorded(trajectory, ids1, ids2, *args, **kw):
        seen.append((list(ids1), list(ids2)))
        return histograms(trajectory, ids1, ids2, *args, **kw)

    monkeypatch.setattr(module, "pair_histograms", recorded)
    c1, c2, ids1, ids2 = conditions()[k]
    r = getattr(analyser, name)(c1, c2, 3.0, 12).analysis(frames())
    assert seen == [(ids1, ids2)]
    assert np.all(np.isfinite(r.data["mean"])) and len(r.data["mean"]) == 12
