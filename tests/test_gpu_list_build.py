"""GPU tests of the neighbour-list build against float64 distances: boxes whose stencil wraps
onto itself and boxes where it does not, every cell width, crowded cells, cells shared by several
workgroups, and exclusions inside and outside the window of the exclusion masks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def partners(n, offsets):
    """Symmetric CSR of the pairs (i, i + d)."""
    rows = [sorted([i + d for d in offsets if i + d < n] + [i - d for d in offsets if i >= d]) for i in range(n)]
    return np.cumsum([0] + [len(r) for r in rows]), np.array([j for r in rows for j in r], int)


# (atoms, box, cutoff, skin, cells per list radius, excluded index distances, clustered)
CASES = [
    (1, (30.0, 31.0, 32.0), 9.0, 1.0, 2, (), False),
    (63, (18.5, 18.5, 18.5), 8.0, 1.0, 2, (1, 2), False),       # 27 cells, eight workgroups each
    (648, (18.64, 19.5, 21.25), 9.0, 0.3, 2, (1, 2, 40), False),  # wraps; exclusions outside the window
    (1500, (18.0, 40.0, 70.0), 8.0, 1.0, 2, (1, 31, 32), False),  # wraps along two axes only
    (4100, (48.0, 52.0, 60.0), 6.0, 1.5, 2, (1, 2, 30), False),
    (2500, (50.0, 41.0, 45.0), 9.0, 1.0, 1, (1, 33), False),
    (3000, (45.0, 47.0, 51.0), 9.0, 1.0, 3, (), False),
    (14000, (33.0, 33.0, 33.0), 7.0, 1.0, 1, (1, 40), False),   # crowded cells: over 192 home atoms
    (700, (60.0, 33.0, 60.0), 7.0, 1.0, 2, (5,), True),
]


@pytest.mark.parametrize("n,box,rc,skin,cells,offsets,clustered", CASES)
def test_lists_against_float64(n, box, rc, skin, cells, offsets, clustered):
    from scipy.spatial import cKDTree
    from mdpy_amd.engine import Engine
    print("case: %d atoms, box %s, %d cells a radius" % (n, box, cells), flush=True)
    rng = np.random.default_rng(n)
    box = np.array(box)
    x = (rng.random((n, 3)) - 0.5) * box
    if clustered:  # some atoms close together around the corner of the box
        m = 50
        x[:m] = 0.5 * box + rng.normal(size=(m, 3)) * 1.0
    ptr, idx = partners(n, offsets)
    e = Engine.bare(n, box, positions=x + box * rng.integers(-1, 2, (n, 3)))
    e.set_masses(np.ones(n))
    e.set_charges(np.zeros(n))
    e.set_lj(np.tile([0.1, 1.0, 0.1, 1.0], (n, 1)))
    e.set_exclusions(ptr, idx)
    e.set_scaling(np.zeros(n + 1, int), [])
    e.configure_nonbonded(rc, skin=skin)
    e.set_list_cells(cells)
    got = e.neighbor_pairs()
    got = set(map(tuple, np.asarray(got).tolist()))
    listed = e.pair_counts()[0]
    rl2 = (rc + skin) ** 2
    i, j = cKDTree(np.mod(x, box), boxsize=box).query_pairs(1.001 * (rc + skin), output_type="ndarray").T
    keep = ~np.isin(np.abs(i - j), offsets)
    i, j = np.minimum(i, j)[keep], np.maximum(i, j)[keep]
    d = x[j] - x[i]
    d -= box * np.round(d / box)
    r2 = (d * d).sum(1)
    want = set(zip(i[r2 <= rc * rc].tolist(), j[r2 <= rc * rc].tolist()))
    # the radius carries 1e-5 of slack, and rounding less than that again
    lo, hi = 2 * int((r2 < rl2).sum()), 2 * int((r2 < rl2 * (1 + 2e-5)).sum())
    assert got == want
    assert lo <= listed <= hi
    assert e.status() == 0
    e.close()


@pytest.mark.parametrize("n,box", [(500, (17.0, 18.0, 19.0)), (2000, (40.0, 42.0, 44.0))])
@pytest.mark.parametrize("far", [3, 45])
def test_scaled_pairs_inside_and_outside_the_window(n, box, far):
    """1-4 pairs take their own LJ parameters, by mask bits or by list: with the scaled epsilon 0 the
    forces are those of the same pairs excluded (no charges)."""
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    print("case: %d atoms, partners %d apart" % (n, far), flush=True)
    rng = np.random.default_rng(n + far)
    box, m = np.array(box), int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g + 0.5) * box / m + rng.uniform(-0.2, 0.2, (n, 3)) - 0.5 * box
    ptr, idx = partners(n, (far,))
    none = np.zeros(n + 1, int)
    F = []
    for scaled in (True, False):
        e = Engine.bare(n, box, positions=x)
        e.set_masses(np.ones(n))
        e.set_charges(np.zeros(n))
        e.set_lj(np.tile([0.1, 2.0, 0.0, 2.0], (n, 1)))
        e.set_exclusions(*((none, []) if scaled else (ptr, idx)))
        e.set_scaling(*((ptr, idx) if scaled else (none, [])))
        e.configure_nonbonded(7.5, skin=0.8)
        F.append(e.compute_forces_only(L.TERM_LJ).cpu().numpy().copy())
        assert e.status() == 0
        e.close()
    # 32-bit terms summed in another grouping: 1e-6 of the largest force is some 10 of its roundings
    assert np.abs(F[0]).max() > 0
    assert np.abs(F[0] - F[1]).max() <= 1e-6 * np.abs(F[0]).max()
