"""GPU tests of the kernels that walk all pairs in slices: plain Coulomb against a float64 double
loop, at atom counts around the tile and slice edges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def box_of(n, seed, L=25.0):
    rng = np.random.default_rng(seed)
    return rng.uniform(-0.5 * L, 0.5 * L, (n, 3)), np.array([L, L * 1.07, L * 0.93])


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 1000])
def test_plain_coulomb_slices(n):
    """Exclusions inside and across tiles, zero charges (one of them on top of another atom). Each
    component carries at most one fixed-point rounding (2^-41) and float64 sums of n terms."""
    import ctypes
    from mdpy_amd import _lib as L
    from mdpy_amd.engine import Engine
    from mdpy_amd.unit import ONE_OVER_4PI_EPS0
    print("case: plain Coulomb, %d atoms" % n, flush=True)
    x, box = box_of(n, n)
    rng = np.random.default_rng(n + 1)
    q = rng.uniform(-1, 1, n)
    q[rng.random(n) < 0.1] = 0.0
    if n > 64:
        x[64], q[64] = x[3], 0.0
    rows = [[] for _ in range(n)]
    for _ in range(n):
        a, b = rng.integers(0, n, 2)
        if a != b and b not in rows[a]:
            rows[a].append(int(b))
            rows[b].append(int(a))
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    idx = np.array([j for r in rows for j in r], dtype=np.int64)
    e = Engine.bare(n, box, positions=x)
    e.set_masses(np.ones(n))
    e.set_charges(q)
    e.set_exclusions(ptr, idx)
    F, en = e.compute(L.TERM_COUL_PLAIN)
    F = F.cpu().numpy()
    e.close()
    d = x[None, :, :] - x[:, None, :]
    d -= box * np.round(d / box)
    see = (q[:, None] * q[None, :] != 0) & ~np.eye(n, dtype=bool)
    for a, r in enumerate(rows):
        see[a, r] = False
    r2 = np.where(see, (d * d).sum(-1), 1.0)
    w = np.where(see, ONE_OVER_4PI_EPS0 * q[:, None] * q[None, :], 0.0) / np.sqrt(r2)
    ref = -(d * (w / r2)[:, :, None]).sum(1)
    size = (np.abs(d) * np.abs(w / r2)[:, :, None]).sum(1)
    assert np.all(np.abs(F - ref) <= 2.0 ** -41 + 8 * n * 2.0 ** -53 * size)
    blocks = (n + 255) // 256
    assert abs(en["coulomb_plain"] - 0.5 * w.sum()) <= blocks * 2.0 ** -41 + 8 * n * 2.0 ** -53 * np.abs(w).sum()
