"""GPU test that the surrogate's descriptors are summed in the order they always were: the rows of its
list follow cells half a list radius wide. Another order is as accurate, but the last bit of a float32
sum flips bf16 activations, which moves the forces by some 1e-4 for no reason a user could see.

The recorded values (tests/golden/data/surrogate_water1536.npz) were computed with the list build that
preceded the one on box fractions: descriptors and forces of every 24th atom."""
import os

import numpy as np
import pytest

from conftest import GOLDEN
from oracle import mlp as M

pytestmark = pytest.mark.gpu

RECORD = os.path.join(GOLDEN, "data", "surrogate_water1536.npz")


def evaluate(mean=None, std=None):
    """Descriptors, forces and energy of a 512-water box with seeded networks."""
    from mdpy_amd import systems
    from mdpy_amd.engine import Engine
    from mdpy_amd.mlp import Surrogate
    s = systems.water_box(8, 3.1, seed=11, cutoff=9.0, pme_grid=(24, 24, 24), name="w512")
    e = Engine(s, skin=1.0)
    e.set_positions(s.positions)
    sur = Surrogate(e, M.elements_of(s.types), rd=6.0, skin=1.0, seed=1)
    rng = np.random.default_rng(4)
    nets = [M.init_net(rng, 256) for _ in range(2)]
    sur.set_params(nets)
    G = sur.descriptors().cpu().numpy()
    if mean is None:
        mean, std = G.mean(0), G.std(0) + 1e-3
    sur.set_norm(mean, std)
    F, E = sur.eval()
    F = F.cpu().numpy().copy()
    sur.close()
    e.close()
    return G, F, E, mean, std


def test_surrogate_sums_keep_their_order():
    z = np.load(RECORD)
    print("case: recorded descriptors and forces, 1,536 atoms", flush=True)
    G, F, E, _, _ = evaluate(z["mean"], z["std"])
    G, F = G[::24], F[::24]
    changed = np.count_nonzero(G != z["G"]) / G.size
    err = np.linalg.norm(F - z["F"]) / np.linalg.norm(z["F"])
    print("  descriptors that differ in any bit %.2e, forces %.2e" % (changed, err), flush=True)
    # the same sums of the same roundings: equal bits, but for atoms with a partner within rounding of the
    # list radius (about one in 25,000: whether it is listed shifts the 64s that are summed together). A
    # list in another order changes nearly half of the descriptors, and the forces by 4e-4
    assert changed <= 1e-3 and np.allclose(G, z["G"], rtol=1e-5, atol=1e-7)
    assert err <= 1e-6 and abs(E - float(z["E"])) <= 1e-6 * abs(float(z["E"]))
