"""GPU test of the surrogate's force-matching gradients at the sizes where their kernels' splits end:
fewer rows of an element than chunks of the column sums, one more, and a few thousand; atoms with
fewer and with more neighbours than a wave. Against the float64 oracle."""
import numpy as np
import pytest

from oracle import mlp as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,spacing", [(2, 3.1), (43, 3.1), (129, 2.6), (300, 3.3)])
def test_gradients_at_small_and_odd_sizes(waters, spacing):
    import torch
    from mdpy_amd import systems
    from mdpy_amd.engine import Engine
    from mdpy_amd.mlp import Surrogate
    print("case: %d waters" % waters, flush=True)
    m = max(5, int(np.ceil(waters ** (1 / 3))))
    s = systems.water_box(m, spacing, n_waters=waters, seed=waters, cutoff=6.0, pme_grid=(16, 16, 16))
    e = Engine(s, skin=1.0)
    e.set_positions(s.positions)
    elem = M.elements_of(s.types)
    sur = Surrogate(e, elem, rd=6.0, skin=1.0, seed=1)
    x, box = e.positions(), np.asarray(s.box, dtype=np.float64)
    rng = np.random.default_rng(waters)
    nets = []
    for _ in range(2):
        n = M.init_net(rng, 256)
        for k in ("b1", "b2", "b3"):
            n[k] = rng.standard_normal(n[k].shape) * 0.1
        for k in ("W1", "W2", "W3"):  # weights that bfloat16 holds exactly
            u = np.ascontiguousarray(n[k], dtype=np.float32).view(np.uint32) & 0xFFFF0000
            n[k] = u.astype(np.uint32).view(np.float32).astype(np.float64)
        nets.append(n)
    G, _ = M.descriptors(x, box, elem)
    mean, std = G.mean(0), G.std(0) + 1e-1
    sur.set_params(nets)
    sur.set_norm(mean, std)
    fref = rng.standard_normal(x.shape) * 0.02
    loss = sur.train_step(torch.tensor(x, device="cuda"), torch.tensor(fref, device="cuda"), 0.0)
    got = sur.get_grads()
    ref = M.Surrogate(nets, mean.astype(np.float32).astype(np.float64), std.astype(np.float32).astype(np.float64))
    want_loss, want, _ = ref.loss_and_grad(x, box, elem, fref)
    sur.close()
    e.close()
    assert loss == pytest.approx(want_loss, rel=2e-2)
    # a gradient sums products of bfloat16-rounded activations, tangents and adjoints: up to six
    # roundings of 2^-9 in a term
    for el in range(2):
        for k in ("W1", "b1", "W2", "b2", "W3", "b3", "w4"):
            a, b = got[el][k].reshape(-1), np.asarray(want[el][k]).reshape(-1)
            err = np.linalg.norm(a - b) / np.linalg.norm(b)
            print("  elem %d %s %.3e" % (el, k, err), flush=True)
            assert err < 6 * 2.0 ** -9, (el, k)
