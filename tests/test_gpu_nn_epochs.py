"""kmi_nn_train_epochs (targets read where the dataset keeps them, the step's loss and the weight
copies in the Adam launch) against single train steps on the same mini-batches.

Both run the same products in the same order on the same values, so the parameters must be equal
bit for bit; the mean loss is the mean of the steps' losses up to one rounding per addition.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _shuffles(n, epochs, seed):
    """The epochs' permutations: Fisher–Yates on splitmix64."""
    s = seed & M64
    out = []
    for _ in range(epochs):
        p = list(range(n))
        for i in range(n - 1, 0, -1):
            s = (s + 0x9E3779B97F4A7C15) & M64
            z = s
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
            z ^= z >> 31
            j = z % (i + 1)
            p[i], p[j] = p[j], p[i]
        out.append(p)
    return out


# channels that the gradient's rows fill, pad by one to five, and spread over two stores; direct
# and general convolution kernels (hidden maps of 16 to 64, channel counts outside 32 and 64)
@pytest.mark.parametrize("arch,n,batch", [
    (dict(in_dim=2, latent_hw=16, out_c=3), 11, 4),
    (dict(in_dim=3, latent_hw=4, out_c=8), 9, 8),
    (dict(in_dim=1, hidden=64, latent_hw=8, latent_c=32, c1=64, c2=32, out_c=11), 7, 3),
    (dict(in_dim=5, hidden=32, latent_hw=3, latent_c=8, c1=24, c2=64, out_c=1), 5, 1),
    (dict(in_dim=2, hidden=64, latent_hw=8, latent_c=64, c1=16, c2=8, out_c=2), 6, 2),
])
def test_epochs_equal_single_steps(kmi, backend, arch, n, batch):
    from kraken_mi355x.nn import WarmStartNet

    r = np.random.default_rng(n)
    side = 8 * arch["latent_hw"]
    x = r.standard_normal((n, arch["in_dim"])).astype(np.float32)
    y = r.standard_normal((n, side, side, arch["out_c"])).astype(np.float32)
    epochs, seed, lr = 2, 77, 1e-3
    print(f"[epochs] {arch} n={n} batch={batch}", flush=True)
    a = WarmStartNet(max_batch=batch, seed=3, backend=backend, **arch)
    b = WarmStartNet(max_batch=batch, seed=3, backend=backend, **arch)
    a.set_dataset(x, y)
    mean = a.train_epochs(epochs, batch, lr, seed=seed)
    for p in _shuffles(n, epochs, seed):
        losses = [b.train_step(x[p[k:k + batch]], y[p[k:k + batch]], lr) for k in range(0, n - batch + 1, batch)]
    assert np.array_equal(a.get_params(), b.get_params())
    assert abs(mean - np.mean(losses)) <= len(losses) * np.finfo(np.float64).eps * mean
    a.close()
    b.close()
