"""The surrogate's streamed kernels (csrc/gasp_cnn_stream.h, L <= 64) at the sizes
of real training batches: whole images through a workgroup (a network's default
batch of 256 at L = 64), groups that are not full, several chains of the weight
gradient per workgroup, and several images per workgroup in inference.  Tolerances
against the oracle as in test_gpu_cnn.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(L, n, seed):
    from oracle import cnn_oracle as K

    rs = np.random.default_rng(seed)
    p = (K.init_params(seed).astype(np.float64) + rs.normal(0.0, 0.05, K.NPARAM)).astype(np.float32)
    frac = rs.uniform(0.05, 0.95, n)[:, None, None]
    spins = np.where(rs.random((n, L, L)) < frac, 1, -1).astype(np.int8)
    return K, p, spins, rs.uniform(0, 1, n).astype(np.float32)


# on 256 CUs images are not cut into bands from 129 to 256 groups of 64 columns on (L = 64: 193); last group: 3 of 4, 1 of 2
@pytest.mark.parametrize("L,n", [(16, 515), (32, 259)])
def test_gradient_of_whole_images(gpu, engine_lib, L, n):
    K, p, spins, y = _case(L, n, 21)
    print(f"[training grad] L={L} n={n}", flush=True)
    with engine_lib.Surrogate(L, n) as net:
        net.set_params(p)
        loss, g = net.gradient(spins, y)
    rl, rg, _ = K.loss_and_grad(p.astype(np.float64), spins.astype(np.float64), y.astype(np.float64), bf16=True)
    assert abs(loss - rl) < 1e-3 * max(1.0, abs(rl))
    Gg, Gr = K.unflatten(g), K.unflatten(rg)
    for name, _ in K.SHAPES:
        a, b = Gg[name].ravel(), Gr[name].ravel()
        assert np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12) < 2e-2, name


# n = 256 at L = 64: whole images, three chains a workgroup; in parts of 8: bands of eight rows, 32 chains
@pytest.mark.parametrize("L,n,part", [(64, 256, 8), (32, 512, 16), (16, 1024, 32)])
def test_batch_is_the_mean_of_its_parts(gpu, engine_lib, L, n, part):
    """The loss and the gradient of a batch are the means over its parts.  n / part is a power of two, so that every
    rounding to bfloat16 is the same: what differs is the order of float32 sums.  These are of at most 2^22 terms in
    chains of under 200 additions, so a sum is off by at most 200 x 2^-24 = 1.2e-5 of the sum of its terms' sizes; with
    terms that cancel to a percent of that, 1.2e-3 of the result."""
    K, p, spins, y = _case(L, n, 22)
    print(f"[training parts] L={L} n={n} part={part}", flush=True)
    with engine_lib.Surrogate(L, n) as net:
        net.set_params(p)
        loss, g = net.gradient(spins, y)
    with engine_lib.Surrogate(L, part) as net:
        net.set_params(p)
        parts = [net.gradient(spins[i:i + part], y[i:i + part]) for i in range(0, n, part)]
    assert abs(loss - np.mean([q[0] for q in parts])) < 1e-6 * max(1.0, loss)
    Gg, Gr = K.unflatten(g), K.unflatten(np.mean([q[1].astype(np.float64) for q in parts], 0))
    for name, _ in K.SHAPES:
        a, b = Gg[name].ravel(), Gr[name].ravel()
        assert np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12) < 1.2e-3, name


@pytest.mark.parametrize("L,n", [(64, 200), (32, 259), (16, 515)])
def test_losses_do_not_depend_on_the_bands(gpu, engine_lib, L, n):
    """Whole images pool their features in net_fwd, single ones (cut into bands) in `head`, in the same order: the mean
    loss, summed in float64, has the same bits as the mean of the single images' losses."""
    K, p, spins, y = _case(L, n, 23)
    print(f"[training losses] L={L} n={n}", flush=True)
    with engine_lib.Surrogate(L, n) as net:
        net.set_params(p)
        loss, _ = net.gradient(spins, y)
        total = 0.0
        for k in range(n):
            total += net.gradient(spins[k:k + 1], y[k:k + 1])[0]
    assert np.float32(loss) == np.float32(total / n)


# several images a workgroup (the spins of the next are read beside this one's), in one upload and in two
@pytest.mark.parametrize("n,batch", [(300, 300), (1500, 1500)])
def test_forward_of_many_images(gpu, engine_lib, n, batch):
    K, p, spins, _ = _case(64, n, 24)
    print(f"[training fwd] n={n}", flush=True)
    with engine_lib.Surrogate(64, batch) as net:
        net.set_params(p)
        got = net.predict(spins)
    pick = np.unique(np.r_[0, 255, 256, n - 1, np.arange(7, n, n // 8)])
    ref = K.forward(p.astype(np.float64), spins[pick].astype(np.float64), bf16=True)["pB"]
    assert np.max(np.abs(got[pick] - ref)) < 2e-3
