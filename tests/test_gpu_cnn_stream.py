"""The surrogate's streamed kernels (csrc/gasp_cnn_stream.h, L <= 64) against the
CPU oracle at the sizes where their division of the work changes: images side by
side in a group and groups that are not full (L = 16 and 32), more groups than
workgroups, bands of an image, chains of several bands, and inference in several
pieces.  Tolerances as in test_gpu_cnn.py."""
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


# L = 16: 275 groups of four images, the last with one; 32: 23 groups, the last half full; 64: bands of 8 rows
@pytest.mark.parametrize("L,n,batch", [(16, 1097, 1097), (32, 45, 45), (64, 7, 7), (64, 7, 3)])
def test_forward(gpu, engine_lib, L, n, batch):
    K, p, spins, _ = _case(L, n, 3)
    print(f"[stream fwd] L={L} n={n} batch={batch}", flush=True)
    with engine_lib.Surrogate(L, batch) as net:
        net.set_params(p)
        got = net.predict(spins)
    ref = K.forward(p.astype(np.float64), spins.astype(np.float64), bf16=True)["pB"]
    assert np.max(np.abs(got - ref)) < 2e-3


# chains: 32 of 5 or 6 bands (64, 10: at most four per image of the largest batch), one band each (32, 5), 768 of 1 or
# 2 bands (16, 250)
@pytest.mark.parametrize("L,n,batch", [(16, 250, 250), (16, 3, 64), (32, 5, 64), (64, 10, 10)])
def test_gradient(gpu, engine_lib, L, n, batch):
    K, p, spins, y = _case(L, n, 4)
    print(f"[stream grad] L={L} n={n} batch={batch}", flush=True)
    with engine_lib.Surrogate(L, batch) as net:
        net.set_params(p)
        loss, g = net.gradient(spins, y)
    rl, rg, _ = K.loss_and_grad(p.astype(np.float64), spins.astype(np.float64), y.astype(np.float64), bf16=True)
    assert abs(loss - rl) < 1e-3 * max(1.0, abs(rl))
    Gg, Gr = K.unflatten(g), K.unflatten(rg)
    for name, _ in K.SHAPES:
        a, b = Gg[name].ravel(), Gr[name].ravel()
        assert np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12) < 2e-2, name


def test_pieces_and_batches_agree(gpu, engine_lib):
    """4500 grids of L = 16 in one call (two pieces on 256 CUs), in batches of
    1000 and one by one: the same network, up to the order of the pooled sums
    (1024 float32 additions of non-negative numbers: a relative 1024 x 2^-24)."""
    K, p, spins, _ = _case(16, 4500, 5)
    print("[stream pieces]", flush=True)
    out = []
    for batch in (4500, 1000):
        with engine_lib.Surrogate(16, batch) as net:
            net.set_params(p)
            out.append(net.predict(spins))
            if batch == 1000:
                out.append(np.concatenate([net.predict(spins[i:i + 1]) for i in range(0, 4500, 300)]))
    assert np.max(np.abs(out[0] - out[1])) < 1e-4
    assert np.max(np.abs(out[0][::300] - out[2])) < 1e-4


def test_epoch_is_steps(gpu, engine_lib):
    """An epoch over resident data is the same steps as train_step on its batches."""
    K, p, spins, y = _case(16, 70, 6)
    order = np.random.default_rng(1).permutation(70).astype(np.int32)
    print("[stream epoch]", flush=True)
    with engine_lib.Surrogate(16, 32) as net:
        net.set_params(p)
        net.set_data(spins, y)
        mean = net.train_epoch(order, 32, 1e-3)
        a = net.params()
        net.set_params(p)
        losses = [net.train_step(spins[order[i:i + 32]], y[order[i:i + 32]], 1e-3) for i in (0, 32, 64)]
        b = net.params()
    assert np.array_equal(a, b)
    assert abs(mean - (32 * losses[0] + 32 * losses[1] + 6 * losses[2]) / 70) < 1e-6
