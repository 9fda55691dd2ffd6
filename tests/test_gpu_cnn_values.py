"""Grids of other values than +-1 (a 0/1 coding, say) through the surrogate at
L <= 64, whose streamed kernels read a spin's sign only: such a batch is evaluated
on its values, as at L >= 128, by the separate kernels.  Against the CPU oracle
with the tolerances of test_gpu_cnn.py; conv1's weight gradient, which takes the
spins' signs at every L, is left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(L, n, seed):
    from oracle import cnn_oracle as K

    rs = np.random.default_rng(seed)
    p = (K.init_params(seed).astype(np.float64) + rs.normal(0.0, 0.05, K.NPARAM)).astype(np.float32)
    frac = rs.uniform(0.1, 0.9, n)[:, None, None]
    spins = np.where(rs.random((n, L, L)) < frac, 1, -1).astype(np.int8)
    return K, p, spins, rs.uniform(0, 1, n).astype(np.float32)


# one grid of 0/1 among +-1: in the first of two pieces (L = 16: 4096 grids each), in the last, in the only one; every
# value of an int8 that a wrong test of the bits could let through, one of them alone
@pytest.mark.parametrize("L,n,batch,where", [(16, 4500, 4500, 7), (16, 4500, 4500, 4499), (16, 70, 32, 40), (32, 5, 8, 4),
                                             (64, 3, 8, 0)])
@pytest.mark.parametrize("value", [0, 3, -2, 127, -128, 65])
def test_forward(gpu, engine_lib, L, n, batch, where, value):
    K, p, spins, _ = _case(L, n, 11)
    print(f"[values fwd] L={L} n={n} batch={batch} grid {where} value {value}", flush=True)
    if value == 0:
        spins[where] = spins[where] > 0
    else:
        spins[where, L - 1, L - 1] = value
    with engine_lib.Surrogate(L, batch) as net:
        net.set_params(p)
        got = net.predict(spins)
        spins2 = np.where(spins > 0, 1, -1).astype(np.int8)
        again = net.predict(spins2)  # +-1 again
    pick = np.unique(np.r_[where, 0, n - 1, np.arange(0, n, max(1, n // 40))])
    for g, s in ((got, spins), (again, spins2)):
        ref = K.forward(p.astype(np.float64), s[pick].astype(np.float64), bf16=True)["pB"]
        assert np.max(np.abs(g[pick] - ref)) < 2e-3


@pytest.mark.parametrize("L,n,batch", [(16, 9, 16), (16, 40, 40), (32, 5, 5), (64, 3, 8)])
def test_gradient(gpu, engine_lib, L, n, batch):
    K, p, spins, y = _case(L, n, 12)
    print(f"[values grad] L={L} n={n} batch={batch}", flush=True)
    spins[n // 2] = spins[n // 2] > 0
    with engine_lib.Surrogate(L, batch) as net:
        net.set_params(p)
        loss, g = net.gradient(spins, y)
    rl, rg, _ = K.loss_and_grad(p.astype(np.float64), spins.astype(np.float64), y.astype(np.float64), bf16=True)
    assert abs(loss - rl) < 1e-3 * max(1.0, abs(rl))
    Gg, Gr = K.unflatten(g), K.unflatten(rg)
    for name, _ in K.SHAPES:
        if name != "w1":
            a, b = Gg[name].ravel(), Gr[name].ravel()
            assert np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-12) < 2e-2, name


def test_training(gpu, engine_lib):
    """A step takes the gradient of the values, once, and an epoch over stored data is its steps."""
    K, p, spins, y = _case(16, 70, 13)
    print("[values training]", flush=True)
    spins[::3] = spins[::3] > 0
    order = np.random.default_rng(1).permutation(70).astype(np.int32)
    with engine_lib.Surrogate(16, 32) as net:
        net.set_params(p)
        _, g = net.gradient(spins[:20], y[:20])
        net.train_step(spins[:20], y[:20], 1e-3)
        one = net.params()
        net.set_params(p)
        net.set_data(spins, y)
        mean = net.train_epoch(order, 32, 1e-3)
        a = net.params()
        net.set_params(p)
        losses = [net.train_step(spins[order[i:i + 32]], y[order[i:i + 32]], 1e-3) for i in (0, 32, 64)]
        b = net.params()
    ref, _, _ = K.adam_step(p.astype(np.float64), g.astype(np.float64), np.zeros(K.NPARAM), np.zeros(K.NPARAM), 1)
    assert np.max(np.abs(one - ref)) < 1e-6
    assert np.array_equal(a, b)
    assert abs(mean - (32 * losses[0] + 32 * losses[1] + 6 * losses[2]) / 70) < 1e-6


def test_data_that_do_not_fit(gpu, engine_lib):
    """Training data beyond the device's memory are refused, and epochs with them, until there are some again."""
    import ctypes as C

    G = engine_lib
    K, p, spins, y = _case(64, 6, 14)
    print("[values data]", flush=True)
    order = np.arange(6, dtype=np.int32)
    with G.Surrogate(64, 6) as net:
        net.set_params(p)
        net.set_data(spins, y)
        rc = G.lib().gasp_cnn_set_data(net.ptr, spins.ctypes.data_as(C.POINTER(C.c_int8)),
                                       y.ctypes.data_as(C.POINTER(C.c_float)), 2**31 - 1)  # 8.8 TB, refused before it is read
        assert rc != 0
        with pytest.raises(G.GaspError):
            net.train_epoch(order, 6, 1e-3)
        with pytest.raises(G.GaspError):
            net.train_epoch(order[:1], 1, 1e-3)
