"""An error that a call has reported is not reported again by the next calls: after
an allocation that the device's memory cannot hold, everything else still runs."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _works(G):
    rng = G.RngState(64, 3, mt=True)
    with G.Engine(16, 64, 2, rng, 0.4, 0.06) as e:
        e.set_grids(-np.ones((64, 16, 16), np.int32))
        e.sweep(1)
        assert e.magnetisation().shape == (64,)
    rng.free()


def test_engine_beyond_memory(gpu, engine_lib):
    G = engine_lib
    L, R = 8192, 100000  # 6.7 TB of spins at a byte each
    print("[errors] engine", flush=True)
    rng = G.RngState(R, 1)
    for method in (0, 1):
        with pytest.raises(G.GaspError):
            G.Engine(L, R, method, rng, 0.4, 0.06)
        _works(G)
    rng.free()


def test_surrogate_beyond_memory(gpu, engine_lib):
    G = engine_lib
    print("[errors] surrogate", flush=True)
    with pytest.raises(G.GaspError):
        G.Surrogate(64, 1 << 24)  # 17 TB of activations
    _works(G)
    spins = np.ones((4, 16, 16), np.int8)
    labels = np.ones(4, np.float32)
    with G.Surrogate(16, 4) as net:
        net.set_params(np.zeros(net.nparam, np.float32))
        rc = G.lib().gasp_cnn_set_data(net.ptr, spins.ctypes.data_as(C.POINTER(C.c_int8)),
                                       labels.ctypes.data_as(C.POINTER(C.c_float)), 2**31 - 1)
        assert rc != 0
        assert np.all(net.predict(spins) == 0.5)
        net.set_data(spins, labels)
        assert net.train_epoch(np.arange(4), 4, 1e-3) > 0
    _works(G)
