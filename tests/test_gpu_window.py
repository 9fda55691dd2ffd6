"""The window kernel (one replica per workgroup, csrc/gasp_window.h), which the
automatic launch shape takes for the smaller replica counts of methods 0, 1 and
2, bit for bit against the CPU oracle: both key layouts, each number of waves
that the rule gives on a 256-CU device, both random streams, lattices whose
sites and whose attempts are odd in number, the measurement without sweeps,
frozen replicas, and a launch long enough to use up the rounds of its keys."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BETA, H = 0.54, 0.07


def _grids(R, L, seed, up=0.5):
    rs = np.random.default_rng(seed)
    return np.where(rs.random((R, L, L)) < up, 1, -1).astype(np.int32)


def _mag(g):
    return (g.reshape(len(g), -1).sum(1) / np.float32(g[0].size)).astype(np.float32)


# a dword per site: L = 2 .. 24 one wave, 32 two, 45 two or four, 64 eight, 128 eight; L = 201 is the largest
# with the spins in the entries, 202, 256 and 300 keep bits and a table
@pytest.mark.parametrize("method,L,R", [(2, 2, 70), (1, 3, 65), (2, 5, 33), (2, 16, 300), (1, 17, 100), (2, 24, 64),
                                        (2, 32, 100), (0, 45, 20), (1, 64, 9), (2, 75, 5), (2, 128, 3), (0, 201, 2),
                                        (0, 202, 2), (2, 256, 3), (0, 300, 2)])
@pytest.mark.parametrize("mt", [False, True])
def test_automatic_shape_bit_exact(gpu, engine_lib, oracle, method, L, R, mt):
    G, O = engine_lib, oracle
    print(f"[window] method={method} L={L} R={R} mt={mt}", flush=True)
    seed, beta = 4711 + L, 0.3
    g0 = _grids(R, L, seed)
    rng = G.RngState(R, seed, mt=mt)
    with G.Engine(L, R, method, rng, beta, H) as e:
        e.set_grids(g0)
        e.sweep(0)
        assert np.array_equal(e.magnetisation(), _mag(g0))
        e.sweep(2)
        e.sweep(1)
        got, mag, body, one = e.get_grids(), e.magnetisation(), e.gridstates(), e.gather([R - 1])
    rng.free()
    ref = O.sweep_mt_per_replica(L, g0.copy(), seed, 3, beta, H) if mt else O.sweep_philox(L, g0.copy(), seed, 0, 3 * L * L, beta, H)
    assert np.array_equal(got, ref)
    assert np.array_equal(mag, _mag(ref))
    assert np.array_equal(body, np.packbits((ref.reshape(-1) > 0).astype(np.uint8), bitorder="little"))
    assert np.array_equal(one[0], ref[R - 1].astype(np.int8))


# workgroups per CU: 4 waves each at L = 64 with 1024 replicas, 2 with 2048; at L = 200 a table from 512 replicas on
@pytest.mark.parametrize("method,L,R", [(2, 64, 1024), (1, 64, 2048), (0, 200, 700)])
def test_full_device(gpu, engine_lib, oracle, method, L, R):
    G, O = engine_lib, oracle
    print(f"[window full] method={method} L={L} R={R}", flush=True)
    g0 = _grids(R, L, 5, 0.03)
    rng = G.RngState(R, 99)
    with G.Engine(L, R, method, rng, BETA, H) as e:
        e.set_grids(g0)
        e.sweep(1)
        e.sweep(1)
        got = e.get_grids()
    rng.free()
    assert np.array_equal(got, O.sweep_philox(L, g0.copy(), 99, 0, 2 * L * L, BETA, H))


@pytest.mark.parametrize("method,L,R", [(2, 16, 70), (1, 33, 40), (0, 64, 12), (2, 210, 3)])
def test_caller_grids(gpu, engine_lib, oracle, method, L, R):
    """gasp_sweep_grids works on the caller's int32 grids in place, two calls in
    a row (the second starts at an odd attempt where L is odd)."""
    G, O = engine_lib, oracle
    print(f"[window grids] method={method} L={L} R={R}", flush=True)
    g0 = _grids(R, L, 8)
    ip = C.POINTER(C.c_int)
    d, nb = C.c_void_p(), C.c_void_p()
    G.lib().gpuInitGrid(L, R, 64, g0.ctypes.data_as(ip), C.byref(d), C.byref(nb))
    G.check()
    rng = G.RngState(R, 31)
    got = np.empty_like(g0)
    try:
        for n in (1, 2):
            G.check(G.lib().gasp_sweep_grids(L, R, method, rng.ptr, 0.3, H, d, n, None, None))
        G._d2h(got, d)
    finally:
        rng.free()
        G.lib().gasp_free(d)
        G.lib().gasp_free(nb)
    assert np.array_equal(got, O.sweep_philox(L, g0.copy(), 31, 0, 3 * L * L, 0.3, H))


@pytest.mark.parametrize("L", [2, 64])
def test_classes_that_never_flip(gpu, engine_lib, oracle, L):
    """At beta = 6 the thresholds of the costly flips are 0: no draw is below."""
    G, O = engine_lib, oracle
    R = 20
    print(f"[window never] L={L}", flush=True)
    g0 = _grids(R, L, 3)
    rng = G.RngState(R, 5)
    with G.Engine(L, R, 2, rng, 6.0, H) as e:
        e.set_grids(g0)
        e.sweep(4)
        got = e.get_grids()
    rng.free()
    assert np.array_equal(got, O.sweep_philox(L, g0.copy(), 5, 0, 4 * L * L, 6.0, H))


@pytest.mark.parametrize("method", [1, 2])
def test_frozen_replicas_keep_their_spins(gpu, engine_lib, oracle, method):
    G, O = engine_lib, oracle
    L, R = 32, 90
    print(f"[window freeze] method={method}", flush=True)
    g0 = _grids(R, L, 12)
    fates = np.where(np.arange(R) % 3 == 0, np.arange(R) % 2, -1).astype(np.int32)
    rng = G.RngState(R, 6)
    with G.Engine(L, R, method, rng, 0.3, H) as e:
        e.set_grids(g0)
        e.set_freeze(True)
        e.set_fates(fates)
        e.sweep(2, G.CHECK_FATES, -2.0, 2.0)
        got, mag, counts, after = e.get_grids(), e.magnetisation(), e.counts(), e.fates()
    rng.free()
    ref = O.sweep_philox(L, g0.copy(), 6, 0, 2 * L * L, 0.3, H)
    ref[fates != -1] = g0[fates != -1]
    assert np.array_equal(got, ref)
    assert np.array_equal(mag, _mag(ref))
    assert np.array_equal(after, fates)
    assert list(counts[1:]) == [int((fates == 0).sum()), int((fates == 1).sum())]


def test_more_rounds_than_keys(gpu, engine_lib, oracle):
    """Four sites commit at most two attempts a round (a neighbour of both
    remaining sites is in every stencil), so 1.2 million attempts in one
    launch take more rounds than the 2^18 that a packed key can count."""
    G, O = engine_lib, oracle
    L, R, n = 2, 3, 300000
    print("[window rounds]", flush=True)
    g0 = _grids(R, L, 1)
    rng = G.RngState(R, 17)
    with G.Engine(L, R, 2, rng, 0.3, H) as e:
        e.set_grids(g0)
        e.sweep(n)
        got = e.get_grids()
    rng.free()
    assert np.array_equal(got, O.sweep_philox(L, g0.copy(), 17, 0, n * L * L, 0.3, H))
