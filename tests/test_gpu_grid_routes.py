"""gasp_sweep_grids and gasp_sweep_grids_noalloc on both of their routes, whichever
kernel the launch shape takes: in place on the caller's grids (one replica per
workgroup), and through the native layout (pack, sweep, unpack)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BETA, H = 0.4, 0.06
# an explicit shape keeps a method's other kernels
EXPLICIT = {0: (16, 1), 1: (16, 2), 2: (16, 2), 3: (2, 1)}


@pytest.fixture
def automatic(engine_lib):
    yield
    engine_lib.set_tuning(0, 0)


def _device_grids(G, g):
    L, R = g.shape[1], g.shape[0]
    d, nb = C.c_void_p(), C.c_void_p()
    G.lib().gpuInitGrid(L, R, 64, g.ctypes.data_as(C.POINTER(C.c_int)), C.byref(d), C.byref(nb))
    G.check()
    G.lib().gasp_free(nb)
    return d


def _mag(g):
    return (g.reshape(len(g), -1).sum(1) / np.float32(g[0].size)).astype(np.float32)


@pytest.mark.parametrize("explicit", [False, True])
@pytest.mark.parametrize("method,L,R", [(0, 16, 40), (0, 40, 20), (1, 33, 70), (2, 32, 100), (2, 210, 2)])
def test_other_values_count_as_down(gpu, engine_lib, oracle, automatic, explicit, method, L, R):
    """A call without sweeps measures and leaves +-1, as one with sweeps does: any value but 1 is a down spin."""
    G, O = engine_lib, oracle
    if explicit:
        G.set_tuning(*((8, 8) if L == 210 else EXPLICIT[method]))
    print(f"[routes 0 sweeps] method={method} L={L} R={R} explicit={explicit}", flush=True)
    g0 = np.random.default_rng(L).integers(-1, 3, (R, L, L)).astype(np.int32)
    want = np.where(g0 == 1, 1, -1).astype(np.int32)
    d, d_mag = _device_grids(G, g0), _device_grids(G, np.zeros((R, 1, 1), np.int32))
    rng = G.RngState(R, 5)
    got, mag = np.empty_like(g0), np.empty(R, np.float32)
    try:
        for n in (0, 1):
            G.check(G.lib().gasp_sweep_grids(L, R, method, rng.ptr, BETA, H, d, n, d_mag, None))
            G._d2h(got, d)
            G._d2h(mag, d_mag)
            if n:
                want = O.sweep_philox(L, want, 5, 0, L * L, BETA, H)
            assert np.array_equal(got, want), n
            assert np.array_equal(mag, _mag(want)), n
    finally:
        rng.free()
        G.lib().gasp_free(d)
        G.lib().gasp_free(d_mag)


# explicit shapes; 256 slots spread a method-0 replica over four waves; and counts above the lines of the one-replica kernel
@pytest.mark.parametrize("method,L,R,shape", [(0, 64, 9, (256, 4)), (0, 17, 50, (16, 1)), (1, 24, 70, (16, 2)),
                                              (1, 33, 100, (8, 1)), (2, 64, 130, (16, 2)), (2, 33, 70, (8, 1)),
                                              (2, 32, 200, (16, 4)), (2, 48, 1000, (16, 2)), (0, 9, 16500, None),
                                              (1, 9, 16500, None), (2, 9, 16500, None)])
@pytest.mark.parametrize("noalloc", [False, True])
def test_native_layout_route(gpu, engine_lib, oracle, automatic, noalloc, method, L, R, shape):
    """Two calls in a row with a magnetisation buffer, then one without, which moves the lattice in the workspace."""
    G, O = engine_lib, oracle
    if shape:
        G.set_tuning(*shape)
    assert G.get_window(method, L, R) == (0, 0)
    print(f"[routes native] method={method} L={L} R={R} shape={shape} noalloc={noalloc}", flush=True)
    fn = G.lib().gasp_sweep_grids_noalloc if noalloc else G.lib().gasp_sweep_grids
    rs = np.random.default_rng(L + R)
    want = np.where(rs.random((R, L, L)) < 0.35, 1, -1).astype(np.int32)
    got, mag = np.empty_like(want), np.empty(R, np.float32)
    d, d_mag = _device_grids(G, want), _device_grids(G, np.zeros((R, 1, 1), np.int32))
    rng = G.RngState(R, 77)
    at = 0
    try:
        for n, with_mag in ((2, True), (1, True), (1, False)):
            G.check(fn(L, R, method, rng.ptr, BETA, H, d, n, d_mag if with_mag else None, None))
            want = O.sweep_philox(L, want, 77, at, n * L * L, BETA, H)
            at += n * L * L
            G._d2h(got, d)
            assert np.array_equal(got, want), (n, with_mag)
            if with_mag:
                G._d2h(mag, d_mag)
                assert np.array_equal(mag, _mag(want)), n
    finally:
        rng.free()
        G.lib().gasp_free(d)
        G.lib().gasp_free(d_mag)
