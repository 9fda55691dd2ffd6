"""Which form of the one-replica-per-workgroup kernel the automatic launch shape
takes on a device of 256 CUs with 160 KB of LDS: the shapes of test_gpu_window.py
(all kernels give the same trajectories, so their results do not tell), and the
first lattices that keep bits and a table (L = 202 still has a dword per site)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (method, L, R): (waves per replica, table entries)
SHAPES = {(2, 2, 70): (1, 0), (1, 3, 65): (1, 0), (2, 5, 33): (1, 0), (2, 16, 300): (1, 0), (1, 17, 100): (1, 0),
          (2, 24, 64): (1, 0), (2, 32, 100): (2, 0), (0, 45, 20): (2, 0), (1, 64, 9): (8, 0), (2, 75, 5): (8, 0),
          (2, 128, 3): (8, 0), (0, 201, 2): (8, 0), (0, 202, 2): (8, 0), (0, 203, 2): (8, 32768), (2, 256, 3): (8, 32768),
          (0, 300, 2): (8, 32768), (2, 64, 1024): (4, 0), (1, 64, 2048): (2, 0), (0, 200, 700): (8, 8192),
          (2, 16, 70): (1, 0), (1, 33, 40): (2, 0), (0, 64, 12): (8, 0), (2, 210, 3): (8, 32768), (2, 2, 20): (1, 0),
          (2, 64, 20): (8, 0), (1, 32, 90): (2, 0), (2, 32, 90): (2, 0), (2, 2, 3): (1, 0)}


@pytest.mark.parametrize("mt", [False, True])
@pytest.mark.parametrize("method,L,R", sorted(SHAPES))
def test_kernel(gpu, engine_lib, method, L, R, mt):
    G = engine_lib
    print(f"[window shape] method={method} L={L} R={R} mt={mt}", flush=True)
    rng = G.RngState(R, 1, mt=mt)
    with G.Engine(L, R, method, rng, 0.3, 0.07) as e:
        assert e.window() == SHAPES[method, L, R]
    rng.free()
    assert G.get_window(method, L, R) == SHAPES[method, L, R]


@pytest.mark.parametrize("mt", [False, True])
@pytest.mark.parametrize("L", [202, 203])
def test_both_sides_of_the_table(gpu, engine_lib, oracle, L, mt):
    G, O = engine_lib, oracle
    R = 2
    print(f"[window table] L={L} mt={mt}", flush=True)
    rs = np.random.default_rng(L)
    g0 = np.where(rs.random((R, L, L)) < 0.5, 1, -1).astype(np.int32)
    rng = G.RngState(R, 3, mt=mt)
    with G.Engine(L, R, 0, rng, 0.3, 0.07) as e:
        assert (e.window()[1] > 0) == (L == 203)
        e.set_grids(g0)
        e.sweep(1)
        e.sweep(2)
        got = e.get_grids()
    rng.free()
    ref = O.sweep_mt_per_replica(L, g0.copy(), 3, 3, 0.3, 0.07) if mt else O.sweep_philox(L, g0.copy(), 3, 0, 3 * L * L, 0.3, 0.07)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("method,L,R", [(2, 32, 100), (1, 64, 9), (0, 45, 20)])
@pytest.mark.parametrize("shape", [(0, 0), (16, 2)])
def test_run_statistics(gpu, engine_lib, shape, method, L, R):
    """A driver run reports the shape of the kernel that ran."""
    G = engine_lib
    print(f"[window stats] method={method} L={L} R={R} shape={shape}", flush=True)
    rng = G.RngState(R, 1)
    G.set_tuning(*shape)
    try:
        waves = G.get_window(method, L, R)[0]
        want = (64 * waves, waves) if waves else G.get_tuning(method, L, R)
        assert (waves > 0) == (shape == (0, 0))
        st = G.run_driver(L, -np.ones((R, L, L), np.int32), beta=0.3, h=0.07, rng=rng, method=method, tot_nsweeps=4,
                          mag_output_int=2, grid_output_int=4, itask=0, dn_thr=-0.9, up_thr=0.9, ninputs=1,
                          outfunc=lambda *a: 0)["stats"]
    finally:
        G.set_tuning(0, 0)
        rng.free()
    assert (st.slots_per_replica, st.waves_per_group) == want and st.method == method
