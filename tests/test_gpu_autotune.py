"""gasp_autotune beside the kernel of one replica per workgroup, which no (slots,
waves) names: what it returns belongs to the shape that it returns, and it bars
that kernel from later engines only where it has timed it and found it slower."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BETA, H = 0.5, 0.05


@pytest.fixture
def settings(engine_lib):
    yield engine_lib
    engine_lib.set_tuning(0, 0)
    engine_lib.set_conflict_filter(0)
    engine_lib.set_lattice_staging(0)
    engine_lib.set_dependence_tables(0)


# settings under which the tuner's engines cannot run the kernel; a shape of its own for each, as results are kept
@pytest.mark.parametrize("setting,value,method,L,R", [("set_lattice_staging", 3, 2, 18, 130),
                                                      ("set_dependence_tables", 4096, 0, 34, 20),
                                                      ("set_conflict_filter", 2, 2, 20, 140),
                                                      ("set_conflict_filter", 1, 1, 22, 150)])
def test_not_timed_is_not_slower(gpu, settings, setting, value, method, L, R):
    G = settings
    print(f"[autotune] {setting}({value}) method={method} L={L} R={R}", flush=True)
    auto = G.get_window(method, L, R)
    assert auto[0] > 0
    getattr(G, setting)(value)
    G.autotune(method, L, R, 1, BETA, H)
    assert G.get_window(method, L, R) == (0, 0)
    getattr(G, setting)(0)
    assert G.get_window(method, L, R) == auto


def test_a_batch_leaves_the_automatic_choice(gpu, settings):
    from gpu_2dising_amd.batched import Batch

    G = settings
    groups = [(24, 192, 2), (36, 48, 0)]
    print("[autotune] after a batch", flush=True)
    auto = [G.get_window(m, L, R) for L, R, m in groups]
    Batch(groups, chk=2, probe_sweeps=1).close()
    assert [G.get_window(m, L, R) for L, R, m in groups] == auto
    assert all(a[0] > 0 for a in auto)


def test_what_it_returns_is_the_shapes_own(gpu, settings):
    """64 replicas of 64 x 64: one per workgroup is several times faster than the best of the shapes, so that its rate
    could not be taken for the shape's."""
    G = settings
    method, L, R = 2, 64, 64
    print("[autotune] returned rate", flush=True)
    s, w, k, rate = G.autotune(method, L, R, 20, BETA, H, 20)
    assert G.get_window(method, L, R)[0] > 0

    def timed(shape):
        G.set_tuning(*shape)
        rng = G.RngState(R, 3)
        with G.Engine(L, R, method, rng, BETA, H) as e:
            window = e.window()[0] > 0
            e.set_grids(-np.ones((R, L, L), np.int32))
            e.sweep(20)
            e.sync()
            ms = e.kernel_ms()
            e.sweep(20)
            e.sync()
            ms = e.kernel_ms() - ms
        rng.free()
        G.set_tuning(0, 0)
        return window, 20 * L * L * R / (ms * 1e-3)

    (own_window, own), (auto_window, auto) = timed((s, w)), timed((0, 0))
    print(f"returned {rate:.3g}, shape {own:.3g}, automatic {auto:.3g}", flush=True)
    assert not own_window and auto_window
    assert abs(np.log(rate / own)) < abs(np.log(rate / auto))


def test_refined_batch_keeps_the_kernels_it_timed(gpu, settings, oracle):
    from gpu_2dising_amd.batched import Batch

    G = settings
    groups = [(16, 160, 2), (32, 64, 2), (40, 20, 0)]
    print("[autotune] refined batch on automatic settings", flush=True)
    b = Batch(groups, chk=4, probe_sweeps=2, refine=True, refine_replays=1, conflict_filter=0, lattice_staging=0,
              dependence_tables=0)
    try:
        auto = [G.get_window(m, L, R) for L, R, m in groups]
        assert any(a[0] for a in auto)
        for g, a in zip(b.groups, auto):
            assert g.engine.window() == a, g.L
            assert (g.slots == 0 and g.waves == 0) == (a[0] > 0)
        b.graph.launch(2)
        for g in b.groups:
            idx = np.arange(g.R)
            grids = g.start.copy()
            oracle.sweep_philox_replicas(g.L, grids, idx, g.seed, 0, 2 * b.chk * g.L * g.L, g.beta, g.h)
            assert np.array_equal(g.engine.get_grids(), grids), g.L
    finally:
        b.close()
