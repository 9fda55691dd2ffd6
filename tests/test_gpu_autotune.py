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
