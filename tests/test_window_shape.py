"""The rule that gives the smaller replica counts of methods 0, 1 and 2 to the
kernel of one replica per workgroup, where it does not depend on the device: the
counts at which its lines lie (256 CUs), and the settings that keep the method's
other kernels."""
import pytest


@pytest.fixture
def settings(engine_lib):
    yield engine_lib
    engine_lib.set_tuning(0, 0)
    engine_lib.set_conflict_filter(0)
    engine_lib.set_lattice_staging(0)
    engine_lib.set_dependence_tables(0)


# replicas per CU: 64, for method 2 52 from L = 33 on, 40 from L = 65 on; method 0 has no line from L = 32 on
@pytest.mark.parametrize("method,L,most", [(2, 8, 16384), (2, 32, 16384), (2, 33, 13312), (2, 64, 13312), (2, 65, 10240),
                                           (1, 33, 16384), (1, 64, 16384), (1, 65, 10240), (0, 31, 16384)])
def test_lines(engine_lib, method, L, most):
    assert engine_lib.get_window(method, L, most)[0] > 0
    assert engine_lib.get_window(method, L, most + 1) == (0, 0)
    assert engine_lib.get_window(method, L, 1)[0] > 0


def test_method_0_and_3(engine_lib):
    assert engine_lib.get_window(0, 32, 1_000_000)[0] > 0
    assert engine_lib.get_window(3, 32, 64) == (0, 0)
    assert engine_lib.get_window(0, 1, 64) == (0, 0) and engine_lib.get_window(5, 32, 64) == (0, 0)


def test_one_launch(engine_lib):
    """One wave per replica at L = 32: a launch has fewer than 2^32 work-items."""
    assert engine_lib.get_window(0, 32, 2**26 - 1)[0] == 1
    assert engine_lib.get_window(0, 32, 2**26) == (0, 0)


@pytest.mark.parametrize("method", [0, 1, 2])
@pytest.mark.parametrize("setting,value", [("set_tuning", (16, 2)), ("set_tuning", (16, 0)), ("set_tuning", (0, 2)),
                                           ("set_conflict_filter", (1,)), ("set_conflict_filter", (2,)),
                                           ("set_lattice_staging", (1,)), ("set_lattice_staging", (2,)),
                                           ("set_lattice_staging", (3,)), ("set_dependence_tables", (4096,))])
def test_settings_keep_the_other_kernels(settings, method, setting, value):
    G = settings
    getattr(G, setting)(*value)
    assert G.get_window(method, 32, 256) == (0, 0)
    getattr(G, setting)(*(0 for _ in value))
    assert G.get_window(method, 32, 256)[0] > 0
