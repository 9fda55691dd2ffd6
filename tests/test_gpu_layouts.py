"""Kernels that read and write the native layouts: grids in and out, the packed record body, gathered replicas and
the largest cluster, on each layout and at the sizes where a word, a wave or a row ends.  All values are whole
numbers and equal exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (method, explicit launch shape): an explicit shape keeps the method's own layout (bytes, bits, planes), which the
# automatic choice for few replicas replaces by bits; method 3 has planes
LAYOUTS = [(0, (8, 1)), (1, (8, 1)), (2, (8, 0)), (1, None), (3, None)]


def _patterns(R, L, seed):
    rng = np.random.default_rng(seed)
    g = np.where(rng.random((R, L, L)) < rng.uniform(0.02, 0.98, (R, 1, 1)), 1, -1).astype(np.int32)
    x, y = np.meshgrid(np.arange(L), np.arange(L), indexing="ij")
    for r, p in enumerate([x >= 0, x < 0, x % 2 == 0, y % 2 == 0, (x + y) % 2 == 0, (x == 0) | (y == L - 1),
                           (x + 2 * y) % 5 == 0, (y == 0) | (y == L - 1) | (x == L // 2)][:R]):
        g[r] = np.where(p, 1, -1)
    return g


@pytest.mark.parametrize("method,shape", LAYOUTS)
@pytest.mark.parametrize("L,R", [(2, 70), (5, 33), (8, 65), (16, 97), (31, 40), (33, 9), (64, 131), (75, 35), (96, 3)])
def test_layout_kernels(gpu, engine_lib, oracle, method, shape, L, R):
    G, lib = engine_lib, oracle.lib()
    print(f"[layouts] method={method} shape={shape} L={L} R={R}", flush=True)
    g = _patterns(R, L, 100 * L + R)
    rng = G.RngState(R, 1)
    try:
        if shape:
            G.set_tuning(*shape)
        with G.Engine(L, R, method, rng, 0.3, 0.0) as e:
            e.set_grids(g)
            assert np.array_equal(e.get_grids(), g)
            exp = np.packbits((g.reshape(-1) > 0).astype(np.uint8), bitorder="little")
            assert np.array_equal(e.gridstates(), exp)
            idx = np.array([R - 1, 0, R // 2, 0], dtype=np.int32)
            assert np.array_equal(e.gather(idx), g[idx].astype(np.int8))
            for spin in (1, -1):
                ref = [lib.orc_largest_cluster(L, g[r].reshape(-1), spin) for r in range(R)]
                assert np.array_equal(e.largest_cluster(spin), np.array(ref, dtype=np.float32)), spin
            # inputs shared by consecutive replicas
            n = next(k for k in range(R // 2, 0, -1) if R % k == 0)
            e.set_inputs(g[:n])
            assert np.array_equal(e.get_grids(), np.repeat(g[:n], R // n, axis=0))
    finally:
        G.set_tuning(0, 0)
        rng.free()


@pytest.mark.parametrize("L", [162, 165])
def test_largest_cluster_workspace(gpu, engine_lib, oracle, L):
    """On either side of the largest lattice whose labels fit in LDS."""
    G, lib = engine_lib, oracle.lib()
    R = 9
    print(f"[cluster] L={L}", flush=True)
    g = _patterns(R, L, L)
    rng = G.RngState(R, 1)
    with G.Engine(L, R, 1, rng, 0.3, 0.0) as e:
        e.set_grids(g)
        for spin in (1, -1):
            ref = [lib.orc_largest_cluster(L, g[r].reshape(-1), spin) for r in range(R)]
            assert np.array_equal(e.largest_cluster(spin), np.array(ref, dtype=np.float32)), spin
    rng.free()


@pytest.mark.parametrize("R", [1, 64, 1023, 1025, 3000])
def test_counts_of_the_check(gpu, engine_lib, R):
    """The check's counts, summed by one workgroup of 1024 lanes, against the magnetisations and fates."""
    G = engine_lib
    L = 8
    print(f"[counts] R={R}", flush=True)
    rng = G.RngState(R, 3)
    with G.Engine(L, R, 2, rng, 0.3, 0.0) as e:
        e.set_grids(_patterns(R, L, R))
        e.sweep(1, G.CHECK_COUNT, -0.2, 0.2)
        m = e.magnetisation().astype(np.float64)
        assert list(e.counts()) == [int((m > 0.2).sum()), 0, 0, 0][:len(e.counts())]
        e.set_fates(np.full(R, -1, dtype=np.int32))
        for _ in range(2):
            e.sweep(1, G.CHECK_FATES, -0.2, 0.2)
            f = e.fates()
            assert list(e.counts()) == [0, int((f == 0).sum()), int((f == 1).sum()), 0][:len(e.counts())]
    rng.free()
