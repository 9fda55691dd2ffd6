"""A grid's prediction does not depend on the batch it comes in (csrc/gasp_cnn_stream.h,
L <= 64): the same bits from one call, from calls of every other size, and from a
network made for smaller batches, whatever bands and pieces these lead to."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# on 256 CUs, L = 64: bands of 8, 16 and 64 rows; 32: of 8, 16 and 32; 16: of 8 and 16, two pieces
@pytest.mark.parametrize("L,n,sizes", [(64, 300, (1, 20, 60, 150, 200)), (32, 700, (1, 9, 130, 300)), (16, 4500, (3, 500, 1000))])
def test_same_bits_in_every_batch(gpu, engine_lib, L, n, sizes):
    from oracle import cnn_oracle as K

    print(f"[cnn batches] L={L} n={n}", flush=True)
    rs = np.random.default_rng(L)
    p = (K.init_params(L).astype(np.float64) + rs.normal(0.0, 0.05, K.NPARAM)).astype(np.float32)
    frac = rs.uniform(0.05, 0.95, n)[:, None, None]
    spins = np.where(rs.random((n, L, L)) < frac, 1, -1).astype(np.int8)
    with engine_lib.Surrogate(L, n) as net:
        net.set_params(p)
        whole = net.predict(spins)
        for k in sizes:
            assert np.array_equal(net.predict(spins[:k]), whole[:k]), k
            assert np.array_equal(net.predict(spins[n - k:]), whole[n - k:]), k
    with engine_lib.Surrogate(L, n // 7) as net:
        net.set_params(p)
        assert np.array_equal(net.predict(spins), whole)
