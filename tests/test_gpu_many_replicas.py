"""Replica counts beyond the work-items of one launch (2^32): 2^24 replicas on
MT19937 streams, whose draws take 256 lanes a replica.  The streams' state is 42 GB
of device memory; first and last replicas against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_mt19937_streams_of_many_replicas(gpu, engine_lib, oracle):
    G, O = engine_lib, oracle
    L, R, seed, beta, h = 2, 1 << 24, 31, 0.4, 0.06
    print(f"[many] L={L} R={R} mt19937", flush=True)
    start = np.array([[[1, -1], [-1, -1]]], np.int32)
    idx = np.array([0, 1, R - 2, R - 1], np.int32)
    rng = G.RngState(R, seed, mt=True)
    with G.Engine(L, R, 2, rng, beta, h) as e:
        e.set_inputs(start)
        e.sweep(3)
        got = e.gather(idx)
        mag = e.magnetisation()[idx]
    rng.free()
    ref = np.concatenate([O.sweep_mt_per_replica(L, np.repeat(start, 2, 0).copy(), seed + r, 3, beta, h) for r in (0, R - 2)])
    assert np.array_equal(got.astype(np.int32).reshape(ref.shape), ref)
    assert np.array_equal(mag, ref.reshape(4, -1).sum(1).astype(np.float32) / np.float32(4))
