"""A streaming batch larger than the last-level cache is taken in groups of
replicas, each through all the sweeps of the call: every replica's spins,
sums and frames as when it runs in a small batch."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd import lattice as lat
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph

pytestmark = pytest.mark.gpu


def test_groups_of_a_large_batch(gpu):
    Lt = lat.cubic(64, J=-1.0)
    graphs = [compile_graph(3, Lt.nbr, Lt.J, Lt.S, Lt.D, pairs=Lt.corr_pairs) for _ in range(2)]
    graphs[1].npat = 0  # neighbours from the link table: a second link mode
    v = np.random.default_rng(8).normal(size=(Lt.n, 3))
    v /= np.linalg.norm(v, axis=1, keepdims=True)

    def run(first, count, look):
        ks = range(first, first + count)
        b = Batch(3, graphs, [ReplicaSpec(int(k >= 60), k - first) for k in ks], [0.6 + 0.01 * k for k in ks],
                  [0.02] * count, [v] * count, nbins=4, nframes=4, recompute_every=3, serial_base=first)
        b.init()
        b.run(1, 4, 1, kernel=L.KERNEL_STREAM)
        assert b.error_flag() == 0
        return {k: b.replica_spins(k - first) for k in look}, b.accumulators(), b.bin_data(), b.state_data()

    # 90 replicas of 3 MiB: two groups, the second of both link modes
    look = [0, 1, 43, 44, 45, 46, 59, 60, 89]
    every = run(0, 90, look)
    for first, count in ((0, 2), (43, 4), (59, 2), (89, 1)):
        alone = run(first, count, range(first, first + count))
        for k in range(first, first + count):
            assert np.array_equal(every[0][k], alone[0][k]), k
            for x, y in zip(every[1:], alone[1:]):
                # FP64 sums whose workgroups may be added in another order
                np.testing.assert_allclose(x[k], y[k - first], rtol=1e-11, atol=1e-9)
