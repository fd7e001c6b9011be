"""Ising thresholds from LDS and, where they do not fit beside the spins or a
table is too long, from global memory: bit for bit the CPU checker's sweeps,
with replicas of several rows in a workgroup and table lengths from a few
entries to more than LDS holds of them."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd import lattice as lat
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph, exact_ising_table
from oracle import mcref

pytestmark = pytest.mark.gpu
SEED = 0x5EED2026


@pytest.mark.parametrize("rpb,block", [(1, 0), (4, 0), (16, 1024)])
@pytest.mark.parametrize("edge", [6, 30])
@pytest.mark.parametrize("J,h,short", [(-1.0, 0.0, True), (-1.0, 0.25, True), (-100.0, 0.0078125, False)])
def test_thresholds_bitexact(gpu, J, h, short, edge, rpb, block):
    Lt = lat.square(edge, J=J, ising=True)
    g = compile_graph(1, Lt.nbr, Lt.J[:, :, :1], Lt.S, Lt.D)
    n, T = Lt.n, 16
    betas = list(np.linspace(0.2, 1.2, T) / abs(J))
    tab, _ = exact_ising_table([g], betas, [h] * T)
    assert (tab.shape[1] <= 1024) == short
    rng = np.random.default_rng(edge)
    init = [np.where(rng.random(n) < 0.5, 1.0, -1.0) for _ in betas]
    b = Batch(1, [g], [ReplicaSpec(0, k) for k in range(T)], betas, [h] * T, init, store="i8", seed=SEED)
    b.init()
    b.run(6, 0, 1, kernel=L.KERNEL_LDS, reps_per_block=rpb, block=block)
    got = np.stack([b.replica_spins(k).T.astype(np.float32) for k in range(T)]).reshape(T, -1)
    ref = np.ascontiguousarray(np.stack([s[None] for s in init]).astype(np.float32))
    mcref.cb_sweeps(1, 2, Lt.nbr, Lt.J[:, :, :1], Lt.S, Lt.D, g.colour, betas, [h] * T, np.arange(T, dtype=np.uint32),
                    SEED, 0, 6, ref, ising_table=b.ising_table())
    assert np.array_equal(got, ref.reshape(T, -1))
