"""Tempering inside a persistent launch, where each replica reads its partner
row's energy and decides the swap for itself, against one launch per swap:
ladders of every small length, long ones, rows that never meet a partner,
replicas without a ladder beside them, one to sixteen replicas per workgroup,
frames more and less often than swaps, and recomputes on swap sweeps."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd import lattice as lat
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph

pytestmark = pytest.mark.gpu


def _run(lengths, edge, pt_every, spf, rpb, recompute, persist):
    Lt = lat.square(edge, J=-1.0)
    graph = compile_graph(2, Lt.nbr, Lt.J, Lt.S, Lt.D, pairs=Lt.corr_pairs)
    reps, betas, row = [], [], 0
    for k, m in enumerate(lengths):
        for r in range(m):
            reps.append(ReplicaSpec(0, row, nrung=m, ladder=k, rung=r) if m > 1 else ReplicaSpec(0, row))
            betas.append(1 / (0.6 + 0.8 * r / m))
        row += m
    rng = np.random.default_rng(edge)
    spins = []
    for _ in reps:
        a = rng.uniform(0, 2 * np.pi, Lt.n)
        spins.append(np.stack([np.cos(a), np.sin(a)], axis=1))
    b = Batch(2, [graph], reps, betas, [0.05] * len(reps), spins, nbins=4, nframes=16, recompute_every=recompute)
    b.init()
    for frame0 in (0, 8):  # two calls: the second goes on where the first ended
        b.run(5 if frame0 == 0 else 0, 8, spf, sweep0=0 if frame0 == 0 else 5 + 8 * spf, frame0=frame0,
              pt_every=pt_every, kernel=L.KERNEL_LDS, reps_per_block=rpb, no_persist=not persist)
    assert b.error_flag() == 0
    return (np.concatenate([b.replica_spins(k).ravel() for k in range(len(reps))]), b.rung.cpu().numpy(),
            b.who.cpu().numpy(), b.pt_acc.cpu().numpy(), b.accumulators(), b.bin_data(), b.state_data()[:, :4])


@pytest.mark.parametrize("lengths,edge,rpb", [((2, 3, 5), 8, 1), ((1, 7, 1, 4), 12, 4), ((40,), 9, 16),
                                              ((3, 130), 6, 0), ((17, 2), 32, 2)])
@pytest.mark.parametrize("pt_every,spf,recompute", [(1, 1, 0), (1, 3, 4), (2, 1, 6), (3, 2, 0)])
def test_swaps_as_per_launch(gpu, lengths, edge, rpb, pt_every, spf, recompute):
    a = _run(lengths, edge, pt_every, spf, rpb, recompute, True)
    b = _run(lengths, edge, pt_every, spf, rpb, recompute, False)
    assert np.array_equal(a[0].astype(np.float32).view(np.uint32), b[0].astype(np.float32).view(np.uint32))
    for x, y in zip(a[1:4], b[1:4]):
        assert np.array_equal(x, y)
    assert pt_every == 2 or a[3].sum() > 0
    for x, y in zip(a[4:], b[4:]):
        # FP64 sums of the same FP32 changes, in another order
        np.testing.assert_allclose(x, y, rtol=1e-11, atol=1e-9)
