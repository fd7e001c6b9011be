"""Sweeps of graphs with every link count, coupling kind and class count,
against the CPU checker, bit for bit: the kernels have their own code for the
common link counts (4, 6 and 9) and read other graphs' links four at a time,
with one coupling or site class in registers and several in tables."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph
from oracle import mcref

pytestmark = pytest.mark.gpu
SEED = 0x5EED2026


def _ring(nc, n, z, uniform, classes):
    """A ring of n sites, links to the first z of the neighbours +1, -1, +2, -2, ...
    (an odd z: directed)."""
    step = np.array([(k // 2 + 1) * (1 if k % 2 == 0 else -1) for k in range(z)])
    nbr = (np.arange(n)[:, None] + step[None, :]) % n
    rng = np.random.default_rng(7 * z + n)
    J = np.zeros((n, z, 9))
    per = np.tile(rng.uniform(-1, 1, (1, 9)), (z, 1)) if uniform else rng.uniform(-1, 1, (z, 9))
    J[:] = per[None]
    S = np.where(np.arange(n) % classes == 0, 1.0, 1.5)
    D = np.zeros((n, 3))
    if classes > 1:
        D[1::2] = (0.1, -0.05, 0.2)
    return nbr, J if nc > 1 else J[:, :, :1], S, D


@pytest.mark.parametrize("patterns", [True, False])
@pytest.mark.parametrize("kernel", [L.KERNEL_LDS, L.KERNEL_STREAM])
@pytest.mark.parametrize("classes", [1, 2])
@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("nc,store", [(1, "i8"), (2, "f32"), (3, "f32")])
def test_link_counts_bitexact(gpu, nc, store, uniform, classes, kernel, patterns):
    for z, n in ((1, 40), (2, 41), (3, 64), (4, 90), (5, 77), (6, 130), (8, 144), (9, 102), (11, 120)):
        print("links", z, "sites", n, flush=True)
        nbr, J, S, D = _ring(nc, n, z, uniform, classes)
        g = compile_graph(nc, nbr, J, S, D)
        # an Ising coupling includes the target's spin length
        assert g.npat > 0 and (g.ucid >= 0) == ((uniform or z == 1) and (nc > 1 or classes == 1))
        if not patterns:
            g.npat = 0  # neighbours from the link table
        rng = np.random.default_rng(3)
        betas, h = [0.4, 1.7], 0.15
        init = []
        for _ in betas:
            if nc == 1:
                init.append(np.where(rng.random(n) < 0.5, 1.0, -1.0))
            else:
                v = rng.normal(size=(n, nc))
                v *= (np.abs(S) / np.linalg.norm(v, axis=1))[:, None]
                init.append(v.astype(np.float32).astype(np.float64))
        b = Batch(nc, [g], [ReplicaSpec(0, 0), ReplicaSpec(0, 1)], betas, [h, h], init, store=store, seed=SEED)
        b.init()
        b.sweeps(0, 5, kernel=kernel)
        got = np.stack([b.replica_spins(k).T.astype(np.float32) for k in range(2)])
        ref = np.ascontiguousarray(np.stack([np.atleast_2d(s.T) for s in init]).astype(np.float32))
        mcref.cb_sweeps(nc, {"f32": 0, "i8": 2}[store], nbr, J, S, D, g.colour, betas, [h, h],
                        np.arange(2, dtype=np.uint32), SEED, 0, 5, ref)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (z, n)


def test_streaming_batch_of_every_link_mode(gpu):
    """One streaming batch whose replicas need every link mode of the pass
    (patterns or link table, one coupling or several): each replica's spins
    as when it runs alone."""
    def graphs():
        out = []
        for uniform in (False, True):
            for patterns in (True, False):
                nbr, J, S, D = _ring(3, 90, 4, uniform, 1)
                g = compile_graph(3, nbr, J, S, D)
                if not patterns:
                    g.npat = 0
                out.append(g)
        return out

    def run(gs, serial):
        v = np.random.default_rng(1).normal(size=(90, 3))
        v /= np.linalg.norm(v, axis=1, keepdims=True)
        b = Batch(3, gs, [ReplicaSpec(k, k) for k in range(len(gs))], [0.9] * len(gs), [0.1] * len(gs), [v] * len(gs),
                  seed=SEED, serial_base=serial)
        b.init()
        b.run(2, 4, 1, kernel=L.KERNEL_STREAM)
        return [b.replica_spins(k) for k in range(len(gs))], b.accumulators()

    every, acc = run(graphs()[::-1], 0)
    for k, g in enumerate(graphs()[::-1]):
        alone, a1 = run([g], k)
        assert np.array_equal(every[k], alone[0]), k
        np.testing.assert_allclose(acc[k], a1[0], rtol=1e-12)
