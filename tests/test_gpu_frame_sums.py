"""Measured frames of the LDS kernel for every workgroup size (one to sixteen
waves per replica, counts that are not powers of two among them) and packing:
the spin-derived sums equal those of the streaming kernel's separate
measurement, and the tracked state equals a fresh evaluation of the spins."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd import lattice as lat
from mcsolver_amd import workloads as W
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph

pytestmark = pytest.mark.gpu
LATTICES = {
    "ising_sq10": (1, lambda: lat.square(10, J=-1.0, ising=True)),
    "xy_sq9": (2, lambda: lat.square(9, J=-1.0)),
    "heis_honeycomb5": (3, lambda: W.honeycomb_full_tensor(5)),
    "heis_triangular8": (3, lambda: W.triangular_neel_dmi(8)),
}


def _batch(nc, x, nrep, store="f32"):
    g = compile_graph(nc, x.nbr, x.J if nc > 1 else x.J[:, :, :1], x.S, x.D, pairs=x.corr_pairs,
                      circuits=x.circuits if nc == 3 and len(x.circuits) else None, rOrb=x.rOrb,
                      rOrbCluster=x.rOrbCluster, rlink=x.rlink)
    rng = np.random.default_rng(11)
    init = []
    for _ in range(nrep):
        v = rng.normal(size=(x.n, nc))
        init.append(v[:, 0] if nc == 1 else v / np.linalg.norm(v, axis=1, keepdims=True))
    meas = L.MEAS_PAIRS | L.MEAS_RNORM | (L.MEAS_Q if nc == 3 and len(x.circuits) else 0)
    b = Batch(nc, [g], [ReplicaSpec(0, k) for k in range(nrep)], list(np.linspace(0.5, 1.5, nrep)), [0.1] * nrep, init,
              store="i8" if nc == 1 else store, meas=meas, nbins=3, nframes=6, recompute_every=5)
    b.init()
    return b


@pytest.mark.parametrize("block", [64, 128, 192, 256, 320, 512, 1024])
@pytest.mark.parametrize("name", sorted(LATTICES))
def test_frames_of_every_block_size(gpu, name, block):
    nc, mk = LATTICES[name]
    x = mk()
    for nrep in (1, 5):
        print(name, "block", block, "replicas", nrep, flush=True)
        a, r = _batch(nc, x, nrep), _batch(nc, x, nrep)
        a.run(2, 6, 2, kernel=L.KERNEL_LDS, block=block)
        r.run(2, 6, 2, kernel=L.KERNEL_STREAM)
        assert all(np.array_equal(a.replica_spins(k), r.replica_spins(k)) for k in range(nrep))
        A, R = a.accumulators(), r.accumulators()
        # sums over the spins of FP32 terms added in FP64: only the order differs
        cols = [L.A_COUNT, L.A_SIJ, L.A_Q, L.A_SIJR, L.A_LAST] + list(range(L.A_SIR, L.A_SIR + 6)) + [L.A_ER, L.A_ER2]
        np.testing.assert_allclose(A[:, cols], R[:, cols], rtol=1e-11, atol=1e-11)
        # tracked values: FP32 partial sums of about n/threads changes a sweep, at most 14 sweeps
        np.testing.assert_allclose(A, R, rtol=2e-5, atol=2e-5)
        np.testing.assert_allclose(a.bin_data(), r.bin_data(), rtol=2e-5, atol=2e-5)
        sa = a.state_data()
        a.init()  # recomputes the state from the spins
        np.testing.assert_allclose(sa[:, L.S_E:L.S_M + 3], a.state_data()[:, L.S_E:L.S_M + 3], rtol=2e-5, atol=2e-4)
        assert a.error_flag() == 0 and r.error_flag() == 0
