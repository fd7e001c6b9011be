"""The frame's sum of solid angles over circuit lists of every length class
(one, less than a wave, odd, more than a round of a workgroup), one and two
spin lengths, LDS and streaming kernels, against the same FP32 operations in
numpy; and the order in which a graph keeps its circuits."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd import lattice as lat
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph


def _lattice(edge, lengths):
    bonds = [lat.Bond(0, 0, o, [-1.0] * 3 + [0.0] * 6) for o in ((1, 0, 0), (0, 1, 0), (-1, 1, 0))]
    Lt = lat.build_lattice(edge, edge, 1, [[1, 0, 0], [0.5, np.sqrt(3) / 2, 0], [0, 0, 1]], [[0, 0, 0]], bonds, [1.0],
                           [[0, 0, 0.0]], localCircuitList=[((0, (0, 0, 0)), (0, (1, 0, 0)), (0, (0, 1, 0))),
                                                            ((0, (1, 0, 0)), (0, (1, 1, 0)), (0, (0, 1, 0)))])
    S = np.where(np.arange(Lt.n) % lengths == 0, 1.0, 1.5)
    return Lt, S


def _angles(s, S, circ):
    """The kernel's operations (FP32, no contraction) on spins s (n, 3)."""
    f = np.float32
    inv = np.sqrt(f(1) / (S.astype(f) * S.astype(f)))  # sqrt of the stored 1/S^2
    a, b, c = (s[circ[:, k]].astype(f) for k in range(3))
    ia, ib, ic = (inv[circ[:, k]] for k in range(3))
    dot = lambda x, y: x[:, 0] * y[:, 0] + x[:, 1] * y[:, 1] + x[:, 2] * y[:, 2]
    ab, bc, ca = dot(a, b) * (ia * ib), dot(b, c) * (ib * ic), dot(c, a) * (ic * ia)
    x = np.stack([b[:, 1] * c[:, 2] - b[:, 2] * c[:, 1], b[:, 2] * c[:, 0] - b[:, 0] * c[:, 2],
                  b[:, 0] * c[:, 1] - b[:, 1] * c[:, 0]], axis=1)
    re = f(1) + ab + bc + ca
    im = dot(a, x) * (ia * ib * ic)
    with np.errstate(divide="ignore", invalid="ignore"):
        w = f(2) * np.arctan(im / re)
    return np.where(np.abs(re) < f(1e-6), np.where(im > 0, f(np.pi), -f(np.pi)), w).astype(np.float64)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [L.KERNEL_LDS, L.KERNEL_STREAM])
@pytest.mark.parametrize("lengths", [1, 2])
@pytest.mark.parametrize("edge,count", [(6, 1), (6, 63), (12, 257), (12, 288), (24, 1151), (48, 4608)])
def test_charge_of_circuit_lists(gpu, edge, count, lengths, kernel):
    Lt, S = _lattice(edge, lengths)
    circ = Lt.circuits[:count]
    g = compile_graph(3, Lt.nbr, Lt.J, S, Lt.D, circuits=circ)
    rng = np.random.default_rng(count)
    v = rng.normal(size=(Lt.n, 3))
    v *= (S / np.linalg.norm(v, axis=1))[:, None]
    b = Batch(3, [g], [ReplicaSpec(0, 0)], [0.7], [0.0], [v], meas=L.MEAS_Q, nframes=1)
    b.init()
    b.run(0, 1, 1, kernel=kernel)
    want = _angles(b.replica_spins(0), S, circ).sum() / np.pi / 4
    # an angle's error: a few units in the last place of atan (numpy's and the
    # kernel's), at most 2e-6 of up to pi
    assert abs(b.accumulators()[0, L.A_Q] - want) <= count * 2e-6 / np.pi / 4


def test_order_of_circuits():
    Lt, S = _lattice(36, 1)
    g = compile_graph(3, Lt.nbr, Lt.J, S, Lt.D, circuits=Lt.circuits)
    want = g.pos[np.asarray(Lt.circuits)]
    assert g.circ.shape == want.shape and g.circ.dtype == want.dtype
    key = lambda x: x[np.lexsort(x.T[::-1])]
    for k in range(0, len(want), 512):  # within blocks only
        assert np.array_equal(key(g.circ[k:k + 512]), key(want[k:k + 512]))
    col = np.searchsorted(g.col_ptr, g.circ, side="right")
    same = (np.diff(col, axis=0) == 0).all(axis=1)
    assert same.mean() > 0.97  # runs of one kind
    assert (np.diff(g.circ[:, 0])[same] > 0).all()
