"""Wolff clusters on every path of the cluster kernel, against the CPU checker
bit for bit: link patterns, link table and more than 256 couplings; levels
that are longer than the frontier kept in LDS; couplings beyond the table of
r.J.r; members as LDS bits and (graphs too large for that) as stamps."""
import numpy as np
import pytest

from mcsolver_amd import _lib as L
from mcsolver_amd import lattice as lat
from mcsolver_amd.engine import Batch, ReplicaSpec, compile_graph
from oracle import mcref

pytestmark = pytest.mark.gpu
SEED = 0x5EED2026


def _check(nc, Lt, J, beta, h, ncl, links, order):
    nbr, S, D = Lt.nbr, Lt.S, Lt.D
    n = nbr.shape[0]
    g = compile_graph(nc, nbr, J if nc > 1 else J[:, :, :1], S, D)
    assert (g.lcid is not None) == (links == "wide")
    if links == "table":
        g.npat = 0
    rng = np.random.default_rng(n + nc)
    if nc == 1:
        sp = np.ones(n) if order else np.where(rng.random(n) < 0.5, 1.0, -1.0)
    else:
        sp = np.zeros((n, nc)) if order else rng.normal(size=(n, nc))
        sp[:, 0] += 2.0 if order else 0.0
        sp = (sp * (np.abs(S) / np.linalg.norm(sp, axis=1))[:, None]).astype(np.float32).astype(np.float64)
    b = Batch(nc, [g], [ReplicaSpec(0, 0)], [beta], [h], [sp], store="i8" if nc == 1 else "f32", seed=SEED, wolff=True)
    b.init()
    b.sweeps(0, 2, algorithm=L.WOLFF, clusters_per_sweep=ncl)
    ref = np.ascontiguousarray(np.atleast_2d(sp.T).astype(np.float32))
    sizes = mcref.cb_wolff(nc, 0 if nc > 1 else 2, nbr, J if nc > 1 else J[:, :, :1], S, D, g.colour, beta, h, 0, SEED,
                           0, 2 * ncl, ref)
    print("cluster sizes", sizes, flush=True)
    got = b.replica_spins(0).T.astype(np.float32)
    assert np.array_equal(np.atleast_2d(got).view(np.uint32), ref.view(np.uint32))
    assert b.state_data()[0, L.S_TRY] == sizes.sum()
    return sizes


@pytest.mark.parametrize("links", ["patterns", "table", "wide"])
@pytest.mark.parametrize("nc", [1, 2, 3])
def test_levels_longer_than_the_frontier(gpu, nc, links):
    Lt = lat.cubic(30, J=-1.0, ising=nc == 1)
    J = Lt.J.copy()
    if links == "wide":
        J[:, :, 0] *= np.random.default_rng(4).uniform(0.9, 1.1, 6)[None, :] * (1 + (np.arange(Lt.n) % 97) / 970)[:, None]
    for h in (0.0, 0.02):  # the second evaluates the acceptance energy
        sizes = _check(nc, Lt, J, 3.0, h, 3, links, True)
        assert sizes.max() > 20000  # a compact cluster: about 2 L^2 sites in the longest levels


def test_more_couplings_than_the_table(gpu):
    Lt = lat.square(12, J=-1.0)
    for nc in (2, 3):
        J = np.random.default_rng(nc).uniform(-1.5, 0.0, (Lt.n, 4, 9))
        _check(nc, Lt, J, 1.0, 0.0, 12, "wide", False)
        _check(nc, Lt, J, 1.0, 0.1, 12, "wide", False)


def test_members_as_stamps(gpu):
    """1072 x 1072 sites: their bits do not fit into LDS."""
    Lt = lat.square(1072, J=-1.0, ising=True)
    _check(1, Lt, Lt.J, 0.45, 0.0, 3, "patterns", False)
    _check(1, Lt, Lt.J, 0.6, 0.0, 2, "patterns", True)
