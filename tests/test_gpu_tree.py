"""The all-levels octree build against the oracle where its parts meet: sets
of one wave chunk and of one wave tile give or take a particle, buckets of one
particle and larger than the set, keys shared by more particles than a bucket
holds, a chain of single-child levels (far more internal nodes than the tables
first hold), and the last key cell.  Node set, ranges, links and buckets are
equal, from the full sort and from a top-bits one, and so are the nodes'
moments bit for bit, massless particles, leaves and subtrees included."""
import numpy as np
import pytest

from oracle import oracle as O
from paratreet_amd import ics
from tests.helpers import bits, oracle_node_data, rel_err

pytestmark = pytest.mark.gpu


def _chain(n):
    """Pairs of neighbours in nested cells: every level has one internal node
    and the deepest cells hold several particles with the same key."""
    rng = np.random.default_rng(9)
    scale = 2.0 ** -rng.integers(0, 20, n)
    pos = rng.uniform(0.5, 1.0, (n, 3)) * scale[:, None]
    pos[0] = 0.0
    return pos


def _shared_keys(n):
    rng = np.random.default_rng(11)
    return rng.integers(0, 3, (n, 3)).astype(np.float64)


def _corner(n):
    pos = np.random.default_rng(12).uniform(0.0, 1.0, (n, 3))
    pos[n // 2:] = 1.0
    return pos


CASES = [("plummer", 1, 12), ("plummer", 12, 12), ("plummer", 13, 12), ("plummer", 63, 1),
         ("plummer", 64, 7), ("plummer", 65, 64), ("plummer", 255, 12), ("plummer", 257, 3),
         ("plummer", 5000, 64), ("plummer", 5000, 100), ("plummer", 70001, 8), ("chain", 700, 1),
         ("chain", 3000, 16), ("shared", 900, 12), ("corner", 400, 6)]


@pytest.mark.parametrize("kind,n,bucket", CASES, ids=["%s-%d-B%d" % c for c in CASES])
def test_tree_matches_oracle(kind, n, bucket):
    from paratreet_amd.gravity import Configuration, Driver
    pos = {"plummer": lambda: ics.plummer(n, seed=70 + bucket)[0], "chain": lambda: _chain(n),
           "shared": lambda: _shared_keys(n), "corner": lambda: _corner(n)}[kind]()
    rng = np.random.default_rng(n + bucket)
    m, e = rng.uniform(0.5, 1.5, n) / n, rng.uniform(0.005, 0.02, n)
    weight = m.copy()
    if n > 60:
        m[pos[:, 0] > np.quantile(pos[:, 0], 0.7)] = 0.0
    P = O.Pipeline(pos, m, e, bucket=bucket, theta=0.7)
    d = Driver(Configuration(max_particles_per_leaf=bucket))
    d.load(pos, m, e)
    onodes = {int(k): i for i, k in enumerate(P.nodes["key"])}
    # the stage calls (full sort), then two evaluations (the second sorts the
    # top bits only)
    for attempt in range(3):
        if attempt == 0:
            d.remake_universe()
            d.assign_keys()
            d.build_tree()
        else:
            d.compute_forces(theta=0.7, precision=0)
        g = d.nodes()
        at = np.array([onodes[int(k)] for k in g["key"]])
        assert len(at) == len(P.nodes) and len(np.unique(at)) == len(at)
        for f in ("type", "depth", "begin", "count"):
            assert np.array_equal(g[f], P.nodes[f][at]), f
        inner = np.nonzero(g["type"] == 2)[0]
        for c in range(8):
            ch = g["first_child"][inner] + c
            assert np.array_equal(g["key"][ch], g["key"][inner] * np.uint64(8) + np.uint64(c))
            assert np.array_equal(g["parent"][ch], inner)
        assert np.all(g["first_child"][g["type"] != 2] == -1) and g["parent"][0] == -1
        assert np.array_equal(g["key"][d.buckets()], P.nodes["key"][O.buckets(P.nodes)])
        sk, perm = d.sorted()
        assert np.array_equal(sk, P.sorted_keys)
        assert np.array_equal(perm.astype(np.int64), P.perm.astype(np.int64))
        assert np.array_equal(bits(d.node_data()), bits(oracle_node_data(P)[at]))
    P = O.Pipeline(pos, weight, e, bucket=bucket, theta=0.7)
    d.load(pos, weight, e)
    cnt = d.compute_forces(theta=0.7, precision=0)
    oacc, _, ocnt = P.gravity_unsorted()
    assert tuple(int(v) for v in cnt) == tuple(int(v) for v in ocnt)
    if n > 1:
        acc, _ = d.accelerations()
        moved = np.linalg.norm(oacc, axis=1) > 0
        assert rel_err(acc[moved], oacc[moved]).max() <= 1e-12
    d.close()
