"""Root-path updates (tt_update_branch): branches of a tip and of an internal
node, under the root and deep, under binary and other rows, one after another,
against the full pass over the same lengths.

Every update moves a pattern's logL by the differences of a few node terms in
FP64, so after the handful here it is within a few times 1e-15 of the terms'
size of the full pass: 1e-12 relative for the total.  The branch's stored P(t)
is the one the full pass forms, bit for bit.  Of the wide alphabets 20 is not
held to this: its full pass runs on the matrix cores, which round rows in
another order."""
import numpy as np
import pytest

from test_gpu_cluster import build, close, say

pytestmark = pytest.mark.gpu

CASES = [("cherry", 4, 1), ("two-stages", 4, 255), ("two-stages", 4, 257), ("one-more", 2, 64), ("one-more", 3, 65),
         ("nested", 5, 63), ("nested", 4, 513), ("star", 5, 256), ("star", 4, 64), ("caterpillar", 4, 65),
         ("two-stages", 22, 65), ("nested", 21, 257), ("one-cluster", 21, 63)]


@pytest.mark.parametrize("shape,n,P", CASES, ids=["%s-%d-%d" % c for c in CASES])
def test_path_update(gpu_engine, shape, n, P):
    say(f"[path] {shape} n={n} P={P}")
    a, b = build(gpu_engine, shape, n, P, 11), build(gpu_engine, shape, n, P, 11)
    rng = np.random.default_rng(3)
    inner = np.isin(np.arange(a.n_nodes), a.parent[a.parent >= 0])
    depth = np.zeros(a.n_nodes, int)
    for v in range(1, a.n_nodes):
        depth[v] = depth[a.parent[v]] + 1
    nodes = [int(np.argmax(depth)), 1, a.n_nodes - 1]
    nodes += [int(v) for v in rng.choice(np.arange(1, a.n_nodes), 3)] + [int(v) for v in np.flatnonzero(inner)[1:3]]
    a.loglik()
    for i, node in enumerate(nodes + nodes[:1]):
        t = float(rng.uniform(0.0, 0.2)) if i != 1 else 0.0
        got = a.update_branch(node, t)
        b.set_branch_lengths(np.array([node], np.int32), np.array([t]))
        assert close(got, b.loglik()), (i, node, t)
        assert np.allclose(a.sequence_lh(), b.sequence_lh(), rtol=1e-12, atol=1e-12)
    # the new P(t) reaches the other passes
    assert close(a.marginal(), b.marginal())
    assert np.array_equal(a.profiles(), b.profiles())
    assert close(a.joint(), b.joint())
    assert np.array_equal(a.states(), b.states())
    a.close()
    b.close()
