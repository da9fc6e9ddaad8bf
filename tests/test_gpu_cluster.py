"""Clustered passes (tt_cluster.hip) at the sizes where they can go wrong:
trees of one cluster, of one row more than a cluster, a chain (a caterpillar,
all one cluster) and one with trees along it, a star and nested polytomies; pattern counts around a wave and
around a workgroup's four waves.

The one-launch pass runs the same per-(node, pattern) arithmetic, so profiles,
rows, states, joint messages and argmax rows must be equal bit for bit and
log-likelihoods to the order of their sums (1e-12 relative); a batch of all
shapes equals its trees' own passes; one case per alphabet is held to the FP64
oracle at the parity tests' 1e-7."""
import sys

import numpy as np
import pytest

from treetime_amd import synth
from treetime_amd.engine import DeviceTree, batch_run
from treetime_amd.gtr import GTR

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def tree_of(shape, rng):
    """(parent, branch length), preorder numbering."""
    if shape == "cherry":
        return np.array([-1, 0, 0], np.int32), np.array([0, .1, .2])
    if shape == "star":
        return np.array([-1] + [0] * 90, np.int32), np.r_[0, rng.uniform(.01, .1, 90)]
    if shape in ("caterpillar", "ladder"):  # 120 rows in a chain, one cluster; 300 in two
        par, bl = [-1], [0.0]
        v = 0
        for _ in range(119 if shape == "caterpillar" else 299):
            par += [v, v]
            bl += list(rng.uniform(.01, .05, 2))
            v = len(par) - 1
        par += [v, v]
        bl += [.02, .03]
        return np.array(par, np.int32), np.array(bl)
    if shape == "comb":  # 90 rows in a chain, a cherry or a larger tree on every other one
        par, bl, v = [-1], [0.0], 0
        for k in range(90):
            par += [v, v]
            bl += list(rng.uniform(.01, .05, 2))
            v, open_ = len(par) - 1, [len(par) - 2]
            for _ in range([1, 0, 5, 0][k % 4]):
                x = open_.pop(rng.integers(len(open_)))
                par += [x, x]
                bl += list(rng.uniform(.01, .05, 2))
                open_ += [len(par) - 2, len(par) - 1]
        par, bl, _ = synth.preorder_renumber(np.array(par + [v, v], np.int32), np.array(bl + [.02, .03]))
        return par, bl
    tips = {"one-cluster": 17, "one-more": 18, "two-stages": 90, "nested": 150}[shape]
    par, bl = synth.kingman_tree(tips, 0.1, rng)
    if shape == "nested":  # collapse a third of the inner nodes
        n = len(par)
        gone = np.zeros(n, bool)
        gone[rng.choice(np.arange(tips, n - 1), (tips - 2) // 3, replace=False)] = True
        for v in range(n - 1):
            while gone[par[v]]:
                bl[v] += bl[par[v]]
                par[v] = par[par[v]]
        idx = np.cumsum(~gone) - 1
        par = np.where(par[~gone] >= 0, idx[par[~gone]], -1).astype(np.int32)
        bl = bl[~gone]
    par, bl, _ = synth.preorder_renumber(par, bl)
    return par, bl


def build(engine, shape, n, P, seed):
    rng = np.random.default_rng(seed)
    parent, bl = tree_of(shape, rng)
    pi, W = synth.random_gtr(n, rng, 5.0, 0.5)
    np.fill_diagonal(W, 0.0)
    eig, v, vi = GTR._eig_single_site(W, pi)
    tips = len(parent) - len(np.unique(parent[parent >= 0]))
    lut = np.zeros((n + 2, n), np.float32)
    lut[:n] = np.eye(n)
    lut[n] = 1.0
    lut[n + 1, :2] = 1.0
    base = rng.integers(0, n, P)[None].repeat(tips, 0)
    codes = np.where(rng.random((tips, P)) < 0.2, rng.integers(0, n + 2, (tips, P)), base).astype(np.uint8)
    return DeviceTree(engine, parent, np.maximum(bl, 1e-6), codes, lut, rng.integers(1, 9, P).astype(float), pi, eig, v,
                      vi, 1.0)


def close(a, b, rtol=1e-12):
    return abs(a - b) <= rtol * abs(b)


CASES = [("cherry", 4, 1), ("one-cluster", 4, 63), ("one-more", 4, 64), ("one-more", 5, 65), ("two-stages", 4, 255),
         ("two-stages", 2, 256), ("two-stages", 3, 257), ("nested", 4, 65), ("nested", 5, 257), ("nested", 2, 63),
         ("star", 4, 65), ("star", 5, 1), ("caterpillar", 4, 64), ("caterpillar", 5, 65), ("caterpillar", 3, 1),
         ("comb", 4, 65), ("comb", 5, 64), ("comb", 2, 130), ("ladder", 4, 64), ("ladder", 5, 1)]


@pytest.mark.parametrize("shape,n,P", CASES, ids=["%s-%d-%d" % c for c in CASES])
def test_clustered_equals_one_launch(gpu_engine, monkeypatch, shape, n, P):
    say(f"[cluster] {shape} n={n} P={P}")
    monkeypatch.setenv("TT_TILE", "0")
    cl = build(gpu_engine, shape, n, P, 5)
    monkeypatch.setenv("TT_TILE", "1")
    one = build(gpu_engine, shape, n, P, 5)
    assert cl.pass_shape()[0] == 0 and one.pass_shape()[0] > 0
    inner = np.isin(np.arange(cl.n_nodes), cl.parent[cl.parent >= 0])
    for tips in (False, True, False):
        assert close(cl.marginal(reconstruct_tips=tips), one.marginal(reconstruct_tips=tips))
        assert np.allclose(cl.sequence_lh(), one.sequence_lh(), rtol=1e-12, atol=1e-13)
        assert np.array_equal(cl.profiles(), one.profiles())
        assert np.array_equal(cl.profiles(1), one.profiles(1))
        assert np.array_equal(cl.states(), one.states())
        assert close(cl.joint(reconstruct_tips=tips), one.joint(reconstruct_tips=tips))
        assert np.allclose(cl.sequence_lh(), one.sequence_lh(), rtol=1e-12, atol=1e-13)
        assert np.array_equal(cl.states(), one.states())
        rows = (cl.parent >= 0) & (inner | tips)
        (la, ca), (lb, cb) = cl.joint_debug(), one.joint_debug()
        assert np.array_equal(la, lb) and np.array_equal(ca[rows], cb[rows])
        given = (np.arange(P) % n).astype(np.uint8)
        assert close(cl.joint_from_root(given, reconstruct_tips=tips), one.joint_from_root(given, reconstruct_tips=tips))
        assert np.array_equal(cl.states(), one.states())
    assert close(cl.loglik(), one.loglik())
    # kept normalisers: a root-path update after a clustered pass
    node = cl.n_nodes - 1
    assert close(cl.update_branch(node, 0.04), one.update_branch(node, 0.04))
    one.update_branch(1, 0.03)
    assert close(cl.update_branch(1, 0.03), one.loglik(), 1e-11)
    cl.close()
    one.close()


@pytest.mark.parametrize("n", [4, 5])
def test_clustered_batch_of_shapes(gpu_engine, n):
    """Trees of every shape and stage count in one batch: full and member runs."""
    from treetime_amd.engine import batch_info, batch_run_members

    shapes = [("cherry", 3), ("star", 70), ("nested", 300), ("caterpillar", 65), ("two-stages", 513), ("one-more", 64),
              ("comb", 70)]
    say(f"[cluster] batch n={n}")
    trees = [build(gpu_engine, s, n, P, 7 + i) for i, (s, P) in enumerate(shapes)]
    for kind in ("marginal", "joint", "loglik"):
        for tips in ((False, True, False) if kind != "loglik" else (False,)):
            args = {} if kind == "loglik" else {"reconstruct_tips": tips}
            ref = [getattr(t, kind)(**args) for t in trees]
            states = [t.states() for t in trees]
            prof = [t.profiles() for t in trees]
            got = batch_run(gpu_engine, trees, kind, **args)
            assert batch_info(gpu_engine, trees, kind=kind, **args)["wave_items"] == 3
            for i, t in enumerate(trees):
                assert close(got[i], ref[i]), (kind, tips, i)
                assert close(t.total(), ref[i])
                if kind != "loglik":  # which leaves states and profiles stale
                    assert np.array_equal(t.states(), states[i]), (kind, tips, i)
                if kind == "marginal":
                    assert np.array_equal(t.profiles(), prof[i])
            for part in ([4, 1, 3], [5, 2], [0]):  # the last two as the trees' own passes
                some = batch_run_members(gpu_engine, trees, part, kind, want_logL=True, **args)
                for i, lh in zip(part, some):
                    assert close(lh, ref[i])
                    assert kind == "loglik" or np.array_equal(trees[i].states(), states[i])
    for t in trees:
        t.close()


@pytest.mark.parametrize("mode", ["", "block"], ids=["clustered", "persistent"])
def test_member_runs_on_two_streams(gpu_engine, monkeypatch, mode):
    """Member runs of disjoint trees on two streams, one after another without
    a wait in between: each has its own trees' results."""
    import torch

    from treetime_amd.engine import batch_run_members

    say(f"[cluster] member runs on two streams {mode}")
    if mode:
        monkeypatch.setenv("TT_BATCH_MODE", mode)
    shapes = [("nested", 900), ("caterpillar", 700), ("two-stages", 3000), ("one-more", 64), ("nested", 65), ("star", 300)]
    trees = [build(gpu_engine, s, 4, P, 21 + i) for i, (s, P) in enumerate(shapes)]
    ref = [t.marginal() for t in trees]
    prof = [t.profiles() for t in trees]
    streams = [torch.cuda.Stream() for _ in range(2)]
    batch_run_members(gpu_engine, trees, [0], "marginal")
    for t in trees:  # other rows than the runs below are to leave
        t.joint()
    parts = [[0, 2, 5], [1, 3, 4]]
    for k in range(6):
        batch_run_members(gpu_engine, trees, parts[k % 2], "marginal", stream=streams[k % 2].cuda_stream)
    torch.cuda.synchronize()
    for t, lh, pr in zip(trees, ref, prof):
        assert close(t.total(), lh)
        assert np.array_equal(t.profiles(), pr)
        t.close()


@pytest.mark.parametrize("members", [[1], [2, 0], [0, 1, 2]], ids=["own", "two-own", "pool"])
def test_member_totals_on_a_callers_stream(gpu_engine, members):
    """The log-likelihoods of a member run on a caller's stream are that run's,
    for other branch lengths than the pool's last run had."""
    import torch

    from treetime_amd.engine import batch_run_members

    say(f"[cluster] member totals on a caller's stream {members}")
    trees = [build(gpu_engine, s, 4, P, 31 + i) for i, (s, P) in enumerate([("nested", 300), ("two-stages", 130), ("star", 90)])]
    batch_run(gpu_engine, trees, "marginal")
    stream = torch.cuda.Stream()
    for k, kind in enumerate(("marginal", "joint", "loglik")):
        batch_run(gpu_engine, trees, kind)
        for t in trees:
            nodes = np.flatnonzero(t.parent >= 0)
            t.set_branch_lengths(nodes, np.full(len(nodes), 0.02 + 0.03 * k))
        got = batch_run_members(gpu_engine, trees, members, kind, stream=stream.cuda_stream, want_logL=True)
        for i, lh in zip(members, got):
            assert close(lh, trees[i].total()), (kind, i)
            assert close(lh, getattr(trees[i], kind)()), (kind, i)
    for t in trees:
        t.close()


@pytest.mark.parametrize("shape,P,levels", [("caterpillar", 2700, True), ("comb", 2200, True), ("two-stages", 4200, False)])
def test_wide_chains_walk_levels(gpu_engine, shape, P, levels):
    """20 states: a tree of few rows to a level takes the level kernels, like a
    small one, whatever its size.  Both kinds of pass round rows in their own
    order: the parity tests' bounds."""
    say(f"[cluster] wide chain {shape} P={P}")
    a, b = build(gpu_engine, shape, 20, P, 12), build(gpu_engine, shape, 20, P, 12)
    used = gpu_engine.usage()[0]
    lh = a.marginal()
    assert (gpu_engine.usage()[0] == used) == levels  # the first clustered pass has programs to keep
    prof, site = a.profiles(), a.sequence_lh()
    assert close(batch_run(gpu_engine, [a, b], "marginal")[0], lh, 1e-7)
    assert np.max(np.abs(a.sequence_lh() - site) / np.maximum(1.0, np.abs(site))) <= 1e-6
    assert np.max(np.abs(a.profiles() - prof)) <= 2e-6
    a.close()
    b.close()


@pytest.mark.parametrize("shape,n,tile", [("two-stages", 4, "1"), ("nested", 5, "0"), ("two-stages", 20, "1")])
def test_batch_of_one_tree(gpu_engine, monkeypatch, shape, n, tile):
    """A batch of one tree is the tree's own pass, as a full and as a member
    run, on the plan's stream and on a caller's: results, flags and order."""
    import torch

    from treetime_amd.engine import batch_info, batch_run_members

    say(f"[cluster] batch of one {shape} n={n} tile={tile}")
    monkeypatch.setenv("TT_TILE", tile)
    a, b = build(gpu_engine, shape, n, 257, 6), build(gpu_engine, shape, n, 257, 6)
    s = torch.cuda.Stream()
    for kind in ("marginal", "joint", "loglik"):
        for tips in ((False, True, False) if kind != "loglik" else (False,)):
            args = {} if kind == "loglik" else {"reconstruct_tips": tips}
            ref = getattr(b, kind)(**args)
            for k, stream in enumerate((None, s.cuda_stream, None, s.cuda_stream)):
                a.joint() if kind != "joint" else a.marginal()
                if k < 2:
                    got = batch_run(gpu_engine, [a], kind, stream=stream, **args)[0]
                else:
                    got = batch_run_members(gpu_engine, [a], [0], kind, stream=stream, want_logL=True, **args)[0]
                assert got == ref and a.total() == ref, (kind, tips, k)
                if kind != "loglik":
                    assert np.array_equal(a.states(), b.states()), (kind, tips, k)
                if kind == "marginal":
                    assert np.array_equal(a.profiles(), b.profiles())
            assert batch_info(gpu_engine, [a], kind=kind, **args)["wave_items"] == 2
    a.close()
    b.close()


@pytest.mark.parametrize("n", [4, 20])
def test_from_root_after_trim(gpu_engine, n):
    """tt_tree_trim takes the joint buffers away under the recorded passes
    from given root states (the second such pass is recorded): the next joint
    pass has others, with a tree's buffers where the old ones were."""
    say(f"[cluster] from root after trim n={n}")
    a, b, other = (build(gpu_engine, "two-stages", n, 130, 8) for _ in range(3))
    given = [((np.arange(130) + k) % n).astype(np.uint8) for k in range(4)]
    a.joint()
    for k in range(3):
        a.joint_from_root(given[k])
    a.trim()
    other.joint()
    a.joint()
    b.joint()
    for k in (3, 1):
        assert close(a.joint_from_root(given[k]), b.joint_from_root(given[k]))
        assert np.array_equal(a.states(), b.states())
    for t in (a, b, other):
        t.close()


@pytest.mark.parametrize("n", [4, 5])
def test_clustered_matches_oracle(gpu_engine, monkeypatch, n):
    from helpers import build_oracle, polytomy_job
    from treetime_amd.prepare import device_tree

    say(f"[cluster] oracle n={n}")
    job, prep, alphabet = polytomy_job(140, 300, n, 31, 0.3)
    monkeypatch.setenv("TT_TILE", "0")
    dev = device_tree(gpu_engine, prep)
    ta, nodes, tips = build_oracle(prep, alphabet, job["gtr"])
    assert close(dev.marginal(), ta.marginal(), 1e-7)
    prof = dev.profiles()
    for v, nd in enumerate(nodes):
        if nd.clades:
            assert np.max(np.abs(prof[v] - nd.marginal_profile)) <= 2e-6
    assert close(dev.joint(), ta.joint(), 1e-9)
    dev.close()



@pytest.mark.parametrize("shape,P,extra", [("cherry", 1, 2), ("one-cluster", 63, 10), ("two-stages", 64, 2),
                                           ("two-stages", 65, 10), ("nested", 257, 2), ("star", 65, 50),
                                           ("caterpillar", 130, 2), ("comb", 65, 10), ("ladder", 70, 2)])
def test_clustered_20_states(gpu_engine, shape, P, extra):
    """20 states: lanes past the last pattern, rows of two and of more
    children, tables of the tips' characters and (more than 25 of them) none,
    against the FP64 sums at the parity tests' bounds."""
    say(f"[cluster] {shape} n=20 P={P} codes={20 + extra}")
    n, rng = 20, np.random.default_rng(9)
    parent, bl = tree_of(shape, rng)
    t, N = np.maximum(bl, 1e-6), len(parent)
    pi, W = synth.random_gtr(n, rng, 5.0, 0.5)
    np.fill_diagonal(W, 0.0)
    eig, v, vi = GTR._eig_single_site(W, pi)
    inner = np.isin(np.arange(N), parent[parent >= 0])
    lut = np.concatenate([np.eye(n), rng.integers(0, 2, (extra, n)) + 0.0]).astype(np.float32)
    lut[n:, 0] = 1.0
    base = rng.integers(0, n, P)[None].repeat((~inner).sum(), 0)
    codes = np.where(rng.random(base.shape) < 0.3, rng.integers(0, n + extra, base.shape), base).astype(np.uint8)
    codes[:, 0] = np.arange(len(codes)) % (n + extra)
    mult = rng.integers(1, 9, P).astype(float)
    dt, other = (DeviceTree(gpu_engine, parent, t, codes, lut, mult, pi, eig, v, vi, 1.0) for _ in range(2))
    Q = np.maximum(0.0, (v * np.exp(np.outer(t, eig))[:, None, :]) @ vi)
    sub, out, off = np.ones((N, P, n)), np.empty((N, P, n)), np.zeros(P)
    sub[~inner] = lut[codes]
    for x in range(N - 1, 0, -1):  # preorder numbering: children first
        if inner[x]:
            m = sub[x].max(1)
            sub[x] /= m[:, None]
            off += np.log(m)
        sub[parent[x]] *= sub[x] @ Q[x]
    out[0] = sub[0] * pi
    site = off + np.log(out[0].sum(1))
    for x in range(N):
        if x:
            out[x] = sub[x] * ((out[parent[x]] / (sub[x] @ Q[x])) @ Q[x].T)
        out[x] /= out[x].sum(1, keepdims=True)
    for tips in (False, True, False):  # as a batch: a small tree's own pass walks levels
        got = batch_run(gpu_engine, [dt, other], "marginal", reconstruct_tips=tips)[0]
        assert close(got, float(site @ mult), 1e-7)
        assert np.max(np.abs(dt.sequence_lh() - site) / np.maximum(1.0, np.abs(site))) <= 1e-6
        prof = dt.profiles()
        rows = np.arange(N) if tips else np.flatnonzero(inner)
        assert np.max(np.abs(prof[rows] - out[rows])) <= 2e-6
    assert close(batch_run(gpu_engine, [dt, other], "loglik")[0], got)
    dt.close()
    other.close()
