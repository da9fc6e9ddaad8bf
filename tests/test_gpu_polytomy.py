"""Rows with hundreds of children on branches of 1e-6 to 1e-5: tips of one
state followed by a larger number of another, so that a state trails the
others by hundreds of decades and wins in the end.

Held to FP64 sums of logarithms, as the reference forms them (treeanc.py:
857-877, 980-1011).  Each of the K messages of a row carries its branch's FP32
rounding, 2^-23 relative at most, and one that disagrees adds 11 or more to
the pattern's |logL|: 1e-7 relative for logL.  The patterns are decided by
factors of 1e5 and more, so their profiles are 0 and 1 up to FP32 rounding of
one step: 2e-6, the bound of the other parity tests.  States are equal."""
import numpy as np
import pytest

from test_gpu_cluster import close, say
from treetime_amd import synth
from treetime_amd.engine import DeviceTree, batch_run
from treetime_amd.gtr import GTR

pytestmark = pytest.mark.gpu

# (first tips, then tips): counts per state in tip order
ORDERS = [(60, 80), (80, 60), (20, 25), (100, 200), (200, 100), (9, 7), (130, 170)]


def polytomy(shape, rng):
    """(parent, length), preorder numbering, tips in the order they are listed."""
    if shape == "star":
        par = [-1] + [0] * 300
    else:  # 40 tips and 3 rows of 260 tips under the root, one of them inside another
        par = [-1] + [0] * 40
        inner = 0
        for k in range(3):
            par.append(inner if k == 2 else 0)
            inner = len(par) - 1
            par += [inner] * 260
    return np.array(par, np.int32), np.r_[0.0, rng.uniform(1e-6, 1e-5, len(par) - 1)]


def case(shape, n, seed):
    rng = np.random.default_rng(seed)
    parent, t = polytomy(shape, rng)
    pi, W = synth.random_gtr(n, rng, 50.0, 0.2)
    np.fill_diagonal(W, 0.0)
    eig, v, vi = GTR._eig_single_site(W, pi)
    tips = np.flatnonzero(~np.isin(np.arange(len(parent)), parent))
    lut = np.concatenate([np.eye(n), np.ones((1, n))]).astype(np.float32)
    cols = []
    for k, (a, c) in enumerate(ORDERS * 10):  # 70 patterns: a wave and a few
        x, y = rng.choice(n, 2, replace=False)
        col = np.full(len(tips), n)
        at = k % 3 if shape == "star" else 40 + 260 * (k % 3)  # the later rows of a nested tree, or the root's
        ends = len(tips) if shape == "star" else min(len(tips), at + 260)
        if shape != "star":
            a, c = (a, c) if a + c <= 260 else (int(a * 260 / (a + c)), 260 - int(a * 260 / (a + c)))
        col[at:min(at + a, ends)] = x
        col[at + a:min(at + a + c, ends)] = y
        cols.append(col)
    codes = np.array(cols).T.astype(np.uint8).copy()
    mult = rng.integers(1, 9, codes.shape[1]).astype(float)
    return dict(parent=parent, t=t, codes=codes, lut=lut, mult=mult, pi=pi, eig=eig, v=v, vi=vi, tips=tips, n=n)


def device(engine, c):
    return DeviceTree(engine, c["parent"], c["t"], c["codes"], c["lut"], c["mult"], c["pi"], c["eig"], c["v"], c["vi"],
                      1.0)


def exact(c, t=None):
    """(logL per pattern, profiles, joint logL per pattern, joint states) in 64 bits."""
    parent, n, N = c["parent"], c["n"], len(c["parent"])
    t = c["t"] if t is None else t
    Q = np.maximum(0.0, (c["v"] * np.exp(np.outer(t, c["eig"]))[:, None, :]) @ c["vi"])
    Qj = np.log(np.maximum(1e-12, Q))
    rows = np.zeros((N, c["codes"].shape[1], n))
    best = np.zeros_like(rows)
    back = np.zeros(rows.shape, int)
    with np.errstate(divide="ignore"):
        rows[c["tips"]] = np.log(c["lut"][c["codes"]].astype(float))
    best[c["tips"]] = np.log(np.maximum(1e-12, c["lut"][c["codes"]].astype(float)))
    for x in range(N - 1, 0, -1):
        m = rows[x].max(1, keepdims=True)
        rows[parent[x]] += np.log(np.exp(rows[x] - m) @ Q[x]) + m
        s = best[x][:, :, None] + Qj[x]
        back[x] = s.argmax(1)
        best[parent[x]] += s.max(1)
    root = rows[0] + np.log(c["pi"])
    site = np.log(np.exp(root - root.max(1, keepdims=True)).sum(1)) + root.max(1)
    prof = np.zeros_like(rows)
    states = np.zeros(rows.shape[:2], int)
    jroot = best[0] + np.log(c["pi"])
    states[0] = jroot.argmax(1)
    sub = np.exp(rows - rows.max(2, keepdims=True))
    prof[0] = np.exp(root - root.max(1, keepdims=True))
    prof[0] /= prof[0].sum(1, keepdims=True)
    for x in range(1, N):
        up = np.maximum(1e-12, prof[parent[x]]) / (sub[x] @ Q[x])
        prof[x] = sub[x] * (up @ Q[x].T)
        prof[x] /= prof[x].sum(1, keepdims=True)
        states[x] = np.take_along_axis(back[x], states[parent[x]][:, None], 1)[:, 0]
    return site, prof, jroot.max(1), states


def check_marginal(c, dt, lh, ref, rows):
    site, prof = ref[:2]
    assert close(lh, float(site @ c["mult"]), 1e-7)
    assert np.max(np.abs(dt.sequence_lh() - site) / np.maximum(1.0, np.abs(site))) <= 1e-7
    assert np.max(np.abs(dt.profiles()[rows] - prof[rows])) <= 2e-6
    assert np.array_equal(dt.states()[rows], prof[rows].argmax(2))


def several(engine, c, kind, check):
    """A batch large enough that its trees do not take their own passes in turn."""
    trees = [device(engine, c) for _ in range(12)]
    for dt, lh in zip(trees, batch_run(engine, trees, kind)):
        check(dt, lh)
    for dt in trees:
        dt.close()


CASES = [("star", 2), ("star", 4), ("star", 5), ("nested", 3), ("nested", 4), ("nested", 5)]


@pytest.mark.parametrize("shape,n", CASES, ids=["%s-%d" % c for c in CASES])
@pytest.mark.parametrize("tile", ["0", "1"], ids=["clustered", "one-launch"])
def test_trailing_state_marginal(gpu_engine, monkeypatch, tile, shape, n):
    say(f"[polytomy] marginal {shape} n={n} tile={tile}")
    monkeypatch.setenv("TT_TILE", tile)
    c = case(shape, n, 3)
    dt, ref = device(gpu_engine, c), exact(c)
    assert (dt.pass_shape()[0] > 0) == (tile == "1")
    inner = np.unique(c["parent"][1:])
    check_marginal(c, dt, dt.marginal(), ref, inner)
    check_marginal(c, dt, dt.marginal(reconstruct_tips=True), ref, np.arange(len(c["parent"])))
    dt.close()
    several(gpu_engine, c, "marginal", lambda dt, lh: check_marginal(c, dt, lh, ref, inner))


@pytest.mark.parametrize("shape,n", [("star", 20), ("nested", 20), ("star", 22), ("nested", 21)])
def test_trailing_state_wide(gpu_engine, shape, n):
    say(f"[polytomy] wide {shape} n={n}")
    c = case(shape, n, 4)
    dt, ref = device(gpu_engine, c), exact(c)
    inner = np.unique(c["parent"][1:])
    if n != 20:
        check_marginal(c, dt, dt.marginal(), ref, inner)
    dt.close()
    several(gpu_engine, c, "marginal", lambda dt, lh: check_marginal(c, dt, lh, ref, inner))


@pytest.mark.parametrize("shape,n", [("star", 4), ("nested", 5), ("nested", 20), ("star", 22)])
def test_trailing_state_update(gpu_engine, shape, n):
    """Root-path updates recompute the same rows; the start of a small tree of
    20 states is a pass of level kernels, whose normalisers are products too."""
    say(f"[polytomy] update {shape} n={n}")
    c = case(shape, n, 5)
    dt = device(gpu_engine, c)
    dt.loglik()
    t = c["t"].copy()
    for node in (1, len(t) - 1, len(t) // 2):
        t[node] = 2e-5
        got, site = dt.update_branch(node, 2e-5), exact(c, t)[0]
        assert close(got, float(site @ c["mult"]), 1e-7), node
        assert np.max(np.abs(dt.sequence_lh() - site) / np.maximum(1.0, np.abs(site))) <= 1e-7
    dt.close()


@pytest.mark.parametrize("shape,n", CASES + [("nested", 20), ("star", 21)])
def test_trailing_state_joint(gpu_engine, monkeypatch, shape, n):
    """The max-product rows of the joint pass, every path that forms them."""
    say(f"[polytomy] joint {shape} n={n}")
    c = case(shape, n, 6)
    site, states = exact(c)[2:]
    inner = np.unique(c["parent"][1:])

    def check(dt, lh):
        assert close(lh, float(site @ c["mult"]), 1e-9)
        assert np.array_equal(dt.states()[inner], states[inner])
        assert np.allclose(dt.sequence_lh(), site, rtol=1e-9)

    for tile in ("0", "1"):
        monkeypatch.setenv("TT_TILE", tile)
        dt = device(gpu_engine, c)
        check(dt, dt.joint())
        dt.close()
    several(gpu_engine, c, "joint", check)
