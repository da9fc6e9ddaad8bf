"""Performance cases of the pruning engine: the calls a user's program makes,
over the sizes, alphabets and options that trees and alignments come in.

Sizes follow the repository's own workloads (treetime_amd.synth.WORKLOADS and
the uneven nucleotide mix of bench.py): coalescent trees of 50 to 5000 tips,
random GTR models, alignments simulated down the tree and kept as compressed
patterns (a few constant ones that carry most sites, the others private).
Inputs are made on the GPU from the seed.  Every case goes through the
package's public handles (Engine, DeviceTree, batch_run); results that stay
on the device are the tree's own buffers (tt_get_device_buffers)."""
import ctypes
import math
import random

import numpy as np
import torch

from treetime_amd import GTR, _native, synth
from treetime_amd.engine import DeviceTree, Engine, batch_run, code_lut
from treetime_amd.prepare import effective_lengths

ALPHABET = {4: "nuc_nogap", 5: "nuc", 20: "aa_nogap"}
AMBIGUOUS = {4: "N", 5: "N", 20: "X"}
TINY = 1e-12


def listed():
    return [
        # one small tree, the drop-in call of an interactive analysis: latency and launches
        {"name": "marginal-200", "kind": "marginal", "states": 4, "tips": 200, "patterns": 1135, "depth": 0.02,
         "polytomies": 0.0, "noise": 0.015, "tip_states": False},
        # the smallest call: a gene tree of a few dozen sequences, the default alphabet (gap as fifth state)
        {"name": "joint-60-gap", "kind": "joint", "states": 5, "tips": 60, "patterns": 301, "depth": 0.1,
         "polytomies": 0.0, "noise": 0.02, "tip_states": False},
        # an outbreak tree with collapsed branches, default alphabet, tips reconstructed as well
        {"name": "marginal-2000-gap-poly", "kind": "marginal", "states": 5, "tips": 2000, "patterns": 2501,
         "depth": 0.01, "polytomies": 0.25, "noise": 0.02, "tip_states": True},
        # the large single-tree workload, both reconstructions
        {"name": "marginal-5000", "kind": "marginal", "states": 4, "tips": 5000, "patterns": 2637, "depth": 0.01,
         "polytomies": 0.0, "noise": 0.02, "tip_states": False},
        {"name": "joint-5000", "kind": "joint", "states": 4, "tips": 5000, "patterns": 2637, "depth": 0.01,
         "polytomies": 0.0, "noise": 0.02, "tip_states": False},
        # protein alignments (20 states, matrix cores), large marginal and ordinary joint
        {"name": "protein-marginal-1000", "kind": "marginal", "states": 20, "tips": 1000, "patterns": 4534,
         "depth": 0.3, "polytomies": 0.0, "noise": 0.0, "tip_states": False},
        {"name": "protein-joint-400", "kind": "joint", "states": 20, "tips": 400, "patterns": 1501, "depth": 0.3,
         "polytomies": 0.0, "noise": 0.01, "tip_states": False},
        # trial branch lengths, one call each: what a server or a line search over one branch asks for
        {"name": "branch-trials-500", "kind": "trials", "states": 4, "tips": 500, "patterns": 903, "depth": 0.02,
         "polytomies": 0.0, "noise": 0.015, "trials": 12},
        # one round of optimize_tree_marginal with infer_gtr: marginal pass, transition counts, all branch optima
        {"name": "optimize-1500", "kind": "optimize", "states": 4, "tips": 1500, "patterns": 1203, "depth": 0.02,
         "polytomies": 0.0, "noise": 0.015},
        # a pool of uneven trees (segments, genes, bootstrap replicates) in one batched call, both kinds
        {"name": "batch-marginal-20", "kind": "batch_marginal", "states": 4, "trees": 20, "sizes_seed": 3001,
         "depth": 0.02, "noise": 0.015},
        {"name": "batch-joint-20", "kind": "batch_joint", "states": 4, "trees": 20, "sizes_seed": 3006,
         "depth": 0.02, "noise": 0.015},
        # pattern compression of a device-resident alignment before the tree is built
        {"name": "compress-5000x30000", "kind": "compress", "sequences": 5000, "columns": 30000, "variable": 2600},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["marginal", "marginal", "marginal", "joint", "joint", "trials", "optimize", "batch_marginal",
                       "batch_joint", "compress"])
    if kind == "compress":
        n, l = _log_int(rng, 40, 5000), _log_int(rng, 500, 30000)
        return {"kind": kind, "sequences": n, "columns": l, "variable": max(1, int(l * rng.uniform(0.03, 0.4)))}
    if kind in ("batch_marginal", "batch_joint"):
        return {"kind": kind, "states": 4, "trees": rng.randint(5, 20), "sizes_seed": rng.randrange(1 << 30),
                "depth": rng.choice([0.005, 0.02, 0.05]), "noise": 0.015}
    if kind == "trials":
        return {"kind": kind, "states": rng.choice([4, 4, 5, 20]), "tips": _log_int(rng, 50, 1000),
                "patterns": _log_int(rng, 100, 3000), "depth": 0.02, "polytomies": rng.choice([0.0, 0.2]),
                "noise": 0.015, "trials": 12}
    if kind == "optimize":
        return {"kind": kind, "states": rng.choice([4, 4, 5]), "tips": _log_int(rng, 50, 1500),
                "patterns": _log_int(rng, 100, 1200), "depth": rng.choice([0.005, 0.02, 0.05]),
                "polytomies": rng.choice([0.0, 0.2]), "noise": 0.015}
    states = rng.choice([4, 4, 5, 5, 20])
    tips = _log_int(rng, 20, 1000 if states == 20 else 5000)
    patterns = _log_int(rng, 60, 4500 if states == 20 else 6000)
    patterns = max(60, min(patterns, (4000000 if states == 20 else 13000000) // tips))
    return {"kind": kind, "states": states, "tips": tips, "patterns": patterns,
            "depth": 0.3 if states == 20 else rng.choice([0.005, 0.02, 0.1]), "polytomies": rng.choice([0.0, 0.0, 0.3]),
            "noise": rng.choice([0.0, 0.015]), "tip_states": rng.random() < 0.3}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _batch_sizes(case):
    """(tips, patterns) of every tree of a batch; a fixed list of the case."""
    r = random.Random(case["sizes_seed"])
    sizes = [(_log_int(r, 50, 4000), _log_int(r, 300, 16000)) for _ in range(case["trees"])]
    total = sum(a * b for a, b in sizes)
    cap = 120000000
    if total > cap:
        sizes = [(a, max(65, int(b * cap / total))) for a, b in sizes]
    return sizes


def _tree(tips, depth, polytomies, rng):
    """(parent, branch length) in preorder numbering: a coalescent tree of
    root height ``depth`` whose shortest internal branches are collapsed."""
    n = 2 * tips - 1
    parent = np.full(n, -1, dtype=np.int64)
    height = np.zeros(n)
    ks = np.arange(tips, 1, -1)
    wait = np.cumsum(rng.exponential(2.0 / (ks * (ks - 1.0))))
    pick = rng.random((tips - 1, 2))
    live = list(range(tips))
    for s in range(tips - 1):
        new = tips + s
        for u in pick[s]:
            i = int(u * len(live))
            parent[live[i]] = new
            live[i] = live[-1]
            live.pop()
        live.append(new)
        height[new] = wait[s]
    height *= depth / height[-1]
    bl = np.where(parent >= 0, height[parent] - height, 0.0)
    drop = int(polytomies * (tips - 2))
    if drop:
        inner = np.arange(tips, n - 1)
        gone = np.zeros(n, dtype=bool)
        gone[inner[np.argsort(bl[inner], kind="stable")[:drop]]] = True
        for v in range(n - 1):  # parents have larger numbers: climb over collapsed nodes
            p = parent[v]
            while gone[p]:
                bl[v] += bl[p]
                p = parent[p]
            parent[v] = p
        keep = np.where(~gone)[0]
        new = np.full(n, -1, dtype=np.int64)
        new[keep] = np.arange(len(keep))
        parent = np.where(parent[keep] >= 0, new[parent[keep]], -1)
        bl = bl[keep]
    parent, bl, _ = synth.preorder_renumber(parent.astype(np.int32), bl)
    return parent, bl


def _levels(parent):
    """Depth of every node, and the nodes of each depth (parents precede
    their children in preorder numbering)."""
    depth = np.zeros(len(parent), dtype=np.int64)
    for v in range(1, len(parent)):
        depth[v] = depth[parent[v]] + 1
    order = np.argsort(depth, kind="stable")
    cut = np.searchsorted(depth[order], np.arange(depth.max() + 2))
    return depth, [order[cut[d]:cut[d + 1]] for d in range(depth.max() + 1)]


def _expqt(m, t):
    """P(t) [branch][child state][parent state] in 64 bits."""
    e = torch.exp(m["mu"] * t[:, None] * m["eig"][None, :])
    return torch.clamp(torch.matmul(m["v"][None] * e[:, None, :], m["vi"][None].contiguous()), min=0.0)


def _columns(tree, m, n_cols, g):
    """(tips, n_cols) states of columns evolved down the tree."""
    n, dev = m["n"], "cuda"
    states = torch.empty((len(tree["parent"]), n_cols), dtype=torch.uint8, device=dev)
    u = torch.rand(n_cols, device=dev, generator=g, dtype=torch.float64)
    states[0] = torch.bucketize(u, torch.cumsum(m["pi"], 0)[:-1]).to(torch.uint8)
    cum = torch.cumsum(_expqt(m, tree["t64"]), 1).float()  # over the child state
    for nodes in tree["levels"][1:]:
        ps = states[tree["parent_d"][nodes]].long()
        u = torch.rand(ps.shape, device=dev, generator=g)
        child = torch.zeros(ps.shape, dtype=torch.uint8, device=dev)
        for k in range(n - 1):
            child += (u > torch.gather(cum[nodes, k, :], 1, ps)).to(torch.uint8)
        states[nodes] = child
    return states[tree["tips"]]


def _model(states, seed):
    rng = np.random.default_rng(seed)
    pi, W = synth.random_gtr(states, rng, 2.0 if states == 20 else 5.0, 1.0 if states == 20 else 0.5)
    gtr = GTR.custom(mu=1.0, pi=pi, W=W, alphabet=ALPHABET[states])
    d = {k: torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")
         for k, x in (("pi", gtr.Pi), ("eig", gtr.eigenvals), ("v", gtr.v), ("vi", gtr.v_inv))}
    return dict(d, gtr=gtr, n=states, mu=float(gtr.mu))


def _inputs(case, seed):
    """Host arrays of one DeviceTree, and the same on the GPU for exact()."""
    rng = np.random.default_rng(seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = _model(case["states"], seed)
    P = case["patterns"]
    sites = 4 * P
    parent, bl = _tree(case["tips"], case["depth"], case.get("polytomies", 0.0), rng)
    t = effective_lengths(bl, sites)
    is_tip = np.ones(len(parent), dtype=bool)
    is_tip[parent[parent >= 0]] = False
    _, levels = _levels(parent)
    dev = "cuda"
    tree = {"parent": parent, "t": t, "t64": torch.as_tensor(t, device=dev),
            "parent_d": torch.as_tensor(parent.astype(np.int64), device=dev),
            "levels": [torch.as_tensor(x, device=dev) for x in levels],
            "tips": torch.as_tensor(np.where(is_tip)[0], device=dev)}
    # variable columns, as many as the patterns that are not constant
    need = max(1, P - case["states"])
    got, have, ask = [], 0, need
    for _ in range(8):
        c = _columns(tree, m, min(ask, 60000), g)
        var = (c != c[:1]).any(0)
        c = c[:, var][:, :need - have]
        got.append(c)
        have += c.shape[1]
        if have >= need:
            break
        ask = int(1.3 * (need - have) / max(have / ask, 0.02)) + 64
    if have < need:
        got.append(_columns(tree, m, need - have, g))
    const = torch.arange(P - need, device=dev, dtype=torch.uint8)[None].expand(case["tips"], P - need)
    st = torch.cat([const] + got, 1)
    letters = torch.as_tensor(np.array([ord(str(x)) for x in m["gtr"].alphabet], dtype=np.uint8), device=dev)
    codes = letters[st.long()]
    if case["noise"] > 0:
        u = torch.rand(codes.shape, device=dev, generator=g)
        u[:, :P - need] = 1.0
        codes[u < case["noise"] * 2 / 3] = ord(AMBIGUOUS[case["states"]])
        if case["states"] != 5:
            codes[(u >= case["noise"] * 2 / 3) & (u < case["noise"])] = ord("-")
    mult = np.ones(P)
    mult[:P - need] = np.floor(1.0 + (sites - P) * m["gtr"].Pi[:P - need])
    tree.update(model=m, codes=codes, mult=mult, lut=code_lut(m["gtr"].profile_map, m["n"]))
    return tree


_ENGINE = []


def _engine():
    if not _ENGINE:
        _ENGINE.append(Engine(0, 0))
    return _ENGINE[0]


class _Buffer:
    """A device buffer of the library as torch sees it."""

    def __init__(self, ptr, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (ptr, False), "version": 2}


def _buffers(dev):
    a, b, c = ctypes.POINTER(ctypes.c_float)(), ctypes.POINTER(ctypes.c_uint8)(), ctypes.POINTER(ctypes.c_double)()
    _native.check(dev.lib.tt_get_device_buffers(dev.handle, ctypes.byref(a), ctypes.byref(b), ctypes.byref(c)))

    def view(p, shape, kind):
        return torch.as_tensor(_Buffer(ctypes.cast(p, ctypes.c_void_p).value, shape, kind, dev), device="cuda")

    return (view(a, (dev.n_nodes, dev.P, dev.n), "<f4"), view(b, (dev.n_nodes, dev.P), "|u1"),
            view(c, (dev.P,), "<f8"))


def _device_tree(x):
    g = x["model"]["gtr"]
    torch.cuda.synchronize()
    return DeviceTree(_engine(), x["parent"], x["t"], x["codes"].cpu().numpy(), x["lut"], x["mult"], g.Pi,
                      g.eigenvals, g.v, g.v_inv, g.mu)


def _batch_case(case, i, size):
    return {"states": case["states"], "tips": size[0], "patterns": size[1], "depth": case["depth"],
            "noise": case["noise"]}


def _trial_list(case, x, seed):
    """(node, trial length, present length) of a line search over branches."""
    rng = np.random.default_rng(seed + 1)
    nodes = rng.choice(np.arange(1, len(x["parent"])), size=case["trials"], replace=False)
    return [(int(v), float(x["t"][v] * f), float(x["t"][v])) for v, f in zip(nodes, rng.uniform(0.3, 3.0, len(nodes)))]


def _alignment(case, seed):
    """(sequences, pitch) bytes: a random root sequence, ``variable`` columns
    with their own share of changed rows, 2% N, gaps at both ends of 1% of the rows."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, l, v = case["sequences"], case["columns"], case["variable"]
    dev = "cuda"
    acgt = torch.tensor([65, 67, 71, 84], dtype=torch.uint8, device=dev)
    a = torch.zeros((n, (l + 15) // 16 * 16), dtype=torch.uint8, device=dev)
    a[:, :l] = acgt[torch.randint(0, 4, (l,), device=dev, generator=g)][None]
    cols = torch.randperm(l, device=dev, generator=g)[:v]
    share = 0.001 + 0.299 * torch.rand(v, device=dev, generator=g)
    hit = torch.rand((n, v), device=dev, generator=g) < share[None]
    other = acgt[torch.randint(0, 4, (n, v), device=dev, generator=g)]
    a[:, cols] = torch.where(hit, other, a[:, cols])
    a[:, :l][torch.rand((n, l), device=dev, generator=g) < 0.02] = 78
    order = torch.randperm(n, device=dev, generator=g)
    rows, rest = order[:max(1, n // 100)], order[max(1, n // 100):]
    edge = torch.randint(1, max(2, min(500, l // 2)), (len(rows), 2), device=dev, generator=g)
    at = torch.arange(l, device=dev)[None]
    gap = (at < edge[:, :1]) | (at >= l - edge[:, 1:])
    a[rows, :l] = torch.where(gap, torch.full_like(a[:1, :l], 45), a[rows, :l])
    # two rows of every variable column that differ for certain
    at = torch.randint(0, len(rest) - 1, (v,), device=dev, generator=g)
    base = torch.randint(0, 4, (v,), device=dev, generator=g)
    a[rest[at], cols] = acgt[base]
    a[rest[at + 1], cols] = acgt[(base + 1) % 4]
    return a


def prepare(case, seed):
    kind = case["kind"]
    if kind == "compress":
        a = _alignment(case, seed)
        n, l = case["sequences"], case["columns"]
        return {"kind": kind, "chars": a, "columns": l, "engine": _engine(),
                "map": torch.zeros(l, dtype=torch.int32, device="cuda"),
                "patterns": torch.zeros(n * l, dtype=torch.uint8, device="cuda"),
                "mult": torch.zeros(l, dtype=torch.float64, device="cuda")}
    if kind.startswith("batch"):
        trees = [_device_tree(_inputs(_batch_case(case, i, s), seed * 31 + i)) for i, s in enumerate(_batch_sizes(case))]
        state = {"kind": kind, "engine": _engine(), "trees": trees, "buffers": [_buffers(t) for t in trees]}
        batch_run(state["engine"], trees, kind[6:])  # the pool's plan, built once as a server does
        return state
    x = _inputs(case, seed)
    dev = _device_tree(x)
    state = {"kind": kind, "tree": dev, "buffers": _buffers(dev), "tip_states": case.get("tip_states", False)}
    if kind == "trials":
        state["list"] = _trial_list(case, x, seed)
        node, _, t = state["list"][0]
        dev.update_branch(node, t)
    return state


def run(state):
    kind = state["kind"]
    if kind == "compress":
        p = state["engine"].compress_alignment_device(state["chars"], state["columns"], "N", state["map"],
                                                      state["patterns"], state["mult"], fill_overhangs=True)
        n = state["chars"].shape[0]
        return {"n_patterns": p, "map": state["map"], "patterns": state["patterns"][:n * p], "mult": state["mult"][:p]}
    if kind.startswith("batch"):
        lh = batch_run(state["engine"], state["trees"], kind[6:])
        if kind == "batch_joint":
            return {"logL": lh, "states": [b[1] for b in state["buffers"]]}
        return {"logL": lh, "profiles": [b[0] for b in state["buffers"]], "states": [b[1] for b in state["buffers"]],
                "site_logL": [b[2] for b in state["buffers"]]}
    dev = state["tree"]
    prof, states, site = state["buffers"]
    if kind == "marginal":
        lh = dev.marginal(reconstruct_tips=state["tip_states"])
        return {"logL": lh, "profiles": prof, "states": states, "site_logL": site}
    if kind == "joint":
        lh = dev.joint(reconstruct_tips=state["tip_states"])
        return {"logL": lh, "states": states, "site_logL": dev.sequence_lh()}
    if kind == "trials":
        out = np.empty(2 * len(state["list"]))
        for i, (node, trial, t) in enumerate(state["list"]):
            out[2 * i] = dev.update_branch(node, trial)
            out[2 * i + 1] = dev.update_branch(node, t)
        return {"logL": out, "site_logL": site}
    lh = dev.marginal()
    nij, ti = dev.mutation_counts()
    t, status, pair = dev.optimize_branch_lengths_marginal()
    return {"logL": lh, "nij": nij, "Ti": ti, "t": t, "status": status, "pair": np.array(pair), "profiles": prof}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _pass_work(kind, states, tips, inner, patterns, tip_states):
    """Each tip character, multiplicity and per-pattern result once, each
    reconstructed profile and state once; the contractions of both directions."""
    n, branches = states, tips + inner - 1
    made = inner + (tips if tip_states else 0)
    if kind == "marginal":
        return (patterns * (tips + 16 + made * (4 * n + 1)), patterns * (2 * n * n * branches + 4 * n * n * (made - 1)))
    return patterns * (tips + 16 + made), patterns * (2 * n * n * inner + 2 * n * branches)


def work(case):
    kind = case["kind"]
    if kind == "compress":
        n, l, v = case["sequences"], case["columns"], case["variable"]
        return {"bytes": n * l + n * (v + 4) + 4 * l + 8 * (v + 4), "flops": 0}
    if kind.startswith("batch"):
        w = [_pass_work(kind[6:], case["states"], a, a - 1, b, False) for a, b in _batch_sizes(case)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    n, tips, P = case["states"], case["tips"], case["patterns"]
    inner = tips - 1 - int(case["polytomies"] * (tips - 2))
    if kind == "trials":  # the rows of a root path (about 2 ln(tips) nodes) read and written, per call
        path = 2 * math.log(tips)
        return {"bytes": 2 * case["trials"] * P * path * (8 * n + 16), "flops": 2 * case["trials"] * P * path * 4 * n * n}
    b, f = _pass_work("marginal" if kind == "optimize" else kind, n, tips, inner, P, case.get("tip_states", False))
    if kind == "optimize":
        # counts and optima read each branch's two profiles once; about 20
        # evaluations of n multiply-adds and a logarithm per branch and pattern
        branches = tips + inner - 1
        b += 2 * branches * P * 8 * n
        f += branches * P * (4 * n * n + 20 * (2 * n + 40))
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same results in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _tip_rows(x):
    lut = torch.as_tensor(x["lut"], device="cuda").double()
    return lut[x["codes"].long()]


def _up(x, combine, tip, P):
    """Log-space rows of every node: children of the deepest level first.
    ``combine(nodes, rows)`` turns rows of nodes into log messages."""
    L = torch.zeros((len(x["parent"]), P, x["model"]["n"]), dtype=torch.float64, device="cuda")
    L[x["tips"]] = tip
    for nodes in reversed(x["levels"][1:]):
        L.index_add_(0, x["parent_d"][nodes], combine(nodes, L[nodes]))
    return L


def _exact_up(x, t=None):
    """Log subtree likelihoods of every node and the log messages' matrices."""
    E = _expqt(x["model"], x["t64"] if t is None else t)

    def combine(nodes, rows):
        mx = rows.amax(-1, keepdim=True)
        return torch.log(torch.matmul(torch.exp(rows - mx), E[nodes].contiguous())) + mx

    with np.errstate(divide="ignore"):
        return _up(x, combine, torch.log(_tip_rows(x)), x["codes"].shape[1]), E


def _exact_site(x, t=None):
    L, _ = _exact_up(x, t)
    return torch.logsumexp(L[0] + torch.log(x["model"]["pi"]), -1)


def _exact_marginal(x, tip_states):
    """(logL, profiles, per-pattern logL, linear subtree rows, P(t))."""
    L, E = _exact_up(x)
    mult = torch.as_tensor(x["mult"], device="cuda")
    site = torch.logsumexp(L[0] + torch.log(x["model"]["pi"]), -1)
    S = torch.exp(L - L.amax(-1, keepdim=True))
    del L
    prof = torch.zeros_like(S)
    r = S[0] * x["model"]["pi"]
    prof[0] = r / r.sum(-1, keepdim=True)
    for nodes in x["levels"][1:]:
        M, s = E[nodes].contiguous(), S[nodes]
        q = torch.clamp(prof[x["parent_d"][nodes]], min=TINY) / torch.matmul(s, M)
        r = torch.matmul(q, M.transpose(1, 2).contiguous()) * s
        prof[nodes] = r / r.sum(-1, keepdim=True)
    shown = prof
    if not tip_states:
        shown = prof.clone()
        shown[x["tips"]] = 0.0
    return float((mult * site).sum()), shown, site, S, E, prof


def _exact_joint(x):
    """(logL, per-pattern logL) of the joint reconstruction."""
    n = x["model"]["n"]
    E = torch.log(torch.clamp(_expqt(x["model"], x["t64"]), min=TINY))

    def combine(nodes, rows):
        best = rows[..., 0:1] + E[nodes, 0][:, None, :]
        for i in range(1, n):
            best = torch.maximum(best, rows[..., i:i + 1] + E[nodes, i][:, None, :])
        return best

    L = _up(x, combine, torch.log(torch.clamp(_tip_rows(x), min=TINY)), x["codes"].shape[1])
    site = (L[0] + torch.log(x["model"]["pi"])).amax(-1)
    return float((torch.as_tensor(x["mult"], device="cuda") * site).sum()), site


def _pair_rows(x, S, E, prof):
    """Child-side and parent-side profiles of every branch (root excluded)."""
    nodes = torch.arange(1, len(x["parent"]), device="cuda")
    pc = S[nodes]
    q = torch.clamp(prof[x["parent_d"][nodes]], min=TINY) / torch.clamp(torch.matmul(pc, E[nodes].contiguous()), min=TINY)
    tip = torch.zeros(len(x["parent"]), dtype=torch.bool, device="cuda")
    tip[x["tips"]] = True
    inner = ~tip[nodes]
    pc = torch.where(inner[:, None, None], pc / pc.sum(-1, keepdim=True), pc)
    return pc, q / q.sum(-1, keepdim=True)


def _best_lengths(x, pc, pp, max_t=4.0):
    """Optimal length of every profile pair: the zero of the derivative of
    sum mult log(pc P(t) pp) - exp(t^2 / 1e4), by bisection."""
    m = x["model"]
    w = torch.as_tensor(x["mult"], device="cuda")[None, :].expand(pc.shape[:2])
    gap = m["gtr"].gap_index
    if gap is not None and x.get("use_gap"):
        w = w * (1 - pc[..., gap]) * (1 - pp[..., gap])
    c = torch.matmul(pc, m["v"]) * torch.matmul(pp, m["vi"].T.contiguous())
    rate = m["mu"] * m["eig"]

    def value(t):
        e = torch.exp(t[:, None] * rate)
        return (w * torch.log(torch.clamp((c * e[:, None, :]).sum(-1), min=0.0) + 1e-24)).sum(1) - torch.exp(t * t / 1e4)

    def slope(t):
        e = torch.exp(t[:, None] * rate)
        f = (c * e[:, None, :]).sum(-1) + 1e-24
        d = (c * (e * rate)[:, None, :]).sum(-1)
        return (w * d / f).sum(1) - 2 * t / 1e4 * torch.exp(t * t / 1e4)

    mult = torch.as_tensor(x["mult"], device="cuda")
    ham = 1 - (mult * (pc * pp).sum(-1)).sum(1) / mult.sum()
    lo, hi = torch.zeros_like(ham), torch.full_like(ham, max_t)
    for _ in range(90):
        mid = 0.5 * (lo + hi)
        up = slope(mid) > 0
        lo, hi = torch.where(up, mid, lo), torch.where(up, hi, mid)
    t = 0.5 * (lo + hi)
    t[~(value(ham) > value(torch.full_like(ham, max_t)))] = math.nan
    return t


def _exact_optimize(x):
    lh, shown, site, S, E, prof = _exact_marginal(x, False)
    n = x["model"]["n"]
    mult = torch.as_tensor(x["mult"], device="cuda")
    nodes = len(x["parent"])
    pc, pp = _pair_rows(x, S, E, prof)
    Eb = E[1:] + 1e-24
    nij = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    ti = torch.zeros(n, dtype=torch.float64, device="cuda")
    for lo in range(0, nodes - 1, 256):
        a, b, M = pc[lo:lo + 256], pp[lo:lo + 256], Eb[lo:lo + 256]
        j = a[..., :, None] * b[..., None, :] * M[:, None]
        j = j * (mult[None, :] / j.sum((-1, -2)))[..., None, None]
        nij += j.sum((0, 1))
        ti += (0.5 * x["t64"][1 + lo:1 + lo + 256, None] * (j.sum(1).sum(-1) + j.sum(1).sum(-2))).sum(0)
    t = torch.zeros(nodes, dtype=torch.float64, device="cuda")
    for lo in range(0, nodes - 1, 512):
        t[1 + lo:1 + lo + 512] = _best_lengths(x, pc[lo:lo + 512], pp[lo:lo + 512])
    kids = np.where(x["parent"] == 0)[0]
    pair = np.array([math.nan, -1.0])
    if len(kids) == 2:
        q = S[int(kids[1])] * x["model"]["pi"]
        q = q / q.sum(-1, keepdim=True)
        pair = np.array([float(_best_lengths(x, pc[int(kids[0]) - 1][None], q[None])[0]), 0.0])
    return {"logL": lh, "nij": nij, "Ti": ti, "t": t, "status": None, "pair": pair, "profiles": shown}


def exact(case, seed):
    kind = case["kind"]
    if kind == "compress":
        return None
    if kind.startswith("batch"):
        out = {"logL": [], "profiles": [], "site_logL": [], "states": [None] * case["trees"]}
        for i, s in enumerate(_batch_sizes(case)):
            x = _inputs(_batch_case(case, i, s), seed * 31 + i)
            if kind == "batch_joint":
                out["logL"].append(_exact_joint(x)[0])
                continue
            lh, prof, site = _exact_marginal(x, False)[:3]
            out["logL"].append(lh)
            out["profiles"].append(prof.cpu())
            out["site_logL"].append(site)
        if kind == "batch_joint":
            return {"logL": np.array(out["logL"]), "states": out["states"]}
        return dict(out, logL=np.array(out["logL"]))
    x = _inputs(case, seed)
    if kind == "marginal":
        lh, prof, site = _exact_marginal(x, case["tip_states"])[:3]
        return {"logL": lh, "profiles": prof, "states": None, "site_logL": site}
    if kind == "joint":
        lh, site = _exact_joint(x)
        return {"logL": lh, "states": None, "site_logL": site}
    if kind == "trials":
        mult = torch.as_tensor(x["mult"], device="cuda")
        base = _exact_site(x)
        lh = np.empty(2 * case["trials"])
        for i, (node, trial, _) in enumerate(_trial_list(case, x, seed)):
            t = x["t64"].clone()
            t[node] = trial
            lh[2 * i] = float((mult * _exact_site(x, t)).sum())
            lh[2 * i + 1] = float((mult * base).sum())
        return {"logL": lh, "site_logL": base}
    return _exact_optimize(x)
