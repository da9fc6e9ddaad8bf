// Cutting a tree into clusters and writing their step programs (host code).
#include "tt_cluster.h"

#include <algorithm>
#include <utility>

// Cluster size.  A stage is one launch: its waves each walk about K nodes, and
// what is left of the tree shrinks about K-fold.  Where a stage has work for
// the whole chip (rows x 64-pattern tiles above 4096 wave programs of 64
// nodes), long programs save launches and rows that go through memory between
// stages; where it has not, a launch costs about as much as ten steps, and
// programs of 16 keep the chain of steps short.  A step of 20 states is longer
// than a launch and its rows take more LDS (2 slots: at most 14 nodes).
static int cluster_size(long rows, long tiles, int n) {
    const bool wide = n > 5;
    return (int)std::max(wide ? 8L : 16L, std::min(wide ? 14L : (long)kClusterMax, rows * tiles / 4096));
}

// A stage cuts larger clusters out of a tree that is a chain, or some: kChain
// programs' rows for every end (what hung on it was cut off in the stage
// before).  Its rows come one after another whatever the cut, and only launches
// are saved; a cluster is then of kChainMax rows, if its rows find room in the
// LDS slots (a chain takes none).  Ladder of 2000 tips x 1000 patterns, n = 4, joint, by that number: 16
// 4159 us, 64 3465, 256 3480, all 4178; 5000 x 2637 12763, 11234, 10548 and
// 10379, marginal 9840, 8092, 7601 and 7394.
constexpr int kChain = 4, kChainMax = 256;

namespace {

// Writes the programs.  Every row's place in its program follows from its
// parent's and the sizes of the subtrees walked before it, so the rows are
// written in one sweep from parents to children, without recursion and, for
// binary rows, with selections instead of branches on the shape of the tree
// (which no branch predictor learns).  The build is most of what a tree's
// first pass takes longer than the next ones: for 5000 tips 641 us, 728 with
// recursive writers and an upload per table, 305 once the plan is there.
struct Builder {
    const ClusterTree &t;
    ClusterPlan &pl;
    struct Row {
        int size;           // rows of the subtree not in a cluster of an earlier stage
        int at;             // last step of its subtree in the postorder program, then first in the preorder program
        int16_t need;       // LDS slots that the subtree takes on the way up, inside the cluster
        int16_t base, dst;  // first slot its subtree may use, and the one its own row goes to (-1: none)
    };
    std::vector<Row> row;  // and one that children outside the cluster write to
    std::vector<int> &cluster = pl.cluster, &need_pre = pl.need_pre;

    Builder(const ClusterTree &t_, ClusterPlan &pl_) : t(t_), pl(pl_), row(t_.n_int + 1) {}
    bool binary(int r) const { return t.child_ptr[r + 1] - t.child_ptr[r] == 2; }

    // Size and slots of row r's subtree, from its children's.
    void measure(int r) {
        int size = 1, up1 = -1, up2 = -1, dn1 = -1, dn2 = -1;  // the two largest needs
        for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e) {
            const int c = t.child_ref[e];
            const bool in = c >= 0 && cluster[c] < 0;
            const int k = in ? c : 0;
            size += in ? row[k].size : 0;
            const int a = in ? row[k].need : -1, b = in ? need_pre[k] : -1;
            up2 = std::max(up2, std::min(up1, a));
            up1 = std::max(up1, a);
            dn2 = std::max(dn2, std::min(dn1, b));
            dn1 = std::max(dn1, b);
        }
        row[r].size = size;
        row[r].need = (int16_t)std::max({0, up1, binary(r) ? up2 + 1 : 0});
        need_pre[r] = std::max({0, dn1, dn2 + 1});
    }

    // Postorder step of row r, after its parent's: of a binary row's two
    // children the one that takes more slots is walked first and kept in a
    // slot while the other is walked, which is then the row just before.
    // Other rows read their children from memory.  Children whose cluster is
    // not set yet are in r's.
    void up(int r, bool root) {
        const Row q = row[r];
        const int cid = cluster[r], none = t.n_int;
        int32_t *st = &pl.post[(size_t)q.at * kClPost];
        st[0] = r;
        st[5] = q.dst + 1;
        st[6] = root ? cid : -1;
        st[7] = t.int_node[r];
        if (binary(r)) {
            const int e = t.child_ptr[r];
            const int ra = t.child_ref[e], rb = t.child_ref[e + 1];
            const int ka = std::max(ra, 0), kb = std::max(rb, 0);
            const int ca = ra >= 0 ? cluster[ka] : -1, cb = rb >= 0 ? cluster[kb] : -1;
            const bool ia = ra >= 0 && ca < 0, ib = rb >= 0 && cb < 0;
            // first: a child kept in a slot, another cluster's row or a tip; last: the child walked last
            const bool swap = ia && (!ib || row[ka].need < row[kb].need);
            const int r0 = swap ? rb : ra, r1 = swap ? ra : rb;
            const bool both = ia && ib, any = ia || ib;
            const int k0 = both ? r0 : none, k1 = any ? r1 : none;
            row[k1].at = q.at - 1;
            row[k1].base = (int16_t)(q.base + (both ? 1 : 0));
            row[k1].dst = -1;
            row[k0].at = q.at - 1 - (any ? row[k1].size : 0);
            row[k0].base = q.base;
            row[k0].dst = q.base;
            st[1] = both ? kSrcSlot | q.base : r0;
            st[2] = any ? kSrcAcc : r1;
            st[3] = t.child_node[e + (swap ? 1 : 0)];
            st[4] = t.child_node[e + (swap ? 0 : 1)];
            st[8] = both ? -1 : swap ? cb : ca;
            st[9] = any ? -1 : swap ? ca : cb;
            if (ia) cluster[ka] = cid;
            if (ib) cluster[kb] = cid;
        } else {
            st[1] = st[2] = kSrcAcc;
            st[5] |= 0x100;
            st[8] = st[9] = -1;
            int at = q.at;
            for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e) {
                const int c = t.child_ref[e];
                if (c < 0) continue;
                if (cluster[c] >= 0) {
                    pl.edge_cluster[e] = cluster[c];
                    continue;
                }
                cluster[c] = cid;
                row[c].at = at - 1;
                row[c].base = q.base;
                row[c].dst = -1;
                at -= row[c].size;
            }
        }
    }

    // Preorder step of row r, whose parent's profile is in slot dst, the row just
    // before (-1), in memory (-2) or not needed (-3: the root), and of its tips: r's own profile is the row just before for the child
    // walked first (the one that takes fewest slots) and waits in a slot for
    // the others, the last of which frees it.
    void down(int r, int tips, int32_t *out) {
        const Row q = row[r];
        const int cid = cluster[r], none = t.n_int, node = t.int_node[r];
        const int src = q.dst >= 0 ? kSrcSlot | q.dst : q.dst == -1 ? kSrcAcc : q.dst == -2 ? 0 : -1;
        int32_t *st = out + (size_t)q.at * kClPre;
        const int c0 = t.child_ptr[r], c1 = t.child_ptr[r + 1];
        int n = 0, at = q.at + 1;
        if (tips)
            for (int e = c0; e < c1; ++e)
                if (t.child_ref[e] < 0) {
                    const int x = t.child_node[e];
                    const int32_t tip[kClPre] = {x, -1, t.tip_row[x], kSrcAcc, node, -1, 0, 0};
                    std::copy(tip, tip + kClPre, out + (size_t)at++ * kClPre);
                }
        auto place = [&](int c, int dst, int base) {
            row[c].at = at;
            row[c].dst = (int16_t)dst;
            row[c].base = (int16_t)base;
            at += row[c].size;
        };
        if (c1 - c0 == 2) {
            const int ra = t.child_ref[c0], rb = t.child_ref[c0 + 1];
            const int ka = std::max(ra, 0), kb = std::max(rb, 0);
            const bool ia = ra >= 0 && cluster[ka] == cid, ib = rb >= 0 && cluster[kb] == cid;
            const bool swap = ib && (!ia || need_pre[kb] < need_pre[ka]);
            const int k0 = ia || ib ? (swap ? kb : ka) : none, k1 = ia && ib ? (swap ? ka : kb) : none;
            n = (ia ? 1 : 0) + (ib ? 1 : 0);
            place(k0, -1, q.base + (n > 1 ? 1 : 0));
            place(k1, q.base, q.base);
        } else {
            std::vector<int> kids;
            for (int e = c0; e < c1; ++e)
                if (t.child_ref[e] >= 0 && cluster[t.child_ref[e]] == cid) kids.push_back(t.child_ref[e]);
            std::stable_sort(kids.begin(), kids.end(), [&](int a, int b) { return need_pre[a] < need_pre[b]; });
            n = (int)kids.size();
            for (int i = 0; i < n; ++i) place(kids[i], i == 0 ? -1 : q.base, i + 1 < n ? q.base + 1 : q.base);
        }
        const int32_t v[kClPre] = {node, r, -1, src, std::max(0, t.parent[node]), n > 1 ? q.base : -1, 0, 0};
        std::copy(v, v + kClPre, st);
    }
};

}  // namespace

ClusterPlan build_clusters(const ClusterTree &t) {
    ClusterPlan pl;
    const long tiles = (t.P + TT_WAVE - 1) / TT_WAVE;
    const int ni = t.n_int;
    for (int r = 0; r < ni && pl.edge_cluster.empty(); ++r)
        if (t.child_ptr[r + 1] - t.child_ptr[r] != 2) pl.edge_cluster.assign(t.child_ptr[ni], -1);
    pl.post.reserve((size_t)ni * (kClPost + kClPre) + t.n_nodes);  // the caller appends a preorder program
    pl.post.resize((size_t)ni * kClPost);
    pl.cluster.assign(ni, -1);
    pl.need_pre.assign(ni, 0);
    Builder b(t, pl);
    std::vector<int> par(ni, -1), left(t.post_nodes, t.post_nodes + ni), rest, roots;  // children before parents
    for (int r = 0; r < ni; ++r) {
        const int p = t.parent[t.int_node[r]];
        if (p >= 0) par[r] = t.int_row[p];
    }
    int steps = 0;
    while (!left.empty()) {
        const int K = cluster_size((long)left.size(), tiles, t.n);
        for (int r : left) b.measure(r);
        auto size = [&](int r) { return b.row[r].size; };
        const long most = (long)left.size() / (kChain * K);  // ends, rows with none below them, of a chain
        long ends = 0;
        for (size_t i = 0; i < left.size() && ends <= most; ++i) ends += size(left[i]) == 1;
        const bool chain = ends <= most;
        const int slots = t.n > 5 ? kClusterSlots20 : kClusterSlots;
        auto in_chain = [&](int r) { return size(r) <= kChainMax && b.row[r].need <= slots && b.need_pre[r] <= slots; };
        auto in_tree = [&](int r) { return size(r) <= K; };
        roots.clear();
        rest.clear();
        // roots: rows that fit (and so do the rows below them) under one that does not
        auto find = [&](auto fits) {
            for (int r : left)
                if (fits(r) && (par[r] < 0 || !fits(par[r]))) roots.push_back(r);
        };
        auto write = [&](auto fits) {
            for (size_t i = left.size(); i-- > 0;) {
                const int r = left[i];
                if (fits(r))
                    b.up(r, par[r] < 0 || !fits(par[r]));
                else
                    rest.push_back(r);
            }
        };
        chain ? find(in_chain) : find(in_tree);
        // programs of about K nodes: the largest clusters first, filled up with the smallest
        std::stable_sort(roots.begin(), roots.end(), [&](int a, int c) { return size(a) > size(c); });
        for (size_t i = 0, j = roots.size(); i < j;) {
            ClusterPlan::Task task{};
            task.stage = pl.n_stages;
            task.post0 = steps;
            task.cluster0 = pl.n_clusters();
            auto add = [&](int r) {
                b.cluster[r] = pl.n_clusters();
                steps += size(r);
                b.row[r].at = steps - 1;
                b.row[r].base = 0;
                b.row[r].dst = -1;
                pl.roots.push_back(r);
            };
            add(roots[i++]);
            while (j > i && steps - task.post0 + size(roots[j - 1]) <= K) add(roots[--j]);
            task.post_n = steps - task.post0;
            task.cluster1 = pl.n_clusters();
            pl.tasks.push_back(task);
        }
        chain ? write(in_chain) : write(in_tree);
        std::reverse(rest.begin(), rest.end());
        left.swap(rest);
        ++pl.n_stages;
    }
    pl.n_tasks = (int)pl.tasks.size();
    return pl;
}

void build_down(const ClusterTree &t, ClusterPlan &pl, int tips, std::vector<int32_t> &out) {
    const size_t first = out.size();
    const int ni = t.n_int;
    out.resize(first + (size_t)(tips ? t.n_nodes : ni) * kClPre);
    Builder b(t, pl);
    for (int i = 0; i < ni; ++i) {  // steps of the subtrees inside their clusters
        const int r = t.post_nodes[i];
        int size = 1;
        for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e) {
            const int c = t.child_ref[e], k = std::max(c, 0);
            size += c < 0 ? tips : pl.cluster[k] == pl.cluster[r] ? b.row[k].size : 0;
        }
        b.row[r].size = size;
    }
    int steps = 0;
    for (ClusterPlan::Task &task : pl.tasks) {
        task.pre0[tips] = steps;
        for (int c = task.cluster0; c < task.cluster1; ++c) {
            Builder::Row &q = b.row[pl.roots[c]];
            q.at = steps;
            q.base = 0;
            q.dst = t.parent[t.int_node[pl.roots[c]]] < 0 ? -3 : -2;
            steps += q.size;
        }
        task.pre_n[tips] = steps - task.pre0[tips];
    }
    for (int i = ni; i-- > 0;) b.down(t.post_nodes[i], tips, &out[first]);
}

void ClusterPlan::items(ClusterRole role, int m, int what, int tips, int tree, int P,
                        std::vector<ClusterItem> &out) const {
    const int groups = (P + 4 * TT_WAVE - 1) / (4 * TT_WAVE), tiles = (P + TT_WAVE - 1) / TT_WAVE;
    const bool joint = what == kClJoint || what == kClFromRoot;
    auto one = [&](int kind, int group) { out.push_back({tree, kind, group, 0, 0, 0, 0, 0}); };
    int stage = -1, kind = kClUp;
    if (role == kRoleLeaf) {
        if (n_stages > 1) stage = 0;
    } else if (role == kRoleMid) {
        const int top = n_stages - 1;
        if (n_stages == 1 ? m == 1 : m <= mids()) {
            stage = n_stages == 1 ? 0 : m <= top ? m : 2 * top - m;
            kind = stage == top ? kClTop : m < top ? kClUp : kClDown;
        }
    } else if (role == kRoleDown) {
        if (!joint) one(kClTotal, 0);
        if (n_stages > 1 && what != kClLoglik) stage = 0, kind = kClDown;
    } else if (role == kRoleTable) {
        for (int g = 0; g * kTableTips < table_tips; ++g) one(kClTable, g);
    } else if (role == kRoleFinal) {
        for (int g = 0; g < tiles; ++g) one(kClFinal, g);
    } else {
        one(kClTotal, 0);
    }
    if (stage < 0 || (kind == kClDown && what == kClLoglik) || (kind == kClUp && what == kClFromRoot)) return;
    for (int k = 0; k < n_tasks; ++k) {
        const Task &q = tasks[k];
        if (q.stage != stage) continue;
        for (int g = 0; g < groups; ++g)
            out.push_back({tree, kind, g, k, q.post0, q.post_n, q.pre0[tips], q.pre_n[tips]});
    }
}

void ClusterLaunches::build(const std::vector<Tree> &trees, int what, int tips) {
    items.clear();
    off.assign(1, 0);
    role.clear();
    int mids = 0;
    for (const Tree &t : trees) mids = std::max(mids, t.plan->mids());
    auto launch = [&](ClusterRole r, int m) {
        for (const Tree &t : trees) t.plan->items(r, m, what, tips, t.index, t.P, items);
        if ((int)items.size() == off.back()) return;
        off.push_back((int)items.size());
        role.push_back(r);
    };
    if (what == kClMarginal || what == kClLoglik) launch(kRoleTable, 0);
    launch(kRoleLeaf, 0);
    for (int m = 1; m <= mids; ++m) launch(kRoleMid, m);
    launch(kRoleDown, 0);
    if (what == kClJoint || what == kClFromRoot) {
        launch(kRoleFinal, 0);
        launch(kRoleTotal, 0);
    }
}
