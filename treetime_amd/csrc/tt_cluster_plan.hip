// Cutting a tree into clusters and writing their step programs (host code).
#include "tt_cluster.h"

#include <algorithm>
#include <utility>

// Cluster size.  A stage is one launch: its waves each walk about K nodes, and
// what is left of the tree shrinks about K-fold.  Where a stage has work for
// the whole chip (rows x 64-pattern tiles above 4096 wave programs of 64
// nodes), long programs save launches and rows that go through memory between
// stages; where it has not, a launch costs about as much as ten steps, and
// programs of 16 keep the chain of steps short.
static int cluster_size(long rows, long tiles) {
    return (int)std::max(16L, std::min((long)kClusterMax, rows * tiles / 4096));
}

namespace {

// Writes the programs of one cluster at a time.
struct Builder {
    const ClusterTree &t;
    ClusterPlan &pl;
    std::vector<int> &cluster = pl.cluster, &need_pre = pl.need_pre;
    std::vector<int> need;  // LDS slots that a row's subtree takes on the way up, inside the cluster
    std::vector<int> order;
    int cid = -1, root = -1;

    Builder(const ClusterTree &t_, ClusterPlan &pl_) : t(t_), pl(pl_) {}
    bool binary(int r) const { return t.child_ptr[r + 1] - t.child_ptr[r] == 2; }
    bool inside(int e) const { return t.child_ref[e] >= 0 && cluster[t.child_ref[e]] == cid; }
    // children of r in the cluster, by the slots they take
    template <class Less>
    std::vector<int> children(int r, Less less) const {
        std::vector<int> c;
        for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e)
            if (inside(e)) c.push_back(t.child_ref[e]);
        std::stable_sort(c.begin(), c.end(), less);
        return c;
    }

    // Postorder steps of the subtree of r, slots from base on; r's row goes to
    // slot dst as well (-1: no).  Of a binary row's two children the one that
    // takes more slots is walked first and kept in a slot while the other is
    // walked, which is then the row just before.  Other rows read their
    // children from memory.
    void up(int r, int base, int dst) {
        int32_t st[kClPost] = {r, kSrcAcc, kSrcAcc, 0, 0, dst + 1, r == root ? cid : -1, t.int_node[r], -1, -1, 0, 0};
        if (binary(r)) {
            int e[2] = {t.child_ptr[r], t.child_ptr[r] + 1};
            // e[1]: the child walked last; e[0]: a child kept in a slot, another cluster's row or a tip
            const bool in0 = inside(e[0]), in1 = inside(e[1]);
            if (in0 && (!in1 || need[t.child_ref[e[0]]] < need[t.child_ref[e[1]]])) std::swap(e[0], e[1]);
            if (in0 && in1) up(t.child_ref[e[0]], base, base);
            if (in0 || in1) up(t.child_ref[e[1]], base + (in0 && in1 ? 1 : 0), -1);
            for (int k = 0; k < 2; ++k) {
                const int ref = t.child_ref[e[k]];
                st[1 + k] = inside(e[k]) ? (k == 1 ? kSrcAcc : kSrcSlot | base) : ref;
                st[3 + k] = t.child_node[e[k]];
                if (ref >= 0 && !inside(e[k])) st[8 + k] = cluster[ref];
            }
        } else {
            st[5] |= 0x100;
            for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e)
                if (inside(e))
                    up(t.child_ref[e], base, -1);
                else if (t.child_ref[e] >= 0)
                    pl.edge_cluster[e] = cluster[t.child_ref[e]];
        }
        pl.post.insert(pl.post.end(), st, st + kClPost);
    }

    // Preorder steps of the subtree of r, whose parent's profile is at src:
    // r's own profile is the row just before for the child walked first (the
    // one that takes fewest slots) and waits in a slot for the others.
    void down(int r, int src, int base, int tips) {
        const int node = t.int_node[r];
        std::vector<int32_t> &out = pl.pre[tips];
        int kids[2], n = 0;
        std::vector<int> many;
        const int *c = kids;
        if (binary(r)) {
            for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e)
                if (inside(e)) kids[n++] = t.child_ref[e];
            if (n == 2 && need_pre[kids[1]] < need_pre[kids[0]]) std::swap(kids[0], kids[1]);
        } else {
            many = children(r, [&](int a, int b) { return need_pre[a] < need_pre[b]; });
            c = many.data();
            n = (int)many.size();
        }
        const int32_t st[kClPre] = {node, r, -1, src, std::max(0, t.parent[node]), n > 1 ? base : -1, 0, 0};
        out.insert(out.end(), st, st + kClPre);
        if (tips)
            for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e)
                if (t.child_ref[e] < 0) {
                    const int x = t.child_node[e];
                    const int32_t tip[kClPre] = {x, -1, t.tip_row[x], kSrcAcc, node, -1, 0, 0};
                    out.insert(out.end(), tip, tip + kClPre);
                }
        for (int i = 0; i < n; ++i)  // the last child reads the slot, after which it is free
            down(c[i], i == 0 ? kSrcAcc : kSrcSlot | base, n > 1 && i + 1 < n ? base + 1 : base, tips);
    }

    void write(int root_row) {
        root = root_row;
        cid = pl.n_clusters();
        pl.roots.push_back(root);
        order.assign(1, root);
        for (size_t i = 0; i < order.size(); ++i) {  // parents before children
            const int r = order[i];
            cluster[r] = cid;
            for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e)
                if (t.child_ref[e] >= 0 && cluster[t.child_ref[e]] < 0) order.push_back(t.child_ref[e]);
        }
        for (size_t i = order.size(); i-- > 0;) {
            const int r = order[i];
            int up1 = -1, up2 = -1, dn1 = -1, dn2 = -1;  // the two largest needs of the children
            for (int e = t.child_ptr[r]; e < t.child_ptr[r + 1]; ++e) {
                if (!inside(e)) continue;
                const int a = need[t.child_ref[e]], b = need_pre[t.child_ref[e]];
                up2 = std::max(up2, std::min(up1, a));
                up1 = std::max(up1, a);
                dn2 = std::max(dn2, std::min(dn1, b));
                dn1 = std::max(dn1, b);
            }
            need[r] = std::max({0, up1, binary(r) ? up2 + 1 : 0});
            need_pre[r] = std::max({0, dn1, dn2 + 1});
        }
        up(root, 0, -1);
    }
};

}  // namespace

ClusterPlan build_clusters(const ClusterTree &t) {
    ClusterPlan pl;
    const long tiles = (t.P + TT_WAVE - 1) / TT_WAVE;
    const int ni = t.n_int;
    for (int r = 0; r < ni && pl.edge_cluster.empty(); ++r)
        if (t.child_ptr[r + 1] - t.child_ptr[r] != 2) pl.edge_cluster.assign(t.child_ptr[ni], -1);
    pl.post.reserve((size_t)ni * kClPost);
    pl.cluster.assign(ni, -1);
    pl.need_pre.assign(ni, 0);
    Builder b(t, pl);
    b.need.assign(ni, 0);
    std::vector<int> par(ni, -1), size(ni);  // parent's row; rows of the subtree not yet in a cluster
    for (int r = 0; r < ni; ++r) {
        const int p = t.parent[t.int_node[r]];
        if (p >= 0) par[r] = t.int_row[p];
    }
    std::vector<int> left(t.post_nodes, t.post_nodes + ni), rest, roots;  // children before parents
    while (!left.empty()) {
        const int K = cluster_size((long)left.size(), tiles);
        for (int r : left) size[r] = 1;
        for (int r : left)
            if (par[r] >= 0) size[par[r]] += size[r];
        roots.clear();
        for (int r : left)
            if (size[r] <= K && (par[r] < 0 || size[par[r]] > K)) roots.push_back(r);
        // programs of about K nodes: the largest clusters first, filled up with the smallest
        std::stable_sort(roots.begin(), roots.end(), [&](int a, int c) { return size[a] > size[c]; });
        for (size_t i = 0, j = roots.size(); i < j;) {
            ClusterPlan::Task task{};
            task.stage = pl.n_stages;
            task.post0 = (int)(pl.post.size() / kClPost);
            task.cluster0 = pl.n_clusters();
            int sum = size[roots[i]];
            b.write(roots[i++]);
            while (j > i && sum + size[roots[j - 1]] <= K) {
                sum += size[roots[--j]];
                b.write(roots[j]);
            }
            task.post_n = (int)(pl.post.size() / kClPost) - task.post0;
            task.cluster1 = pl.n_clusters();
            pl.tasks.push_back(task);
        }
        rest.clear();
        for (int r : left)
            if (b.cluster[r] < 0) rest.push_back(r);
        left.swap(rest);
        ++pl.n_stages;
    }
    pl.n_tasks = (int)pl.tasks.size();
    return pl;
}

void build_down(const ClusterTree &t, ClusterPlan &pl, int tips) {
    if (!pl.pre[tips].empty()) return;
    pl.pre[tips].reserve((size_t)(tips ? t.n_nodes : t.n_int) * kClPre);
    Builder b(t, pl);
    for (ClusterPlan::Task &task : pl.tasks) {
        task.pre0[tips] = (int)(pl.pre[tips].size() / kClPre);
        for (b.cid = task.cluster0; b.cid < task.cluster1; ++b.cid) {
            const int root = pl.roots[b.cid];
            b.down(root, t.parent[t.int_node[root]] < 0 ? -1 : 0, 0, tips);
        }
        task.pre_n[tips] = (int)(pl.pre[tips].size() / kClPre) - task.pre0[tips];
    }
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
    launch(kRoleLeaf, 0);
    for (int m = 1; m <= mids; ++m) launch(kRoleMid, m);
    launch(kRoleDown, 0);
    if (what == kClJoint || what == kClFromRoot) {
        launch(kRoleFinal, 0);
        launch(kRoleTotal, 0);
    }
}
