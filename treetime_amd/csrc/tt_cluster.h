// Host schedule of the clustered passes (tt_cluster.hip): a tree cut into
// connected clusters of internal nodes, each walked by one wave for 64
// patterns, in a few launches instead of one per level.
#pragma once
#include <stdint.h>

#include <vector>

#include "tt_common.h"

// Sources of a child's row in a postorder step and of the parent's profile in
// a preorder step: < 0 a tip (row -src - 1); below kSrcSlot a row of an
// earlier launch, read from memory; the wave's LDS slot src & 0xff; or the
// row of the step just before, still in registers.
constexpr int kSrcSlot = 0x20000000;
constexpr int kSrcAcc = 0x40000000;
// LDS slots of a wave, up to 5 states and for 20: k rows wait at once only in a
// cluster of at least 2^(k + 1) - 1 nodes
constexpr int kClusterSlots = 5;
constexpr int kClusterSlots20 = 2;
constexpr int kClusterMax = 64;
// postorder step: {row, src0, src1, node0, node1, slot written + 1 (0: none) with bit 8 set for a row that has not two
//                  children, cluster ended or -1, node id, clusters of src0 and src1 or -1, 0, 0}
constexpr int kClPost = 12;
// preorder step: {node, internal row or -1, tip row or -1, parent's source, parent's node, slot written or -1, 0, 0}
constexpr int kClPre = 8;

// Passes: from-root is the joint pass's way down from given root states.
enum ClusterPass { kClMarginal = 0, kClLoglik = 1, kClJoint = 2, kClFromRoot = 3 };
// What a workgroup of four waves does: a task's steps for patterns [256 group,
// 256 (group + 1)), up, down or both at the root; the joint log-likelihood of
// patterns [64 group, 64 (group + 1)); the tree's total; the tables of tips
// [kTableTips group, kTableTips (group + 1)).
enum ClusterKind { kClUp = 0, kClTop = 1, kClDown = 2, kClFinal = 3, kClTotal = 4, kClTable = 5 };
// Kernels: the leaf stage up, anything in between, the leaf stage down, the
// joint log-likelihood per pattern, the total (after a joint pass), the tips'
// tables (before a marginal pass of 20 states).
enum ClusterRole { kRoleLeaf = 0, kRoleMid = 1, kRoleDown = 2, kRoleFinal = 3, kRoleTotal = 4, kRoleTable = 5 };
constexpr int kTableTips = 4;
struct ClusterItem {
    int32_t tree, kind, group, task;  // task: row of the joint score partials
    int32_t post0, post_n;            // postorder steps
    int32_t pre0, pre_n;              // preorder steps
};

struct ClusterPlan {
    int n_tasks = 0, n_stages = 0;
    int table_tips = 0;  // tips with tables
    std::vector<int32_t> post, edge_cluster;  // postorder program; cluster of every child edge of a non-binary row
    std::vector<int> cluster, need_pre, roots;        // cluster of every row, its slots going down; root of every cluster
    struct Task {
        int stage, post0, post_n, pre0[2], pre_n[2], cluster0, cluster1;
    };
    std::vector<Task> tasks;  // by stage; the last holds the root's cluster
    int n_clusters() const { return (int)roots.size(); }
    // A pass's launches: first the leaf stage's tasks going up, then mids()
    // ones (the other stages up, the root's cluster both ways, the stages
    // down again, but for the leaf stage), then the leaf stage down.  Several
    // trees share launches: a tree's m-th one in the batch's m-th, all leaf
    // stages going down in the last.
    int mids() const { return n_stages == 1 ? 1 : 2 * n_stages - 3; }
    void items(ClusterRole role, int m, int what, int tips, int tree, int P, std::vector<ClusterItem> &out) const;
};

// A pass over one tree or several: items of launch l at [off[l], off[l + 1]).
struct ClusterLaunches {
    std::vector<ClusterItem> items;
    std::vector<int> off;
    std::vector<ClusterRole> role;
    // trees: (index, plan, patterns), in the order their items are listed
    struct Tree {
        int index;
        const ClusterPlan *plan;
        int P;
    };
    void build(const std::vector<Tree> &trees, int what, int tips);
};

struct ClusterTree {
    int n_nodes, n_int, root, P, n;
    const int32_t *parent, *int_row, *tip_row, *int_node, *child_ptr, *child_ref, *child_node;
    const int32_t *post_nodes;  // internal rows, children before parents
};
ClusterPlan build_clusters(const ClusterTree &t);                     // clusters and postorder programs
// preorder program without (0) / with (1) the tips, appended to out
void build_down(const ClusterTree &t, ClusterPlan &pl, int tips, std::vector<int32_t> &out);

// Device side of a plan.
struct ClusterDev {
    const int32_t TT_C *post;
    const int32_t TT_C *pre[2];
    const int32_t TT_C *edge_cluster;
    double TT_G *part;    // [n_clusters][P] log normalisers of the clusters' subtrees
    double TT_G *score;   // [n_tasks][P] joint score of a task's branches
    double TT_G *bpart;   // [groups of 64 patterns] sum of mult * logL
    double *out;          // batch: the tree's log-likelihood
    const int32_t TT_C *tip_nodes;  // [n_tips]
    int32_t n_tasks;
};

namespace ttk {
bool cluster_states(int n, bool joint);  // alphabets with clustered passes
// one launch of a pass (ClusterPass) over one tree's items, or over a batch's
hipError_t cluster_launch(const TreeDev &T, const ClusterDev &C, const ClusterItem *items, int n_items, ClusterRole role,
                          int what, bool tips, hipStream_t s);
hipError_t pool_launch(int n, const BatchTreeDev *trees, const ClusterDev *cl, const ClusterItem *items, int n_items,
                       ClusterRole role, int what, bool tips, hipStream_t s);
}  // namespace ttk
