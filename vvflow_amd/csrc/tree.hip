// tree.hip -- the adaptive binary tree of TSortedTree.cpp rebuilt
// level-synchronously on the GPU.
//
// stree::build (TSortedTree.cpp:232-265) splits nodes recursively at the
// centre of their tight bounding box with an in-place Hoare partition
// (DistributeContent, :81-99).  That partition pairs the k-th element left
// of the split position that belongs right with the k-th element right of
// it, counted from the end, that belongs left; everything else stays.  Each
// level is therefore replayed exactly with one exclusive scan of the
// "goes left" flags: misplaced elements get their rank on their side and
// swap with the partner of complementary rank.  Bounding boxes are exact
// FP64 min/max (atomics on an order-preserving integer image), so node
// centres, leaf decisions and the resulting permutation are bit-identical to
// the reference.  Segments (body panels) follow a stable partition
// (:139-148), i.e. each segment descends like findNode and keeps its order.
// The heat and streak lists (hRange, sRange) are partitioned the same way
// as the vortex list, each in place within its own range: the elements of
// the build are the vortices, then the heat particles, then the streak
// particles, and every node holds one range per list.
//
// The levels run over the whole list only while nodes are large: a node with
// at most kSubElems elements and kSubSegs segments is taken by one workgroup,
// which builds its whole subtree in LDS (k_subtree).  Node ids of the levels
// over the whole list are contiguous per level (TreeArrays::levels), those of
// a subtree contiguous per level of the subtree (sub_lev).  After the build,
// subtree leaf counts and monopoles (CalculateCMass, :150-197) go bottom-up
// and leaf DFS ranks (the bottomNodes order) top-down, one workgroup per
// subtree and one for the levels above; and the near/far lists of every leaf
// (FindNearNodes, :199-217) come from walks of waves of 64 DFS-consecutive
// leaves.

#include "common.hpp"

#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <algorithm>
#include <array>
#include <cmath>
#include <functional>

#pragma clang fp contract(off)

namespace vvhd {
namespace {

constexpr int kBlock = 256;

inline int nblocks(int64_t n, int b = kBlock) { return (int)std::max<int64_t>(1, (n + b - 1) / b); }

// --------------------------------------------------------------- kernels --

struct NodeView {
    double *x, *y, *h, *w;
    uint64_t *blx, *bly, *trx, *try_;
    int32_t *v0, *v1, *ch1, *parent, *depth, *nseg, *split;
    uint64_t* path;
    int32_t *h0, *h1, *s0, *s1;
};

NodeView view(TreeArrays& t) {
    return NodeView{t.x.p,  t.y.p,   t.h.p,      t.w.p,     t.blx.p,   t.bly.p,  t.trx.p,   t.try_.p,
                    t.v0.p, t.v1.p,  t.ch1.p,    t.parent.p, t.depth.p, t.nseg.p, t.split.p, t.path.p,
                    t.h0.p, t.h1.p,  t.s0.p,     t.s1.p};
}

// List of element k: 0 vortex, 1 heat, 2 streak.
__device__ inline int elem_list(int k, int hbase, int sbase) { return k < hbase ? 0 : (k < sbase ? 1 : 2); }

// A node's range of list cls.
__device__ inline void list_range(const NodeView& nv, int node, int cls, int& r0, int& r1) {
    if (cls == 0) {
        r0 = nv.v0[node];
        r1 = nv.v1[node];
    } else if (cls == 1) {
        r0 = nv.h0[node];
        r1 = nv.h1[node];
    } else {
        r0 = nv.s0[node];
        r1 = nv.s1[node];
    }
}

__device__ inline void set_list_range(const NodeView& nv, int node, int cls, int r0, int r1) {
    int32_t* a = cls == 0 ? nv.v0 : (cls == 1 ? nv.h0 : nv.s0);
    int32_t* b = cls == 0 ? nv.v1 : (cls == 1 ? nv.h1 : nv.s1);
    a[node] = r0;
    b[node] = r1;
}

__device__ inline void init_node(NodeView nv, int id, int parent, int depth, uint64_t path, int v0, int v1, int h0,
                                 int h1, int s0, int s1) {
    nv.parent[id] = parent;
    nv.depth[id] = depth;
    nv.path[id] = path;
    nv.v0[id] = v0;
    nv.v1[id] = v1;
    nv.h0[id] = h0;
    nv.h1[id] = h1;
    nv.s0[id] = s0;
    nv.s1[id] = s1;
    nv.ch1[id] = -1;
    nv.nseg[id] = 0;
    nv.split[id] = 0;
    nv.blx[id] = ord_from_double(DBL_MAX);
    nv.bly[id] = ord_from_double(DBL_MAX);
    nv.trx[id] = ord_from_double(-DBL_MAX);
    nv.try_[id] = ord_from_double(-DBL_MAX);
}

// One root per simulation: root s holds the vortices [sim_off[s], sim_off[s+1]).
// The heat elements [hbase, sbase) and streak elements [sbase, nelem) belong
// to root 0 (one simulation only).
__global__ void k_init_roots(NodeView nv, int nroots, const int64_t* sim_off, int32_t* counters, int2* lev, int hbase,
                             int sbase, int nelem) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nroots) {
        if (s == 0)
            init_node(nv, s, -1, 0, 0, (int)sim_off[s], (int)sim_off[s + 1], hbase, sbase, sbase, nelem);
        else
            init_node(nv, s, -1, 0, 0, (int)sim_off[s], (int)sim_off[s + 1], nelem, nelem, nelem, nelem);
    }
    if (s == 0) {
        counters[0] = nroots;   // nodes
        counters[1] = 0;        // leaves
        counters[2] = 0;        // level begin
        counters[3] = nroots;   // level end
        counters[4] = 0;        // 1: node capacity exceeded, 2: tree too deep
        counters[5] = 0;        // max depth
        counters[6] = 0;        // nodes of the level that k_subtree left
        counters[7] = 0;        // subtrees
        counters[8] = 0;        // nodes of the level handed to k_subtree
        counters[9] = nroots;   // first id of the next level
        lev[0] = make_int2(0, nroots);
    }
}

// Element -> root (its simulation).
__global__ void k_fill_roots(int32_t* enode, int n, const int64_t* sim_off, int nroots) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int lo = 0, hi = nroots - 1;   // last root whose offset <= k
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sim_off[mid] <= k)
            lo = mid;
        else
            hi = mid - 1;
    }
    enode[k] = lo;
}

// Adds 1 to count[node] for every active lane, a claim for all lanes of a node:
// a counter takes one every 12 ns or so, and neighbouring segments share theirs.
// Called by all lanes of the wave.
__device__ inline void count_wave(int32_t* count, int node, bool active) {
    for (uint64_t left = __ballot(active); left;) {
        const int lead = __builtin_amdgcn_readlane(node, (int)__builtin_ctzll(left));
        const uint64_t same = __ballot(active && node == lead);
        if (lane_id() == (int)__builtin_ctzll(left)) atomicAdd(&count[lead], (int)__popcll(same));
        left &= ~same;
    }
}

// Segments start at the root of their body's simulation.
__global__ void k_seg_roots(NodeView nv, const int32_t* seg_root, int nseg, int32_t* seg_node) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = i < nseg ? seg_root[i] : 0;
    if (i < nseg) seg_node[i] = r;
    count_wave(nv.nseg, r, i < nseg);
}

// Adds a point to a node's bounding box; NaN coordinates are ignored, as by
// std::max/std::min in Stretch.
__device__ inline void bbox_add(NodeView nv, int node, double px, double py) {
    if (!isnan(px)) {
        atomicMin((unsigned long long*)&nv.blx[node], (unsigned long long)ord_from_double(px));
        atomicMax((unsigned long long*)&nv.trx[node], (unsigned long long)ord_from_double(px));
    }
    if (!isnan(py)) {
        atomicMin((unsigned long long*)&nv.bly[node], (unsigned long long)ord_from_double(py));
        atomicMax((unsigned long long*)&nv.try_[node], (unsigned long long)ord_from_double(py));
    }
}

// Wave-aggregated bbox update: lanes targeting the same node reduce first and
// one lane performs the atomics, for up to four distinct nodes per wave; the
// rest fall back to per-lane atomics.  Called by all lanes of the wave.
__device__ inline void bbox_add_wave(NodeView nv, int node, double px, double py, bool active) {
    uint64_t left = __ballot(active);
    for (int round = 0; round < 4 && left; round++) {
        const int leader = (int)__builtin_ctzll(left);
        const int lead_node = __shfl(node, leader, kWave);
        const bool mine = active && ((left >> lane_id()) & 1ull) && node == lead_node;
        const uint64_t m_same = __ballot(mine);
        const bool vx = mine && !isnan(px), vy = mine && !isnan(py);
        double lx = vx ? px : DBL_MAX, hx = vx ? px : -DBL_MAX;
        double ly = vy ? py : DBL_MAX, hy = vy ? py : -DBL_MAX;
        for (int o = kWave / 2; o > 0; o >>= 1) {
            lx = fmin(lx, __shfl_xor(lx, o, kWave));
            hx = fmax(hx, __shfl_xor(hx, o, kWave));
            ly = fmin(ly, __shfl_xor(ly, o, kWave));
            hy = fmax(hy, __shfl_xor(hy, o, kWave));
        }
        if (lane_id() == leader) {
            if (lx <= hx) {
                atomicMin((unsigned long long*)&nv.blx[lead_node], (unsigned long long)ord_from_double(lx));
                atomicMax((unsigned long long*)&nv.trx[lead_node], (unsigned long long)ord_from_double(hx));
            }
            if (ly <= hy) {
                atomicMin((unsigned long long*)&nv.bly[lead_node], (unsigned long long)ord_from_double(ly));
                atomicMax((unsigned long long*)&nv.try_[lead_node], (unsigned long long)ord_from_double(hy));
            }
        }
        left &= ~m_same;
    }
    if (active && ((left >> lane_id()) & 1ull)) bbox_add(nv, node, px, py);
}

// Bounding boxes of the nodes of a level with at most kTopNodes nodes (the
// root, and the children of the first levels), from the elements in their
// final positions: every element k with enode[k] - base in [0, kTopNodes)
// adds to that node.  A node's elements form one contiguous range, so each
// thread keeps a running box for the node of its current element (order-
// preserving integer images, NaN coordinates skipped) and adds it to the
// block's LDS slot of that node only when the node changes; one lane per
// block and node then issues the global atomics.  Each block covers
// kTopChunk consecutive elements, kTopPer per thread, loaded before use.
constexpr int kTopNodes = 512;
constexpr int kTopPer = 4;
constexpr int kTopChunk = kBlock * kTopPer;

__global__ __launch_bounds__(kBlock) void k_bbox_top(NodeView nv, const int32_t* base_ptr, const int32_t* enode,
                                                     const double* x, const double* y, int n) {
    __shared__ unsigned long long s_lx[kTopNodes], s_ly[kTopNodes], s_hx[kTopNodes], s_hy[kTopNodes];
    const unsigned long long lo0 = ord_from_double(DBL_MAX), hi0 = ord_from_double(-DBL_MAX);
    for (int t = threadIdx.x; t < kTopNodes; t += blockDim.x) {
        s_lx[t] = lo0;
        s_ly[t] = lo0;
        s_hx[t] = hi0;
        s_hy[t] = hi0;
    }
    __syncthreads();
    const int base = base_ptr ? *base_ptr : 0;
    const int k0 = blockIdx.x * kTopChunk + threadIdx.x;
    int nodes[kTopPer];
    double px[kTopPer], py[kTopPer];
#pragma unroll
    for (int j = 0; j < kTopPer; j++) {
        const int k = k0 + j * kBlock;
        nodes[j] = -1;
        if (k < n) {
            nodes[j] = (enode ? enode[k] : 0) - base;
            px[j] = x[k];
            py[j] = y[k];
        }
    }
    int cur = -1;
    unsigned long long lx = lo0, hx = hi0, ly = lo0, hy = hi0;
    auto flush = [&]() {
        if (cur < 0) return;
        if (lx != lo0) atomicMin(&s_lx[cur], lx);
        if (hx != hi0) atomicMax(&s_hx[cur], hx);
        if (ly != lo0) atomicMin(&s_ly[cur], ly);
        if (hy != hi0) atomicMax(&s_hy[cur], hy);
    };
#pragma unroll
    for (int j = 0; j < kTopPer; j++) {
        const int node = nodes[j];
        if (node < 0 || node >= kTopNodes) continue;
        if (node != cur) {
            flush();
            cur = node;
            lx = ly = lo0;
            hx = hy = hi0;
        }
        if (!isnan(px[j])) {
            const unsigned long long o = ord_from_double(px[j]);
            lx = o < lx ? o : lx;
            hx = o > hx ? o : hx;
        }
        if (!isnan(py[j])) {
            const unsigned long long o = ord_from_double(py[j]);
            ly = o < ly ? o : ly;
            hy = o > hy ? o : hy;
        }
    }
    flush();
    __syncthreads();
    for (int t = threadIdx.x; t < kTopNodes; t += blockDim.x) {
        const int id = base + t;
        if (s_lx[t] != lo0) atomicMin((unsigned long long*)&nv.blx[id], s_lx[t]);
        if (s_hx[t] != hi0) atomicMax((unsigned long long*)&nv.trx[id], s_hx[t]);
        if (s_ly[t] != lo0) atomicMin((unsigned long long*)&nv.bly[id], s_ly[t]);
        if (s_hy[t] != hi0) atomicMax((unsigned long long*)&nv.try_[id], s_hy[t]);
    }
}

// Bounding boxes of a new level's nodes once k_swap has put every element in
// place: a node's elements are then the range [v0, v1), so LPN lanes per
// node (64, or 16 when nodes are small) reduce it (order-preserving integer
// images, NaN coordinates skipped, as the atomics do) without contending
// with the other nodes; segments add their atomics afterwards.
template <int LPN>
__global__ void k_child_boxes(NodeView nv, const int32_t* counters, const double* x, const double* y) {
    const int lb = counters[2], le = counters[3];
    constexpr int kPer = kWave / LPN;   // nodes per wave
    const int slots = gridDim.x * (blockDim.x / kWave) * kPer;
    const int sub = lane_id() % LPN;
    const uint64_t lo0 = ord_from_double(DBL_MAX), hi0 = ord_from_double(-DBL_MAX);
    const int first = lb + (blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) * kPer + lane_id() / LPN;
    for (int base = lb; base < le; base += slots) {   // uniform trip count: shuffles stay converged
        const int id = first + (base - lb);
        const bool ok = id < le;
        uint64_t lx = lo0, hx = hi0, ly = lo0, hy = hi0;
        for (int cls = 0; cls < 3; cls++) {
            int r0 = 0, r1 = 0;
            if (ok) list_range(nv, id, cls, r0, r1);
            for (int k = r0 + sub; k < r1; k += LPN) {
                const double px = x[k], py = y[k];
                if (!isnan(px)) {
                    const uint64_t o = ord_from_double(px);
                    lx = o < lx ? o : lx;
                    hx = o > hx ? o : hx;
                }
                if (!isnan(py)) {
                    const uint64_t o = ord_from_double(py);
                    ly = o < ly ? o : ly;
                    hy = o > hy ? o : hy;
                }
            }
        }
        for (int o = LPN / 2; o > 0; o >>= 1) {
            const uint64_t a = __shfl_xor(lx, o, kWave), b = __shfl_xor(hx, o, kWave);
            const uint64_t c = __shfl_xor(ly, o, kWave), d = __shfl_xor(hy, o, kWave);
            lx = a < lx ? a : lx;
            hx = b > hx ? b : hx;
            ly = c < ly ? c : ly;
            hy = d > hy ? d : hy;
        }
        if (ok && sub == 0) {
            if (lx != lo0) atomicMin((unsigned long long*)&nv.blx[id], (unsigned long long)lx);
            if (hx != hi0) atomicMax((unsigned long long*)&nv.trx[id], (unsigned long long)hx);
            if (ly != lo0) atomicMin((unsigned long long*)&nv.bly[id], (unsigned long long)ly);
            if (hy != hi0) atomicMax((unsigned long long*)&nv.try_[id], (unsigned long long)hy);
        }
    }
}

// Adds the lanes' segments to their nodes: counts and boxes.  Most nodes' boxes
// hold them already, with their vortices': those need no claim.
__device__ inline void add_segs_wave(NodeView nv, int node, double px, double py, bool active) {
    count_wave(nv.nseg, node, active);
    const bool in = active && ord_from_double(px) >= nv.blx[node] && ord_from_double(px) <= nv.trx[node] &&
                    ord_from_double(py) >= nv.bly[node] && ord_from_double(py) <= nv.try_[node];
    bbox_add_wave(nv, node, px, py, active && !in);
}

// Segments of the root bounding boxes.
__global__ void k_root_segs(NodeView nv, const vvhd_seg* segs, const int32_t* seg_root, int nseg) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = i < nseg;
    bbox_add_wave(nv, on ? seg_root[i] : 0, on ? segs[i].x : 0, on ? segs[i].y : 0, on);
}

// Root bounding boxes when there are more roots than k_bbox_top handles.
__global__ void k_bbox_elems(NodeView nv, const int32_t* enode, const double* x, const double* y, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const bool a = k < n;
    bbox_add_wave(nv, a ? enode[k] : 0, a ? x[k] : 0, a ? y[k] : 0, a);
}

// First leaf (DFS rank) of every root, from the subtree leaf counts.
// First leaf of every root and its preorder position: a tree of k leaves
// has 2k - 1 nodes, so root s starts at 2 first - s.
__global__ void k_root_first(const int32_t* nleaves, int nroots, int32_t* first, int32_t* root_first,
                             int32_t* pre) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    int f = 0;
    for (int s = 0; s < nroots; s++) {
        first[s] = f;
        root_first[s] = f;
        pre[s] = 2 * f - s;
        f += nleaves[s];
    }
    root_first[nroots] = f;
}

// Leaf -> simulation.
__global__ void k_leaf_sim(const int32_t* root_first, int nroots, int nleaf, int32_t* leaf_sim) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nleaf) return;
    int lo = 0, hi = nroots - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (root_first[mid] <= l)
            lo = mid;
        else
            hi = mid - 1;
    }
    leaf_sim[l] = lo;
}

// snode::Stretch tail + DivideNode decision (TSortedTree.cpp:36-56, 122-125)
// for the nodes of the current level; split nodes get a pair of children.
__global__ void k_decide(NodeView nv, int32_t* counters, int cap, double min_node, double max_node) {
    const int lb = counters[2], le = counters[3];
    const int lane = lane_id();
    const uint64_t below = (1ull << lane) - 1;
    // whole waves step through the level, so the counters are claimed once
    // per wave (leaf slots, pairs of child ids) and lanes take their ranks
    const int stride = gridDim.x * blockDim.x;
    for (int b0 = lb + blockIdx.x * blockDim.x + threadIdx.x - lane; b0 < le; b0 += stride) {
        const int id = b0 + lane;
        const bool valid = id < le && nv.split[id] == 0;   // not taken as a subtree
        bool leaf = false;
        int depth = 0;
        if (valid) {
            const double blx = double_from_ord(nv.blx[id]), bly = double_from_ord(nv.bly[id]);
            const double trx = double_from_ord(nv.trx[id]), try_ = double_from_ord(nv.try_[id]);
            const double x = (blx + trx) * 0.5;
            const double y = (bly + try_) * 0.5;
            const double h = try_ - bly;
            const double w = trx - blx;
            nv.x[id] = x;
            nv.y[id] = y;
            nv.h[id] = h;
            nv.w[id] = w;
            const double mx = (h < w) ? w : h;   // std::max(h, w)
            const double mn = (w < h) ? w : h;   // std::min(h, w)
            const int nvort = nv.v1[id] - nv.v0[id];
            const int nlist = max(max(nvort, nv.nseg[id]), max(nv.h1[id] - nv.h0[id], nv.s1[id] - nv.s0[id]));
            leaf = (mx < max_node && mn <= min_node) || (mx < max_node && nlist < kLeafMaxList);
            depth = nv.depth[id] + 1;
        }
        const uint64_t lm = __ballot(valid && leaf), sm = __ballot(valid && !leaf);
        int sbase = 0, dmax = depth;
        for (int o = kWave / 2; o > 0; o >>= 1) dmax = max(dmax, __shfl_xor(dmax, o, kWave));
        if (lane == 0) {
            if (lm) atomicAdd(&counters[1], __popcll(lm));
            if (sm) {
                sbase = atomicAdd(&counters[0], 2 * __popcll(sm));
                atomicMax(&counters[5], dmax);
            }
        }
        sbase = __shfl(sbase, 0, kWave);
        if (!valid) continue;
        if (leaf) {
            nv.split[id] = 1;
            continue;
        }
        const int c = sbase + 2 * __popcll(sm & below);
        if (c + 2 > cap) {
            counters[4] = 1;
            nv.split[id] = 1;   // stop here; reported as an error by the host
            continue;
        }
        nv.split[id] = 2;
        nv.ch1[id] = c;
        init_node(nv, c, id, depth, nv.path[id] << 1, nv.v0[id], nv.v0[id], nv.h0[id], nv.h0[id], nv.s0[id], nv.s0[id]);
        init_node(nv, c + 1, id, depth, (nv.path[id] << 1) | 1ull, nv.v1[id], nv.v1[id], nv.h1[id], nv.h1[id],
                  nv.s1[id], nv.s1[id]);
    }
}

__device__ inline bool goes_left(const NodeView& nv, int node, double px, double py) {
    return (nv.h[node] < nv.w[node]) ? (px < nv.x[node]) : (py < nv.y[node]);
}

// Per element: "goes left" flag of elements in split nodes (else 0); 0 past
// the last element.
struct GoesLeftFlag {
    NodeView nv;
    const int32_t* enode;
    const double* x;
    const double* y;
    int n;
    __device__ int32_t operator()(int k) const {
        if (k >= n) return 0;
        const int node = enode[k];
        return (nv.split[node] == 2 && goes_left(nv, node, x[k], y[k])) ? 1 : 0;
    }
};

// Ranks of misplaced elements: left_pos[r0 + r] / right_pos[r0 + q], with
// [r0, r1) the range of the element's list in its node.  P is the exclusive
// prefix of the flags over all elements (n + 1 entries).  The first element
// of a split node's range also records that list's split position and number
// of misplaced pairs (node_L / node_m at list * cap + node) and sets the
// children's ranges.  Thread 0 advances the level range (the nodes of the
// next level were allocated by k_decide) and records it in lev[depth].
// The flags come from k_flag_count, before any swap of this level: k_swap
// reads them too and must not derive them from coordinates that the swaps
// may be rewriting.
__global__ void k_ranks(NodeView nv, const int32_t* enode, const int32_t* P, int n, int hbase, int sbase, int cap,
                        int32_t* node_L, int32_t* node_m, int32_t* left_pos, int32_t* right_pos, int32_t* counters,
                        const int32_t* flag, int2* lev, int depth) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) {
        counters[2] = counters[9];
        counters[3] = counters[0];
        counters[9] = counters[0];
        counters[6] = 0;
        counters[8] = 0;
        lev[depth] = make_int2(counters[2], counters[3]);
    }
    if (k >= n) return;
    const int node = enode[k];
    if (nv.split[node] != 2) return;
    const int cls = elem_list(k, hbase, sbase);
    int v0, v1;   // a split node's own range is unchanged
    list_range(nv, node, cls, v0, v1);
    const int P0 = P[v0];
    const int Lc = P[v1] - P0;
    const int Labs = v0 + Lc;
    if (k == v0) {
        node_L[cls * cap + node] = Labs;
        node_m[cls * cap + node] = Lc - (P[Labs] - P0);   // left-goers sitting right of Labs
        const int c = nv.ch1[node];
        set_list_range(nv, c, cls, v0, Labs);
        set_list_range(nv, c + 1, cls, Labs, v1);
    }
    const bool f = flag[k] != 0;
    if (k < Labs && !f) {
        const int r = (k - v0) - (P[k] - P0);
        left_pos[v0 + r] = k;
    } else if (k >= Labs && f) {
        const int q = P[k] - P[Labs];
        right_pos[v0 + q] = k;
    }
}

// Hoare swaps and element -> child node (the children's boxes follow from the
// elements in their places: k_bbox_top, k_child_boxes).
__global__ void k_swap(NodeView nv, int32_t* enode, const int32_t* flag, const int32_t* P, int n, int hbase,
                       int sbase, int cap, const int32_t* node_L, const int32_t* node_m, const int32_t* left_pos,
                       const int32_t* right_pos, double* x, double* y, int32_t* id) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    bool active = false;
    int node = 0, Labs = 0, v0 = 0, f = 0, c = 0, slot = 0;
    if (k < n) {
        node = enode[k];
        active = nv.split[node] == 2;
    }
    if (active) {
        const int cls = elem_list(k, hbase, sbase);
        int v1;
        list_range(nv, node, cls, v0, v1);
        slot = cls * cap + node;
        Labs = node_L[slot];
        f = flag[k];
        c = nv.ch1[node];
    }
    const bool left_mis = active && k < Labs && !f;
    if (active) enode[k] = (k < Labs) ? c : c + 1;
    // Only the left thread of a misplaced pair reads and writes either position.
    if (left_mis) {
        const int r = (k - v0) - (P[k] - P[v0]);
        const int partner = right_pos[v0 + node_m[slot] - 1 - r];
        const double px = x[k], py = y[k], qx = x[partner], qy = y[partner];
        const int32_t ik = id[k], ip = id[partner];
        x[k] = qx;
        y[k] = qy;
        id[k] = ip;
        x[partner] = px;
        y[partner] = py;
        id[partner] = ik;
    }
}

// Segments descend one level (stable partition == per-segment descent).
__global__ void k_seg_step(NodeView nv, const vvhd_seg* segs, int nseg, int32_t* seg_node) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int node = s < nseg ? seg_node[s] : 0;
    const bool active = s < nseg && nv.split[node] == 2;
    int c = 0;
    double px = 0, py = 0;
    if (active) {
        px = segs[s].x;
        py = segs[s].y;
        c = nv.ch1[node] + (goes_left(nv, node, px, py) ? 0 : 1);
        seg_node[s] = c;
    }
    add_segs_wave(nv, c, px, py, active);
}

// The ids that k_subtree took lie before the children of the level's other
// nodes.
__global__ void k_level_begin(int32_t* counters) {
    if (threadIdx.x == 0) counters[9] = counters[0];
}

// Subtrees in LDS.  A block takes one undecided node of the level after
// another (queue counters[8]); a node that fits is split down to its leaves
// by one workgroup, level by level, with the same steps as the kernels above:
// boxes, decisions, goes-left flags and their prefix, ranks, Hoare swaps.  The
// others are counted in counters[6] and stay for the level kernels.  What
// bounds a level over the whole list is its five to seven launches and passes
// over all elements (45-55 us, 22 levels at 1M and in a cylinder wake of 3k);
// in LDS a level is eight barriers, which wait for LDS operations only (the
// node records go out to memory meanwhile), and all subtrees run at once.
// The sizes keep two blocks on a compute unit (160 KiB of LDS).  A node of a
// subtree holds an element or segment of its own, and unless the box is still
// above max_node only nodes of kLeafMaxList or more split, which bounds the
// nodes of a level (fits_subtree); 64 spare ones are for empty children of
// boxes too small to halve.
constexpr int kSubElems = 1536, kSubSegs = 256, kSubNodes = 512;
constexpr int kSubThreads = 512, kSubWaves = kSubThreads / kWave;
constexpr int kSubPer = kSubElems / kSubThreads;   // elements per thread
constexpr uint16_t kDone = 0xFFFF;
static_assert(kSubNodes <= kSubThreads && kSubElems % kSubThreads == 0, "one node per thread");

__device__ inline bool fits_subtree(int ne, int ns, double mx, double max_node) {
    if (ne > kSubElems || ns > kSubSegs) return false;
    const int all = ne + ns;
    return (mx < max_node ? 2 * (all / kLeafMaxList) : all) + 64 <= kSubNodes;
}

struct SubShared {
    double x[kSubElems], y[kSubElems];
    unsigned long long lx[kSubNodes], ly[kSubNodes], hx[kSubNodes], hy[kSubNodes], path[kSubNodes];
    double sx[kSubSegs], sy[kSubSegs];
    int gid[kSubNodes], nsg[kSubNodes], sid[kSubSegs];
    uint16_t r0[3][kSubNodes], r1[3][kSubNodes];   // per list: a node's range (local elements)
    uint16_t kid[kSubNodes];                       // first child in the next level, or kDone
    uint16_t perm[kSubElems], node[kSubElems], P[kSubElems + 1], pos[kSubElems], snode[kSubSegs];
    int cnt[kSubWaves], cnt2[kSubPer * kSubWaves];
    int cur, slot, base, fail, nseg;
};

// Barrier of the block that waits for LDS operations only.
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__global__ __launch_bounds__(kSubThreads, 4) void k_subtree(NodeView nv, int32_t* counters, int cap, double min_node,
                                                            double max_node, int32_t* enode, double* gx, double* gy,
                                                            int32_t* id, const vvhd_seg* segs, int nseg,
                                                            int32_t* seg_node, int2* sub_lev, int32_t* sub_nlev,
                                                            int sub_cap) {
    __shared__ SubShared S;
    const int t = threadIdx.x, w = t / kWave, lane = lane_id();
    const uint64_t below = (1ull << lane) - 1;
    const unsigned long long lo0 = ord_from_double(DBL_MAX), hi0 = ord_from_double(-DBL_MAX);
    const int first = counters[2], last = counters[3];
    int next = 0;   // thread 0: the node after this one
    if (t == 0) next = first + atomicAdd(&counters[8], 1);
    for (;;) {
        __syncthreads();   // (also the id loads and stores of the node before)
        if (t == 0) {
            S.cur = next;
            S.fail = 0;
            S.nseg = 0;
            S.slot = sub_cap;
        }
        lds_barrier();
        const int r = S.cur;
        if (r >= last) return;   // every block gets here: the queue only grows
        const int gv0 = nv.v0[r], gh0 = nv.h0[r], gs0 = nv.s0[r];
        const int nvt = nv.v1[r] - gv0, nh = nv.h1[r] - gh0, nst = nv.s1[r] - gs0;
        const int ne = nvt + nh + nst, ns = nv.nseg[r], depth0 = nv.depth[r];
        const unsigned long long rlx = nv.blx[r], rly = nv.bly[r], rhx = nv.trx[r], rhy = nv.try_[r];
        if (t == 0) {
            next = first + atomicAdd(&counters[8], 1);
            const double h = double_from_ord(rhy) - double_from_ord(rly), wd = double_from_ord(rhx) - double_from_ord(rlx);
            if (fits_subtree(ne, ns, (h < wd) ? wd : h, max_node)) S.slot = atomicAdd(&counters[7], 1);
            if (S.slot >= sub_cap) atomicAdd(&counters[6], 1);
        }
        lds_barrier();
        const int slot = S.slot;
        if (slot >= sub_cap) continue;
        auto global_of = [&](int k) { return k < nvt ? gv0 + k : (k < nvt + nh ? gh0 + (k - nvt) : gs0 + (k - nvt - nh)); };
        for (int k = t; k < ne; k += kSubThreads) {
            const int gk = global_of(k);
            S.x[k] = gx[gk];
            S.y[k] = gy[gk];
            S.perm[k] = (uint16_t)k;
            S.node[k] = 0;
        }
        if (ns) {
            for (int q = t; q < nseg; q += kSubThreads)
                if (seg_node[q] == r) {
                    const int p = atomicAdd(&S.nseg, 1);
                    S.sid[p] = q;
                    S.sx[p] = segs[q].x;
                    S.sy[p] = segs[q].y;
                    S.snode[p] = 0;
                }
        }
        if (t == 0) {
            S.gid[0] = r;
            S.nsg[0] = 0;
            S.path[0] = nv.path[r];
            S.lx[0] = rlx;
            S.ly[0] = rly;
            S.hx[0] = rhx;
            S.hy[0] = rhy;
            S.r0[0][0] = 0;
            S.r1[0][0] = S.r0[1][0] = (uint16_t)nvt;
            S.r1[1][0] = S.r0[2][0] = (uint16_t)(nvt + nh);
            S.r1[2][0] = (uint16_t)ne;
        }
        lds_barrier();
        // does a point of node i go to its first child (goes_left)
        auto left_of = [&](int i, double px, double py) {
            const double blx = double_from_ord(S.lx[i]), bly = double_from_ord(S.ly[i]);
            const double trx = double_from_ord(S.hx[i]), try_ = double_from_ord(S.hy[i]);
            return (try_ - bly < trx - blx) ? px < (blx + trx) * 0.5 : py < (bly + try_) * 0.5;
        };
        auto add_box = [&](int i, double px, double py) {
            if (!isnan(px)) {
                const unsigned long long o = ord_from_double(px);
                atomicMin(&S.lx[i], o);
                atomicMax(&S.hx[i], o);
            }
            if (!isnan(py)) {
                const unsigned long long o = ord_from_double(py);
                atomicMin(&S.ly[i], o);
                atomicMax(&S.hy[i], o);
            }
        };
        int m = 1, lev = 0;
        for (;; lev++) {
            // boxes of this level's nodes (the root's is known) and their segments:
            // L lanes per node over its ranges, about three elements per lane
            // (one LDS atomic per element and side queues 64 deep on a node's
            // slots: 5 us a level).  Below eight nodes several waves share one.
            if (lev > 0) {
                int L = kWave;
                while (L > 1 && L * m > kSubThreads) L >>= 1;
                const int parts = max(1, kSubThreads / (L * m));   // groups per node
                const int grp = t / L, i = grp / parts, sub = (grp % parts) * L + (t & (L - 1)), step = parts * L;
                double bx0 = DBL_MAX, by0 = DBL_MAX, bx1 = -DBL_MAX, by1 = -DBL_MAX;
                if (i < m)
                    for (int c = 0; c < 3; c++) {
                        const int b = S.r1[c][i];
                        for (int k = S.r0[c][i] + sub; k < b; k += step) {
                            const double px = S.x[k], py = S.y[k];   // fmin and fmax pass over NaN
                            bx0 = fmin(bx0, px);
                            by0 = fmin(by0, py);
                            bx1 = fmax(bx1, px);
                            by1 = fmax(by1, py);
                        }
                    }
                for (int o = L / 2; o > 0; o >>= 1) {
                    bx0 = fmin(bx0, __shfl_xor(bx0, o, kWave));
                    by0 = fmin(by0, __shfl_xor(by0, o, kWave));
                    bx1 = fmax(bx1, __shfl_xor(bx1, o, kWave));
                    by1 = fmax(by1, __shfl_xor(by1, o, kWave));
                }
                if (i < m && (t & (L - 1)) == 0) {
                    if (bx0 != DBL_MAX) atomicMin(&S.lx[i], (unsigned long long)ord_from_double(bx0));
                    if (by0 != DBL_MAX) atomicMin(&S.ly[i], (unsigned long long)ord_from_double(by0));
                    if (bx1 != -DBL_MAX) atomicMax(&S.hx[i], (unsigned long long)ord_from_double(bx1));
                    if (by1 != -DBL_MAX) atomicMax(&S.hy[i], (unsigned long long)ord_from_double(by1));
                }
            }
            if (t < ns && S.snode[t] != kDone) {
                const int i = S.snode[t];
                atomicAdd(&S.nsg[i], 1);
                if (lev > 0) add_box(i, S.sx[t], S.sy[t]);
            }
            lds_barrier();
            // decisions (k_decide), one node per thread
            bool split = false;
            if (t < m) {
                const int gi = S.gid[t];
                const double blx = double_from_ord(S.lx[t]), bly = double_from_ord(S.ly[t]);
                const double trx = double_from_ord(S.hx[t]), try_ = double_from_ord(S.hy[t]);
                const double h = try_ - bly, wd = trx - blx;
                const double mx = (h < wd) ? wd : h;   // std::max(h, w)
                const double mn = (wd < h) ? wd : h;   // std::min(h, w)
                int nlist = S.nsg[t];
                for (int c = 0; c < 3; c++) nlist = max(nlist, (int)S.r1[c][t] - (int)S.r0[c][t]);
                split = !((mx < max_node && mn <= min_node) || (mx < max_node && nlist < kLeafMaxList));
                nv.x[gi] = (blx + trx) * 0.5;
                nv.y[gi] = (bly + try_) * 0.5;
                nv.h[gi] = h;
                nv.w[gi] = wd;
                nv.split[gi] = split ? 2 : 1;
                if (lev > 0) {
                    nv.blx[gi] = S.lx[t];
                    nv.bly[gi] = S.ly[t];
                    nv.trx[gi] = S.hx[t];
                    nv.try_[gi] = S.hy[t];
                    nv.nseg[gi] = S.nsg[t];
                }
            }
            const uint64_t sm = __ballot(split);
            if (lane == 0) S.cnt[w] = __popcll(sm);
            lds_barrier();
            int nsplit = 0, rank = 0;
            for (int q = 0; q < kSubWaves; q++) {
                if (q == w) rank = nsplit;
                nsplit += S.cnt[q];
            }
            rank += __popcll(sm & below);
            if (t < m) S.kid[t] = split ? (uint16_t)(2 * rank) : kDone;
            // ids of the children: the counter's answer is needed only when
            // they are written
            int claim = 0;
            if (t == 0) {
                atomicAdd(&counters[1], m - nsplit);
                if (nsplit) {
                    atomicMax(&counters[5], depth0 + lev + 1);
                    claim = atomicAdd(&counters[0], 2 * nsplit);
                }
            }
            lds_barrier();
            // goes-left flags and their counts; the elements of leaves are done
            uint64_t fmask[kSubPer];
            for (int j = 0; j < kSubPer; j++) {
                const int k = j * kSubThreads + t;
                bool f = false;
                if (k < ne && S.node[k] != kDone) {
                    const int i = S.node[k];
                    if (S.kid[i] == kDone) {
                        enode[global_of(k)] = S.gid[i];
                        S.node[k] = kDone;
                    } else {
                        f = left_of(i, S.x[k], S.y[k]);
                    }
                }
                fmask[j] = __ballot(f);
                if (lane == 0) S.cnt2[j * kSubWaves + w] = __popcll(fmask[j]);
            }
            if (t < ns && S.snode[t] != kDone) {
                const int i = S.snode[t];
                if (S.kid[i] == kDone) {
                    seg_node[S.sid[t]] = S.gid[i];
                    S.snode[t] = kDone;
                } else {
                    S.snode[t] = (uint16_t)(S.kid[i] + (left_of(i, S.sx[t], S.sy[t]) ? 0 : 1));
                }
            }
            if (nsplit == 0) break;
            lds_barrier();
            {
                int run = 0;
                for (int q = 0; q < kSubPer * kSubWaves; q++) {
                    if (q % kSubWaves == w) {
                        const int j = q / kSubWaves, k = j * kSubThreads + t;
                        if (k < ne) S.P[k] = (uint16_t)(run + __popcll(fmask[j] & below));
                    }
                    run += S.cnt2[q];
                }
                if (t == 0) S.P[ne] = (uint16_t)run;
            }
            lds_barrier();
            // ranks of misplaced elements: a node's left ones from the front of
            // its range of pos, the right ones from the back
            for (int j = 0; j < kSubPer; j++) {
                const int k = j * kSubThreads + t;
                if (k >= ne || S.node[k] == kDone) continue;
                const int i = S.node[k], c = k < nvt ? 0 : (k < nvt + nh ? 1 : 2);
                const int a = S.r0[c][i], b = S.r1[c][i];
                const int Pa = S.P[a], Labs = a + S.P[b] - Pa;
                const bool f = (fmask[j] >> lane) & 1;
                if (k < Labs && !f)
                    S.pos[k - (S.P[k] - Pa)] = (uint16_t)k;
                else if (k >= Labs && f)
                    S.pos[b - 1 - (S.P[k] - S.P[Labs])] = (uint16_t)k;
            }
            lds_barrier();
            for (int j = 0; j < kSubPer; j++) {
                const int k = j * kSubThreads + t;
                if (k >= ne || S.node[k] == kDone) continue;
                const int i = S.node[k], c = k < nvt ? 0 : (k < nvt + nh ? 1 : 2);
                const int a = S.r0[c][i], b = S.r1[c][i];
                const int Pa = S.P[a], Lc = S.P[b] - Pa, Labs = a + Lc;
                const bool f = (fmask[j] >> lane) & 1;
                if (k < Labs && !f) {   // the left thread of a pair swaps
                    const int pairs = Lc - (S.P[Labs] - Pa);
                    const int q = S.pos[b - pairs + (k - a) - (S.P[k] - Pa)];
                    const double px = S.x[k], py = S.y[k];
                    const uint16_t pk = S.perm[k];
                    S.x[k] = S.x[q];
                    S.y[k] = S.y[q];
                    S.perm[k] = S.perm[q];
                    S.x[q] = px;
                    S.y[q] = py;
                    S.perm[q] = pk;
                }
                S.node[k] = (uint16_t)(S.kid[i] + (k < Labs ? 0 : 1));
            }
            // children: the parents' records are read before any is replaced
            const int pk = t < m ? S.kid[t] : kDone;
            int pg = 0, pr[3][3];
            unsigned long long ppath = 0;
            if (pk != kDone) {
                pg = S.gid[t];
                ppath = S.path[t] << 1;
                for (int c = 0; c < 3; c++) {
                    const int a = S.r0[c][t], b = S.r1[c][t];
                    pr[c][0] = a;
                    pr[c][1] = a + S.P[b] - S.P[a];
                    pr[c][2] = b;
                }
            }
            if (t == 0) {
                S.base = claim;
                if (claim + 2 * nsplit > cap || 2 * nsplit > kSubNodes) S.fail = 1;
                if (depth0 + lev + 2 >= kMaxLevels) S.fail = 2;
                if (S.fail)
                    counters[4] = S.fail;
                else
                    sub_lev[(size_t)slot * kSubLevels + lev] = make_int2(claim, 2 * nsplit);
            }
            lds_barrier();
            if (S.fail) return;   // uniform; the host reports counters[4]
            const int base = S.base;
            if (pk != kDone) {
                nv.ch1[pg] = base + pk;
                for (int q = 0; q < 2; q++) {
                    const int i = pk + q, gi = base + i;
                    S.gid[i] = gi;
                    S.nsg[i] = 0;
                    S.path[i] = ppath | (unsigned long long)q;
                    S.lx[i] = S.ly[i] = lo0;
                    S.hx[i] = S.hy[i] = hi0;
                    for (int c = 0; c < 3; c++) {
                        S.r0[c][i] = (uint16_t)pr[c][q];
                        S.r1[c][i] = (uint16_t)pr[c][q + 1];
                    }
                    nv.parent[gi] = pg;
                    nv.depth[gi] = depth0 + lev + 1;
                    nv.path[gi] = ppath | (unsigned long long)q;
                    nv.ch1[gi] = -1;
                    nv.v0[gi] = gv0 + pr[0][q];
                    nv.v1[gi] = gv0 + pr[0][q + 1];
                    nv.h0[gi] = gh0 + pr[1][q] - nvt;
                    nv.h1[gi] = gh0 + pr[1][q + 1] - nvt;
                    nv.s0[gi] = gs0 + pr[2][q] - nvt - nh;
                    nv.s1[gi] = gs0 + pr[2][q + 1] - nvt - nh;
                }
            }
            lds_barrier();
            m = 2 * nsplit;
        }
        if (t == 0) sub_nlev[slot] = lev;
        // positions and ids back; the old ids are read before any is replaced
        int32_t ids[kSubPer];
        for (int j = 0; j < kSubPer; j++) {
            const int k = j * kSubThreads + t;
            if (k < ne) {
                const int gk = global_of(k);
                ids[j] = id[global_of(S.perm[k])];
                gx[gk] = S.x[k];
                gy[gk] = S.y[k];
            }
        }
        __syncthreads();
        for (int j = 0; j < kSubPer; j++) {
            const int k = j * kSubThreads + t;
            if (k < ne) id[global_of(k)] = ids[j];
        }
    }
}

// A heat or streak list in tree order: positions from the element arrays,
// the other fields gathered from the list's own arrays (id holds element
// numbers, base is the list's first element).
__global__ void k_gather_list(const int32_t* id, int n, int base, const double* ex, const double* ey, const double* g,
                              const double* vx, const double* vy, const double* ie, double* x2, double* y2, double* g2,
                              double* vx2, double* vy2, double* ie2) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int s = id[k] - base;
    x2[k] = ex[k];
    y2[k] = ey[k];
    g2[k] = g[s];
    vx2[k] = vx[s];
    vy2[k] = vy[s];
    ie2[k] = ie[s];
}

// Gathers the non-key vortex fields into tree order.
__global__ void k_gather(const int32_t* id, int n, const double* g, const double* vx, const double* vy,
                         const double* ie, double* g2, double* vx2, double* vy2, double* ie2) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int s = id[k];
    g2[k] = g[s];
    vx2[k] = vx[s];
    vy2[k] = vy[s];
    ie2[k] = ie[s];
}

struct CMView {
    double *px, *py, *pg, *mx, *my, *mg;
    float *pie, *mie;
};

CMView cm_view(const TreeArrays& t) {
    return CMView{t.cmp_x.p, t.cmp_y.p, t.cmp_g.p, t.cmm_x.p, t.cmm_y.p, t.cmm_g.p, t.cmp_ie.p, t.cmm_ie.p};
}

// Per-sign monopoles of a node (CMp, CMm); ie is _1_eps, infinite or 0.
struct Monopoles {
    double px, py, pg, mx, my, mg;
    float pie, mie;
};

__device__ inline Monopoles get_monopoles(const CMView& cm, int id) {
    return Monopoles{cm.px[id], cm.py[id], cm.pg[id], cm.mx[id], cm.my[id], cm.mg[id], cm.pie[id], cm.mie[id]};
}

__device__ inline void put_monopoles(const CMView& cm, int id, const Monopoles& q) {
    cm.px[id] = q.px;
    cm.py[id] = q.py;
    cm.pg[id] = q.pg;
    cm.mx[id] = q.mx;
    cm.my[id] = q.my;
    cm.mg[id] = q.mg;
    cm.pie[id] = q.pie;
    cm.mie[id] = q.mie;
}

// CalculateCMassFromScratch (TSortedTree.cpp:176-197), in array order.
__device__ inline Monopoles leaf_monopoles(const NodeView& nv, int id, const double* x, const double* y,
                                           const double* g) {
    Monopoles q{0, 0, 0, 0, 0, 0, INFINITY, INFINITY};
    for (int k = nv.v0[id]; k < nv.v1[id]; k++) {
        const double gk = g[k];
        if (gk > 0) {
            q.px += x[k] * gk;
            q.py += y[k] * gk;
            q.pg += gk;
        } else {
            q.mx += x[k] * gk;
            q.my += y[k] * gk;
            q.mg += gk;
        }
    }
    if (q.pg) {
        q.px *= (1. / q.pg);
        q.py *= (1. / q.pg);
    } else {
        q.px = nv.x[id];
        q.py = nv.y[id];
    }
    if (q.mg) {
        q.mx *= (1. / q.mg);
        q.my *= (1. / q.mg);
    } else {
        q.mx = nv.x[id];
        q.my = nv.y[id];
    }
    return q;
}

// CalculateCMass (:150-174) from the children; without circulation
// TObj(x, y, 0): _1_eps = 0.
__device__ inline Monopoles node_monopoles(const NodeView& nv, int id, const Monopoles& a, const Monopoles& b) {
    Monopoles q;
    auto combine = [&](double ax, double ay, double ag, double bx, double by, double bg, double& x, double& y,
                       double& g, float& ie) {
        const double s = ag + bg;
        if (s) {
            const double inv = 1. / s;
            x = (ax * ag + bx * bg) * inv;
            y = (ay * ag + by * bg) * inv;
            g = s;
            ie = INFINITY;
        } else {
            x = nv.x[id];
            y = nv.y[id];
            g = 0;
            ie = 0;
        }
    };
    combine(a.px, a.py, a.pg, b.px, b.py, b.pg, q.px, q.py, q.pg, q.pie);
    combine(a.mx, a.my, a.mg, b.mx, b.my, b.mg, q.mx, q.my, q.mg, q.mie);
    return q;
}

// Leaf count and monopoles of a node.
__device__ inline void up_node(const NodeView& nv, const CMView& cm, int id, const double* x, const double* y,
                               const double* g, int32_t* nleaves) {
    if (nv.split[id] != 2) {
        nleaves[id] = 1;
        put_monopoles(cm, id, leaf_monopoles(nv, id, x, y, g));
        return;
    }
    const int a = nv.ch1[id];
    nleaves[id] = nleaves[a] + nleaves[a + 1];
    put_monopoles(cm, id, node_monopoles(nv, id, get_monopoles(cm, a), get_monopoles(cm, a + 1)));
}

// Leaf f (DFS rank) is node id.
__device__ inline void down_leaf(const NodeView& nv, int id, int f, int32_t* leaf_rank, int32_t* leaf_node,
                                 int32_t* vleaf) {
    leaf_rank[id] = f;
    leaf_node[f] = id;
    for (int k = nv.v0[id]; k < nv.v1[id]; k++) vleaf[k] = f;
    for (int k = nv.h0[id]; k < nv.h1[id]; k++) vleaf[k] = f;
    for (int k = nv.s0[id]; k < nv.s1[id]; k++) vleaf[k] = f;
}

// First leaf rank of a node's children (DFS order), or the leaf itself.
__device__ inline void down_node(const NodeView& nv, int id, const int32_t* nleaves, int32_t* first,
                                 int32_t* leaf_rank, int32_t* leaf_node, int32_t* vleaf, int32_t* pre) {
    const int f = first[id];
    if (nv.split[id] != 2) {
        down_leaf(nv, id, f, leaf_rank, leaf_node, vleaf);
        return;
    }
    const int a = nv.ch1[id];
    first[a] = f;
    first[a + 1] = f + nleaves[a];
    const int p = pre[id];   // the first child's subtree (2 nleaves - 1 nodes) follows the node
    pre[a] = p + 1;
    pre[a + 1] = p + 2 * nleaves[a];
}

// The passes over the finished nodes.  In the levels over the whole list one
// launch takes several consecutive levels, a block for all of them (levels
// [l0, l1) of lev, at most kPassNodes nodes each: a level of a launch of its
// own waits 4-7 us); larger levels are launched by themselves (one = true:
// level l0 spread over the grid).  In the subtrees one block takes one
// subtree.  Bottom-up, leaves go first, all at once.
constexpr int kPassNodes = 8192, kPassThreads = 1024;

__global__ __launch_bounds__(kPassThreads) void k_up_levels(NodeView nv, CMView cm, const int2* lev, int l0, int l1,
                                                            const double* x, const double* y, const double* g,
                                                            int32_t* nleaves) {
    const int t = blockIdx.x * kPassThreads + threadIdx.x, step = gridDim.x * kPassThreads;
    if (l1 - l0 > 1) {
        for (int d = l0; d < l1; d++)
            for (int id = lev[d].x + t; id < lev[d].y; id += step)
                if (nv.split[id] != 2) up_node(nv, cm, id, x, y, g, nleaves);
        __threadfence_block();
        __syncthreads();
    }
    for (int d = l1 - 1; d >= l0; d--) {
        for (int id = lev[d].x + t; id < lev[d].y; id += step)
            if (l1 - l0 == 1 || nv.split[id] == 2) up_node(nv, cm, id, x, y, g, nleaves);
        __threadfence_block();
        __syncthreads();
    }
}

__global__ __launch_bounds__(kPassThreads) void k_down_levels(NodeView nv, const int2* lev, int l0, int l1,
                                                              const int32_t* nleaves, int32_t* first,
                                                              int32_t* leaf_rank, int32_t* leaf_node, int32_t* vleaf,
                                                              int32_t* pre) {
    const int t = blockIdx.x * kPassThreads + threadIdx.x, step = gridDim.x * kPassThreads;
    for (int d = l0; d < l1; d++) {
        for (int id = lev[d].x + t; id < lev[d].y; id += step)
            down_node(nv, id, nleaves, first, leaf_rank, leaf_node, vleaf, pre);
        __threadfence_block();
        __syncthreads();
    }
}

// A subtree's nodes in LDS for the passes: numbered level after level, children
// and leaf counts (and monopoles) of the first kPassLds; nodes beyond them are
// read back from memory.  With every level's children behind two or three
// dependent loads from memory a pass took 15-23 us for nine levels.
constexpr int kPassLds = 1024;
struct SubNodes {
    int2 lev[kSubLevels];
    int off[kSubLevels + 1];   // first node of a level in the numbering
    int kid[kPassLds];         // first child (numbering), or -1
    int nl[kPassLds];          // leaves under the node
    int nlev, count;
};

__device__ inline void load_sub(SubNodes& N, const NodeView& nv, const int2* sub_lev, const int32_t* sub_nlev) {
    const int t = threadIdx.x, nl = sub_nlev[blockIdx.x];
    for (int d = t; d < nl; d += kBlock) N.lev[d] = sub_lev[(size_t)blockIdx.x * kSubLevels + d];
    __syncthreads();
    if (t == 0) {
        int o = 0;
        for (int d = 0; d < nl; d++) {
            N.off[d] = o;
            o += N.lev[d].y;
        }
        N.off[nl] = o;
        N.nlev = nl;
        N.count = o;
    }
    __syncthreads();
    for (int n = t, d = 0; n < min(N.count, kPassLds); n += kBlock) {
        while (N.off[d + 1] <= n) d++;
        const int id = N.lev[d].x + (n - N.off[d]), sp = nv.split[id], ch = nv.ch1[id];
        N.kid[n] = sp == 2 ? N.off[d + 1] + (ch - N.lev[d + 1].x) : -1;
    }
}

__global__ __launch_bounds__(kBlock) void k_up_subs(NodeView nv, CMView cm, const int2* sub_lev,
                                                    const int32_t* sub_nlev, const double* x, const double* y,
                                                    const double* g, int32_t* nleaves) {
    __shared__ SubNodes N;
    __shared__ Monopoles M[kPassLds];
    load_sub(N, nv, sub_lev, sub_nlev);
    __syncthreads();
    const int t = threadIdx.x;
    auto is_leaf = [&](int n, int id) { return n < kPassLds ? N.kid[n] < 0 : nv.split[id] != 2; };
    for (int n = t, d = 0; n < N.count; n += kBlock) {
        while (N.off[d + 1] <= n) d++;
        const int id = N.lev[d].x + (n - N.off[d]);
        if (!is_leaf(n, id)) continue;
        const Monopoles q = leaf_monopoles(nv, id, x, y, g);
        put_monopoles(cm, id, q);
        nleaves[id] = 1;
        if (n < kPassLds) {
            M[n] = q;
            N.nl[n] = 1;
        }
    }
    __threadfence_block();
    __syncthreads();
    for (int d = N.nlev - 2; d >= 0; d--) {   // the last level holds leaves only
        for (int i = t; i < N.lev[d].y; i += kBlock) {
            const int id = N.lev[d].x + i, n = N.off[d] + i;
            if (is_leaf(n, id)) continue;
            const int a = nv.ch1[id], ka = N.off[d + 1] + (a - N.lev[d + 1].x);
            const bool in = ka + 1 < kPassLds;
            const Monopoles q = in ? node_monopoles(nv, id, M[ka], M[ka + 1])
                                   : node_monopoles(nv, id, get_monopoles(cm, a), get_monopoles(cm, a + 1));
            const int cnt = in ? N.nl[ka] + N.nl[ka + 1] : nleaves[a] + nleaves[a + 1];
            put_monopoles(cm, id, q);
            nleaves[id] = cnt;
            if (n < kPassLds) {
                M[n] = q;
                N.nl[n] = cnt;
            }
        }
        __threadfence_block();
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void k_down_subs(NodeView nv, const int2* sub_lev, const int32_t* sub_nlev,
                                                      const int32_t* nleaves, int32_t* first, int32_t* leaf_rank,
                                                      int32_t* leaf_node, int32_t* vleaf, int32_t* pre) {
    __shared__ SubNodes N;
    __shared__ int s_first[kPassLds], s_pre[kPassLds];
    load_sub(N, nv, sub_lev, sub_nlev);
    const int t = threadIdx.x;
    for (int n = t, d = 0; n < min(N.count, kPassLds); n += kBlock) {
        while (N.off[d + 1] <= n) d++;
        N.nl[n] = nleaves[N.lev[d].x + (n - N.off[d])];
    }
    if (t < 2 && N.nlev > 0) {   // the root's children: k_down_levels set them
        s_first[t] = first[N.lev[0].x + t];
        s_pre[t] = pre[N.lev[0].x + t];
    }
    __syncthreads();
    for (int d = 0; d < N.nlev; d++) {
        for (int i = t; i < N.lev[d].y; i += kBlock) {
            const int id = N.lev[d].x + i, n = N.off[d] + i;
            if (n >= kPassLds) {
                down_node(nv, id, nleaves, first, leaf_rank, leaf_node, vleaf, pre);
                continue;
            }
            const int ka = N.kid[n];
            if (ka < 0) {
                down_leaf(nv, id, s_first[n], leaf_rank, leaf_node, vleaf);
                continue;
            }
            const int a = N.lev[d + 1].x + (ka - N.off[d + 1]);
            const int na = ka < kPassLds ? N.nl[ka] : nleaves[a];
            const int f[2] = {s_first[n], s_first[n] + na}, q[2] = {s_pre[n] + 1, s_pre[n] + 2 * na};
            for (int k = 0; k < 2; k++) {
                pre[a + k] = q[k];
                if (ka + k < kPassLds) {
                    s_first[ka + k] = f[k];
                    s_pre[ka + k] = q[k];
                } else {
                    first[a + k] = f[k];
                }
            }
        }
        __threadfence_block();
        __syncthreads();
    }
}

__global__ void k_pack_boxes(NodeView nv, int nnodes, double4* out) {
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nnodes) return;
    out[id] = make_double4(double_from_ord(nv.blx[id]), double_from_ord(nv.bly[id]), double_from_ord(nv.trx[id]),
                           double_from_ord(nv.try_[id]));
}

// What the list walk reads of a node, one 32-byte record per node stored at
// the node's preorder position: centre, h + w (added first, as the far test
// does), node id, and the position that follows its subtree (position + 1
// for a leaf).  A walk then only moves forward through memory: into the
// subtree at position + 1, or past it.
struct TravNode {
    double x, y, hw;
    int32_t id, skip;
};
static_assert(sizeof(TravNode) == 32, "TravNode layout");

__global__ void k_trav_nodes(NodeView nv, int nnodes, const int32_t* pre, const int32_t* nleaves, TravNode* out,
                             int32_t* most, CMView cm, double2* cmk) {
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id < 2) most[id] = 0;
    if (id >= nnodes) return;
    cmk[4 * (size_t)id] = make_double2(cm.px[id], cm.py[id]);
    cmk[4 * (size_t)id + 1] = make_double2(cm.pg[id], cm.mg[id]);
    cmk[4 * (size_t)id + 2] = make_double2(cm.mx[id], cm.my[id]);
    TravNode r;
    r.x = nv.x[id];
    r.y = nv.y[id];
    r.hw = nv.h[id] + nv.w[id];
    r.id = id;
    const int p = pre[id];
    r.skip = p + 2 * nleaves[id] - 1;
    out[p] = r;
}

// FindNearNodes (TSortedTree.cpp:199-217) of every leaf: one walk that logs
// its steps, then a replay of the log at the scanned offsets.
// A wave walks for a group of up to 64 DFS-consecutive leaves of one root, a
// leaf per lane, in preorder without a stack: from a node it moves to the next
// position (the first child) while some lane still needs the node's subtree,
// otherwise past the subtree.  A lane that classifies a node as far (or
// reaches a near leaf) waits until the walk leaves that subtree.  Every step
// at which some lane lists the node is a record {node, far lanes, near lanes}.
// k_list_top walks a group's nodes with more than item_nodes nodes below
// them; a smaller subtree that is still needed becomes an item, noted in the
// group's log and walked by a wave of its own (k_list_items).  k_list_sums
// adds up, in the order of the group's log, what each lane has listed before
// every item and in all; k_list_replay writes the records at these offsets,
// so that the lists hold the reference's preorder.
// Bound by the instructions and load latency of the steps (3.9 M for 57.7 M
// entries at 1M) and by how evenly they spread: cut at depth 6, the longest of
// 98k walks had 3101 steps and 1200 walks held nearly all of them, and the
// steps were walked twice, to count and to write.  No counter is shared
// between waves (50k claims of one address cost 0.7 ms).
struct ListLog {
    int R, S;                    // records and items every group has room for,
    const int64_t *tbase, *ibase;   // or (not null) where each group's begin: room for as many as it has
    int slots;                   // items there is room for in all groups
    int64_t cap;                 // records of all items
    int32_t* tid;                // a group's records: node, or -(item of the group + 1)
    uint64_t *tfar, *tnear;
    int32_t *nrec, *nitem;       // per group: records, items
    int32_t* gnodes;             // per group: nodes of its items (their records at most)
    const int64_t* gbase;        // their exclusive sums
    int2* item;                  // a group's items: position, first record within the group's
    uint64_t* item_mask;         // lanes that need it
    int32_t* item_n;             // its records
    int32_t* item_grp;           // its group (written where ibase is given)
    int2 *lanes, *after;         // items x 64: near and far nodes a lane lists in the item, then before it; and after it
    int32_t* rid;
    uint64_t *rfar, *rnear;
    int32_t* most;               // not 0 where a group's records [0] or items [1] ran out of room
    __device__ int64_t rec0(int g) const { return tbase ? tbase[g] : (int64_t)g * R; }
    __device__ int64_t item0(int g) const { return ibase ? ibase[g] : (int64_t)g * S; }
    __device__ int recs(int g) const { return tbase ? (int)(tbase[g + 1] - tbase[g]) : R; }
    __device__ int items(int g) const { return ibase ? (int)(ibase[g + 1] - ibase[g]) : S; }
    // Item of slot w, its group in grp; -1 where the slot holds none.
    template <bool kExact>
    __device__ int64_t slot(int w, int ngroups, int& grp) const {
        if (kExact) {
            grp = __builtin_amdgcn_readfirstlane(item_grp[w]);
            return w;
        }
        grp = __builtin_amdgcn_readfirstlane(w % ngroups);
        const int k = __builtin_amdgcn_readfirstlane(w / ngroups);
        return k < nitem[grp] ? (int64_t)grp * S + k : -1;
    }
};

// The records of one walk at [o, o + limit): record k of every 64 is collected
// in lane k, 64 go out in one coalesced store.  Records past the limit are
// counted only.
struct LogWriter {
    int32_t* id;
    uint64_t *far, *near;
    int64_t limit;
    const int lane;
    int32_t rid = 0;
    uint64_t rf = 0, rn = 0;
    int cnt = 0;
    int64_t done = 0;
    __device__ inline void push(int32_t i, uint64_t F, uint64_t N) {
        if (lane == cnt) {
            rid = i;
            rf = F;
            rn = N;
        }
        if (++cnt == kWave) flush();
    }
    __device__ inline void flush() {
        if (lane < cnt && done + lane < limit) {
            id[done + lane] = rid;
            far[done + lane] = rf;
            near[done + lane] = rn;
        }
        done += cnt;
        cnt = 0;
    }
};

// Walks positions [P, end) for the lanes' leaves (a lane takes part at
// positions >= resume); subtrees of at most item_nodes nodes go to item(P,
// nodes, lanes) and are passed over.  cn, cf: the lane's listed nodes.
template <typename Item>
__device__ inline void list_walk(const TravNode* __restrict__ tn, int P, int end, int resume, double lx, double ly,
                                 double lh, double lw, double fc, int item_nodes, LogWriter& log, int& cn, int& cf,
                                 Item item) {
    // the position is uniform: records come through the scalar cache, all
    // 32 bytes in one load
    auto rec = [&](int p) {
        const uint4* q4 = reinterpret_cast<const uint4*>(tn + p);
        const uint4 u0 = q4[0], u1 = q4[1];
        TravNode r;
        __builtin_memcpy(&r, &u0, 16);
        __builtin_memcpy(reinterpret_cast<char*>(&r) + 16, &u1, 16);
        return r;
    };
    while (P < end) {
        const TravNode r = rec(P);
        const int skip = __builtin_amdgcn_readfirstlane(r.skip);
        const int id = __builtin_amdgcn_readfirstlane(r.id);
        const bool act = P >= resume;
        const bool leaf = skip == P + 1;
        const double dx = r.x - lx, dy = r.y - ly;
        const double hp = r.hw + lh + lw;
        const bool far = act && (dx * dx + dy * dy > fc * hp * hp);
        const bool near = act && leaf && !far;
        if (far) {
            cf++;
            resume = skip;
        }
        if (near) cn++;
        const uint64_t F = __ballot(far), N = __ballot(near);
        const uint64_t need = leaf ? 0 : __ballot(act && !far);
        if (F | N) log.push(id, F, N);
        if (need == 0) {
            P = max(skip, P + 1);
        } else if (skip - P <= item_nodes) {
            item(P, skip - P, need);
            P = skip;
        } else {
            P = P + 1;
        }
        P = __builtin_amdgcn_readfirstlane(P);
    }
}

__global__ __launch_bounds__(kBlock) void k_list_top(NodeView nv, const TravNode* __restrict__ tn,
                                                     const int32_t* __restrict__ pre,
                                                     const int32_t* __restrict__ groups, int ngroups,
                                                     const int32_t* leaf_node, double fc, int item_nodes, ListLog G) {
    const int grp = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave, lane = lane_id();
    if (grp >= ngroups) return;
    const int l = groups[3 * grp] + lane;
    const bool valid = lane < groups[3 * grp + 1];
    const int L = valid ? leaf_node[l] : 0;
    const int P0 = __builtin_amdgcn_readfirstlane(pre[groups[3 * grp + 2]]);
    const int end = __builtin_amdgcn_readfirstlane(tn[P0].skip);
    const int64_t o = G.rec0(grp), io = G.item0(grp);
    const int R = G.recs(grp), S = G.items(grp);
    LogWriter log{G.tid + o, G.tfar + o, G.tnear + o, R, lane};
    int cn = 0, cf = 0, ni = 0, nodes = 0;
    list_walk(tn, P0, end, valid ? P0 : end, nv.x[L], nv.y[L], nv.h[L], nv.w[L], fc, item_nodes, log, cn, cf,
              [&](int P, int size, uint64_t need) {
                  if (lane == 0 && ni < S) {
                      G.item[io + ni] = make_int2(P, nodes);
                      G.item_mask[io + ni] = need;
                      if (G.ibase) G.item_grp[io + ni] = grp;
                  }
                  log.push(-(ni + 1), 0, 0);
                  ni++;
                  nodes += size;
              });
    log.flush();
    if (lane != 0) return;
    G.nrec[grp] = (int)log.done;
    G.nitem[grp] = ni;
    G.gnodes[grp] = nodes;
    if (log.done > R) G.most[0] = 1;
    if (ni > S) G.most[1] = 1;
}

// kExact: room as counted (ibase); a wave may then take several items.
template <bool kExact>
__global__ __launch_bounds__(kBlock) void k_list_items(NodeView nv, const TravNode* __restrict__ tn,
                                                       const int32_t* __restrict__ groups, int ngroups,
                                                       const int32_t* leaf_node, double fc, ListLog G) {
    const int lane = lane_id();
    if (G.most[0] | G.most[1]) return;   // the walk is repeated
    // item k of all groups, then item k + 1: a group has about 20 of its S items,
    // and with a group's items in neighbouring blocks these fell on the same few
    // XCDs (S = 64: 1.6 against 0.53 ms at 1M)
    const int step = gridDim.x * (kBlock / kWave);
    for (int w = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; w < G.slots; w += step) {
        int grp;
        const int64_t it = G.slot<kExact>(w, ngroups, grp);
        if (it < 0) return;
        const int P0 = __builtin_amdgcn_readfirstlane(G.item[it].x);
        const int end = __builtin_amdgcn_readfirstlane(tn[P0].skip);
        const bool mine = (G.item_mask[it] >> lane) & 1;
        const int l = groups[3 * grp] + lane;
        const int L = mine ? leaf_node[l] : 0;
        const int64_t o = G.gbase[grp] + G.item[it].y;
        const int64_t room = min((int64_t)(end - P0), max((int64_t)0, G.cap - o));
        LogWriter log{G.rid + o, G.rfar + o, G.rnear + o, room, lane};
        int cn = 0, cf = 0;
        list_walk(tn, P0 + 1, end, mine ? P0 : end, nv.x[L], nv.y[L], nv.h[L], nv.w[L], fc, 0, log, cn, cf,
                  [](int, int, uint64_t) {});
        log.flush();
        if (lane == 0) G.item_n[it] = (int)log.done;
        G.lanes[it * kWave + lane] = make_int2(cn, cf);
        if (!kExact) return;
    }
}

// Reads 64 records of a log at once, one per lane, and hands them out in order.
struct LogReader {
    const int32_t* id;
    const uint64_t *far, *near;
    int32_t rid = 0;
    uint64_t rf = 0, rn = 0;
    __device__ inline void load(int64_t o, int left, int lane) {
        if (lane < left) {
            rid = id[o + lane];
            rf = far[o + lane];
            rn = near[o + lane];
        }
    }
    __device__ static inline uint64_t pick(uint64_t v, int k) {
        return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), k) << 32) |
               (uint32_t)__builtin_amdgcn_readlane((int)v, k);
    }
};

// One wave per group: what each lane lists before every item of the group's
// log (left in lanes), and in all (the leaf's counts).
__global__ __launch_bounds__(kBlock) void k_list_sums(const int32_t* __restrict__ groups, int ngroups, ListLog G,
                                                      int32_t* near_cnt, int32_t* far_cnt) {
    const int grp = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave, lane = lane_id();
    if (grp >= ngroups) return;
    const bool whole = (G.most[0] | G.most[1]) == 0;   // otherwise the walk is repeated
    const int nrec = whole ? G.nrec[grp] : 0, ni = whole ? G.nitem[grp] : 0;
    const int64_t io = G.item0(grp), to = G.rec0(grp);
    LogReader rd{G.tid + to, G.tfar + to, G.tnear + to};
    int cn = 0, cf = 0;
    int2 ahead = ni > 0 ? G.lanes[io * kWave + lane] : make_int2(0, 0);   // the next item's counts
    for (int r0 = 0; r0 < nrec; r0 += kWave) {
        rd.load(r0, nrec - r0, lane);
        const int m = min(kWave, nrec - r0);
        for (int k = 0; k < m; k++) {
            const int id = __builtin_amdgcn_readlane(rd.rid, k);
            if (id >= 0) {
                cf += __builtin_amdgcn_inverse_ballot_w64(LogReader::pick(rd.rf, k)) ? 1 : 0;
                cn += __builtin_amdgcn_inverse_ballot_w64(LogReader::pick(rd.rn, k)) ? 1 : 0;
            } else if (-id <= ni) {
                int2* p = G.lanes + (io + (-id - 1)) * kWave + lane;
                const int2 c = ahead;
                if (-id < ni) ahead = p[kWave];
                *p = make_int2(cn, cf);
                cn += c.x;
                cf += c.y;
                G.after[(io + (-id - 1)) * kWave + lane] = make_int2(cn, cf);
            }
        }
    }
    if (lane < groups[3 * grp + 1]) {
        const int l = groups[3 * grp] + lane;
        near_cnt[l] = cn;
        far_cnt[l] = cf;
    }
}

// A lane's list, written four entries at a time: a store of single entries
// touches a line per lane and record (57.7 M of them, 0.47 ms at 1M).
typedef int32_t int4u __attribute__((ext_vector_type(4), aligned(4)));
struct ListOut {
    int32_t* p;
    int32_t b0 = 0, b1 = 0, b2 = 0, b3 = 0;
    int n = 0;
    __device__ inline void push(int32_t id) {
        b0 = b1;
        b1 = b2;
        b2 = b3;
        b3 = id;
        if (++n == 4) {
            *reinterpret_cast<int4u*>(p) = int4u{b0, b1, b2, b3};
            p += 4;
            n = 0;
        }
    }
    __device__ inline void flush() {   // the last n of b0..b3
        if (n == 3) p[0] = b1;
        if (n >= 2) p[n - 2] = b2;
        if (n >= 1) p[n - 1] = b3;
        p += n;
        n = 0;
    }
};

// The records to the lists: a wave an item, then a wave a group for the
// group's own records.
template <bool kExact>
__global__ __launch_bounds__(kBlock) void k_list_replay(const int32_t* __restrict__ groups, int ngroups, ListLog G,
                                                        const int64_t* near_off, const int64_t* far_off,
                                                        int32_t* near_list, int32_t* far_list) {
    const int lane = lane_id();
    auto emit = [&](const LogReader& rd, ListOut& near, ListOut& far, int q, int id) {
        const uint64_t F = LogReader::pick(rd.rf, q), N = LogReader::pick(rd.rn, q);
        if (__builtin_amdgcn_inverse_ballot_w64(F)) far.push(id);
        if (N != 0 && __builtin_amdgcn_inverse_ballot_w64(N)) near.push(id);
    };
    const int step = gridDim.x * (kBlock / kWave);
    for (int w = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; w < G.slots + ngroups; w += step) {
        const bool own = w >= G.slots;
        int grp = __builtin_amdgcn_readfirstlane(w - G.slots);
        const int64_t it = own ? 0 : G.slot<kExact>(w, ngroups, grp);
        if (it < 0) return;
        const int l = groups[3 * grp] + lane;
        const bool valid = lane < groups[3 * grp + 1];
        ListOut near{near_list + (valid ? near_off[l] : 0)}, far{far_list + (valid ? far_off[l] : 0)};
        if (!own) {
            const int2 c = G.lanes[it * kWave + lane];
            near.p += c.x;
            far.p += c.y;
            const int64_t o = G.gbase[grp] + G.item[it].y;
            const int n = G.item_n[it];
            LogReader rd{G.rid, G.rfar, G.rnear}, next = rd;
            next.load(o, n, lane);
            for (int r0 = 0; r0 < n; r0 += kWave) {
                rd = next;
                if (r0 + kWave < n) next.load(o + r0 + kWave, n - r0 - kWave, lane);
                const int m = min(kWave, n - r0);
                for (int q = 0; q < m; q++) emit(rd, near, far, q, __builtin_amdgcn_readlane(rd.rid, q));
            }
            near.flush();
            far.flush();
            if (!kExact) return;
            continue;
        }
        // the group's own records: an item's entries are passed over, up to what
        // the lane has listed before the next record
        const int n = G.nrec[grp];
        const int64_t io = G.item0(grp), to = G.rec0(grp);
        LogReader rd{G.tid + to, G.tfar + to, G.tnear + to};
        int32_t *const bn = near.p, *const bf = far.p;   // the leaf's lists
        for (int r0 = 0; r0 < n; r0 += kWave) {
            rd.load(r0, n - r0, lane);
            const int m = min(kWave, n - r0);
            for (int q = 0; q < m; q++) {
                const int id = __builtin_amdgcn_readlane(rd.rid, q);
                if (id >= 0) {
                    emit(rd, near, far, q, id);
                    continue;
                }
                // after item i the lane stands where item i's entries end
                const int2 c = G.after[(io + (-id - 1)) * kWave + lane];
                near.flush();
                far.flush();
                near.p = bn + c.x;
                far.p = bf + c.y;
            }
        }
        near.flush();
        far.flush();
        if (!kExact) return;
    }
}

// Segments: leaf of each segment, then stable order by (leaf, index).
// Leaf (DFS rank) of every segment, and the segment numbers to sort by it.
__global__ void k_seg_leaf(const int32_t* seg_node, const int32_t* leaf_rank, int nseg, int32_t* seg_leaf,
                           int32_t* ids) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    seg_leaf[s] = leaf_rank[seg_node[s]];
    ids[s] = s;
}

__global__ void k_seg_off(const int32_t* seg_leaf, const int32_t* seg_list, int nseg, int nleaf, int64_t* seg_off) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l > nleaf) return;
    // first position whose leaf >= l
    int lo = 0, hi = nseg;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (seg_leaf[seg_list[mid]] < l)
            lo = mid + 1;
        else
            hi = mid;
    }
    seg_off[l] = lo;
}

// What the host needs of a walk, in one copy: the lists' lengths, the items'
// nodes, whether a group ran out of room (the marks are cleared for the next
// walk), and the most of a group and the sum of the groups' records and items.
constexpr int kTotals = 8, kTotalsThreads = 1024;
__global__ __launch_bounds__(kTotalsThreads) void k_list_totals(const int64_t* near_end, const int64_t* far_end,
                                                                const int64_t* nodes_end, ListLog G, int ngroups,
                                                                int64_t* out) {
    __shared__ int64_t s_part[kTotalsThreads / kWave][4];
    const int k = threadIdx.x;
    int64_t v[4] = {0, 0, 0, 0};   // most records, most items, all records, all items
    for (int g = k; g < ngroups; g += blockDim.x) {
        const int64_t r = G.nrec[g], i = G.nitem[g];
        v[0] = max(v[0], r);
        v[1] = max(v[1], i);
        v[2] += r;
        v[3] += i;
    }
    auto join = [](int64_t* a, const int64_t* b) {
        for (int q = 0; q < 4; q++) a[q] = q < 2 ? max(a[q], b[q]) : a[q] + b[q];
    };
    for (int o = kWave / 2; o > 0; o >>= 1) {
        int64_t u[4];
        for (int q = 0; q < 4; q++) u[q] = __shfl_xor((long long)v[q], o, kWave);
        join(v, u);
    }
    if (lane_id() == 0)
        for (int q = 0; q < 4; q++) s_part[k / kWave][q] = v[q];
    __syncthreads();
    if (k != 0) return;
    for (int w = 1; w < (int)blockDim.x / kWave; w++) join(v, s_part[w]);
    out[0] = *near_end;
    out[1] = *far_end;
    out[2] = *nodes_end;
    out[3] = G.most[0] | G.most[1];
    for (int q = 0; q < 4; q++) out[4 + q] = v[q];
    G.most[0] = G.most[1] = 0;
}

__global__ void k_iota(int32_t* a, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) a[k] = k;
}

// Leaves and leaf groups of a single simulation.
__global__ void k_one_root_leaves(int nl, int32_t* leaf_sim, int32_t* groups) {
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nl) return;
    leaf_sim[l] = 0;
    if (l % kWave) return;
    int32_t* g = groups + 3 * (l / kWave);
    g[0] = l;
    g[1] = min(kWave, nl - l);
    g[2] = 0;
}

template <typename T>
void swap_buf(DBuf<T>& a, DBuf<T>& b) {
    std::swap(a.p, b.p);
    std::swap(a.cap, b.cap);
}

// Exclusive scans of int32 counts into int64 offsets (n + 1 outputs), one
// block per array: for short arrays, where the library's two launches per scan
// cost more than the scan.
constexpr int kScanThreads = 1024, kScanPer = 8;
__global__ __launch_bounds__(kScanThreads) void k_scan_block(const int32_t* in0, int64_t* out0, const int32_t* in1,
                                                             int64_t* out1, int n) {
    __shared__ int64_t s_w[kScanThreads / kWave];
    const int32_t* in = blockIdx.x ? in1 : in0;
    int64_t* out = blockIdx.x ? out1 : out0;
    const int t = threadIdx.x, w = t / kWave, lane = lane_id();
    int64_t carry = 0;
    for (int b = 0; b <= n; b += kScanThreads * kScanPer) {
        int v[kScanPer];
        int64_t mine = 0;
        for (int k = 0; k < kScanPer; k++) {
            const int i = b + t * kScanPer + k;
            v[k] = i < n ? in[i] : 0;
            mine += v[k];
        }
        int64_t incl = mine;
        for (int o = 1; o < kWave; o <<= 1) {
            const int64_t u = __shfl_up(incl, o, kWave);
            if (lane >= o) incl += u;
        }
        if (lane == kWave - 1) s_w[w] = incl;
        __syncthreads();
        int64_t before = carry, total = 0;
        for (int q = 0; q < kScanThreads / kWave; q++) {
            if (q < w) before += s_w[q];
            total += s_w[q];
        }
        before += incl - mine;
        for (int k = 0; k < kScanPer; k++) {
            const int i = b + t * kScanPer + k;
            if (i <= n) out[i] = before;
            before += v[k];
        }
        carry += total;
        __syncthreads();
    }
}

// exclusive scan of int32 counts into int64 offsets (n+1 outputs)
void scan_i32_to_i64(Ctx& c, const int32_t* in, int64_t* out, int64_t n) {
    size_t bytes = 0;
    VVHD_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, (int64_t)0, (size_t)n + 1, rocprim::plus<int64_t>(),
                                     c.stream));
    c.tmp.grow(bytes + 16);
    VVHD_HIP(rocprim::exclusive_scan(c.tmp.p, bytes, in, out, (int64_t)0, (size_t)n + 1, rocprim::plus<int64_t>(),
                                     c.stream));
}

// Exclusive prefix of the goes-left flags in two passes over blocks of kScanSpan
// elements: k_flag_count stores every flag and each block's count,
// k_flag_prefix adds the counts of the blocks before it to a block scan.
// The flag and prefix arrays are padded to whole blocks (zero flags).
constexpr int kScanSpan = 2048;   // 256 threads x 8 elements

__device__ inline int block_sum_256(int v, int* s_w) {
    v = wave_sum_i(v);
    const int w = threadIdx.x / kWave;
    __syncthreads();
    if (lane_id() == 0) s_w[w] = v;
    __syncthreads();
    return s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

__global__ __launch_bounds__(256) void k_flag_count(GoesLeftFlag f, int64_t m, int32_t* flag, int32_t* bcount) {
    __shared__ int s_w[4];
    const int64_t base = (int64_t)blockIdx.x * kScanSpan;
    int cnt = 0;
    for (int i = 0; i < kScanSpan / 256; i++) {
        const int64_t k = base + i * 256 + threadIdx.x;
        const int v = k < m ? f((int)k) : 0;
        flag[k] = v;
        cnt += v;
    }
    cnt = block_sum_256(cnt, s_w);
    if (threadIdx.x == 0) bcount[blockIdx.x] = cnt;
}

__global__ __launch_bounds__(256) void k_flag_prefix(const int32_t* flag, const int32_t* bcount, int32_t* P) {
    __shared__ int s_w[4];
    const int b = blockIdx.x, t = threadIdx.x, w = t / kWave;
    int pre = 0;
    for (int j = t; j < b; j += 256) pre += bcount[j];
    pre = block_sum_256(pre, s_w);
    const int64_t k0 = (int64_t)b * kScanSpan + 8 * t;
    const int4 lo = *reinterpret_cast<const int4*>(flag + k0), hi = *reinterpret_cast<const int4*>(flag + k0 + 4);
    const int v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    int ex[8], tot = 0;
    for (int i = 0; i < 8; i++) {
        ex[i] = tot;
        tot += v[i];
    }
    const int incl = wave_incl_scan(tot);
    __syncthreads();   // s_w is reused
    if (lane_id() == kWave - 1) s_w[w] = incl;
    __syncthreads();
    int woff = 0;
    for (int q = 0; q < w; q++) woff += s_w[q];
    const int start = pre + woff + incl - tot;
    *reinterpret_cast<int4*>(P + k0) = make_int4(start + ex[0], start + ex[1], start + ex[2], start + ex[3]);
    *reinterpret_cast<int4*>(P + k0 + 4) = make_int4(start + ex[4], start + ex[5], start + ex[6], start + ex[7]);
}

// P[k] = number of flags before k, for k < m (flag is written too); the
// arrays hold scan_blocks(m) * kScanSpan entries, bcount scan_blocks(m).
int64_t scan_blocks(int64_t m) { return (m + kScanSpan - 1) / kScanSpan; }

void scan_flags(Ctx& c, const GoesLeftFlag& f, int32_t* flag, int32_t* P, int32_t* bcount, int64_t m) {
    const int64_t nb = scan_blocks(m);
    hipLaunchKernelGGL(k_flag_count, dim3((unsigned)nb), dim3(256), 0, c.stream, f, m, flag, bcount);
    hipLaunchKernelGGL(k_flag_prefix, dim3((unsigned)nb), dim3(256), 0, c.stream, (const int32_t*)flag,
                       (const int32_t*)bcount, P);
}

}  // namespace

void for_level_runs(const TreeArrays& t, bool up, const std::function<void(int, int, int)>& run, int small,
                    int threads) {
    const int n = (int)t.levels.size();
    auto size = [&](int d) { return t.levels[d].second - t.levels[d].first; };
    std::vector<std::array<int, 3>> runs;
    for (int d = 0; d < n;) {
        int e = d + 1;
        if (size(d) <= small)
            while (e < n && size(e) <= small) e++;
        runs.push_back({d, e, size(d) <= small ? 1 : nblocks(size(d), threads)});
        d = e;
    }
    if (up) std::reverse(runs.begin(), runs.end());
    for (const auto& r : runs) run(r[0], r[1], r[2]);
}

void tree_build(Ctx& c, int far_criteria, double min_node, double max_node, int32_t* perm_out) {
    TreeArrays& t = c.t;
    t.built = false;   // until all of it is there: an error on the way leaves no tree
    const int nvort = (int)c.n;
    const int nh = (int)c.heat.n, nst = (int)c.streak.n;
    const int nseg = (int)c.segs_h.size();
    VVHD_CHECK(c.n + c.heat.n + c.streak.n < INT32_MAX / 2, VVHD_EINVAL, "tree_build: too many particles");
    VVHD_CHECK(far_criteria >= 0, VVHD_EINVAL, "tree_build: far_criteria must be non-negative");
    t.far_criteria = far_criteria;
    t.min_node = min_node;
    t.max_node = max_node;
    sim_sync(c);
    const int nroots = c.nsim;
    VVHD_CHECK(nroots == 1 || nh + nst == 0, VVHD_EUNSUPPORTED,
               "tree_build: heat and streak lists with several simulations in one context");
    // elements: the vortices, then the heat and the streak particles
    const int n = nvort + nh + nst;
    t.hbase = nvort;
    t.sbase = nvort + nh;
    t.nelem = n;
    if (nh + nst) {
        reserve_vortices(c, n + 1, true);
        if (nh) {
            VVHD_HIP(hipMemcpyAsync(c.x.p + nvort, c.heat.x.p, (size_t)nh * 8, hipMemcpyDeviceToDevice, c.stream));
            VVHD_HIP(hipMemcpyAsync(c.y.p + nvort, c.heat.y.p, (size_t)nh * 8, hipMemcpyDeviceToDevice, c.stream));
        }
        if (nst) {
            VVHD_HIP(hipMemcpyAsync(c.x.p + t.sbase, c.streak.x.p, (size_t)nst * 8, hipMemcpyDeviceToDevice, c.stream));
            VVHD_HIP(hipMemcpyAsync(c.y.p + t.sbase, c.streak.y.p, (size_t)nst * 8, hipMemcpyDeviceToDevice, c.stream));
        }
    }
    const int cap = 2 * (n + nseg) + 64 + nroots;
    for (auto* b : {&t.x, &t.y, &t.h, &t.w}) b->grow(cap);
    for (auto* b : {&t.blx, &t.bly, &t.trx, &t.try_, &t.path}) b->grow(cap);
    for (auto* b : {&t.v0, &t.v1, &t.ch1, &t.parent, &t.depth, &t.nseg, &t.split, &t.nleaves, &t.arrive, &t.leaf_rank,
                    &t.pre, &t.h0, &t.h1, &t.s0, &t.s1})
        b->grow(cap);
    for (auto* b : {&t.cmp_x, &t.cmp_y, &t.cmp_g, &t.cmm_x, &t.cmm_y, &t.cmm_g}) b->grow(cap);
    t.cmp_ie.grow(cap);
    t.cmm_ie.grow(cap);
    t.counters.grow(16);
    t.leaf_node.grow(cap);
    t.vleaf.grow(n + 1);
    c.iscratch0.grow(n + 1);   // element node
    const int64_t scan_pad = scan_blocks((int64_t)n + 1) * kScanSpan;
    c.iscratch1.grow(std::max<int64_t>(n + 2, scan_pad));   // flags
    c.iscratch2.grow(std::max<int64_t>(n + 2, scan_pad));   // prefix
    c.tmp.grow(scan_blocks((int64_t)n + 1) * sizeof(int32_t) + 16);   // per-block flag counts
    c.iscratch3.grow(2 * (size_t)n + 2);   // left/right positions
    DBuf<int32_t>& enode = c.iscratch0;
    int32_t* flag = c.iscratch1.p;
    int32_t* P = c.iscratch2.p;
    int32_t* left_pos = c.iscratch3.p;
    int32_t* right_pos = c.iscratch3.p + n + 1;
    DBuf<int32_t>& node_L = t.node_L;
    DBuf<int32_t>& node_m = t.node_m;
    DBuf<int32_t>& seg_node = t.seg_node;
    node_L.grow(3 * (size_t)cap);
    node_m.grow(3 * (size_t)cap);
    // subtrees: about n / kSubElems of them are expected; nodes beyond the
    // table stay with the level kernels
    const int sub_cap = 4 * (n / kSubElems + nroots) + 4096;
    t.sub_lev.grow((size_t)sub_cap * kSubLevels);
    t.sub_nlev.grow(sub_cap);
    t.lev_d.grow(kMaxLevels + 2);
    seg_node.grow(nseg + 1);
    NodeView nv = view(t);
    hipStream_t s = c.stream;

    hipLaunchKernelGGL(k_init_roots, dim3(nblocks(nroots)), dim3(kBlock), 0, s, nv, nroots, (const int64_t*)c.sim_off.p,
                       t.counters.p, t.lev_d.p, t.hbase, t.sbase, n);
    hipLaunchKernelGGL(k_iota, dim3(nblocks(n)), dim3(kBlock), 0, s, c.id.p, n);
    hipLaunchKernelGGL(k_fill_roots, dim3(nblocks(n)), dim3(kBlock), 0, s, enode.p, n, (const int64_t*)c.sim_off.p,
                       nroots);
    if (nseg)
        hipLaunchKernelGGL(k_seg_roots, dim3(nblocks(nseg)), dim3(kBlock), 0, s, nv, (const int32_t*)c.seg_root.p,
                           nseg, seg_node.p);
    if (n && nroots <= kTopNodes)
        hipLaunchKernelGGL(k_bbox_top, dim3(nblocks(n, kTopChunk)), dim3(kBlock), 0, s, nv, (const int32_t*)nullptr,
                           (const int32_t*)enode.p, c.x.p, c.y.p, n);
    else if (n)
        hipLaunchKernelGGL(k_bbox_elems, dim3(nblocks(n)), dim3(kBlock), 0, s, nv, (const int32_t*)enode.p, c.x.p,
                           c.y.p, n);
    if (nseg)
        hipLaunchKernelGGL(k_root_segs, dim3(nblocks(nseg)), dim3(kBlock), 0, s, nv, c.segs.p,
                           (const int32_t*)c.seg_root.p, nseg);

    // One level per iteration over the whole list, its kernels taking their node
    // range from the device counters.  Few nodes fit a workgroup before a root
    // has been halved down to kSubElems elements, so the levels up to there are
    // queued without asking; from there on k_subtree takes what fits, and the
    // host reads after it whether anything is left.
    auto launch_level = [&](int d) {
        const int node_blocks = 1024;
        hipLaunchKernelGGL(k_decide, dim3(node_blocks), dim3(kBlock), 0, s, nv, t.counters.p, cap, min_node, max_node);
        scan_flags(c, GoesLeftFlag{nv, enode.p, c.x.p, c.y.p, n}, flag, P, reinterpret_cast<int32_t*>(c.tmp.p), n + 1);
        hipLaunchKernelGGL(k_ranks, dim3(nblocks(n + 1)), dim3(kBlock), 0, s, nv, enode.p, P, n, t.hbase, t.sbase, cap,
                           node_L.p, node_m.p, left_pos, right_pos, t.counters.p, (const int32_t*)flag, t.lev_d.p, d + 1);
        // the children of level d number at most nroots 2^(d+1)
        const bool top = ((int64_t)nroots << std::min<int>(d + 1, 30)) <= kTopNodes;
        hipLaunchKernelGGL(k_swap, dim3(nblocks(n)), dim3(kBlock), 0, s, nv, enode.p, flag, P, n, t.hbase, t.sbase,
                           cap, node_L.p, node_m.p, left_pos, right_pos, c.x.p, c.y.p, c.id.p);
        if (top && n)
            hipLaunchKernelGGL(k_bbox_top, dim3(nblocks(n, kTopChunk)), dim3(kBlock), 0, s, nv,
                               (const int32_t*)(t.counters.p + 2), (const int32_t*)enode.p, c.x.p, c.y.p, n);
        else if (n) {
            // at most nroots 2^(d+1) children; 16 lanes each once they average under 256 elements
            const int64_t kids = std::min<int64_t>((int64_t)nroots << std::min<int>(d + 1, 30), cap);
            const bool small = (int64_t)n < 256 * kids;
            const int64_t waves = small ? (kids + 3) / 4 : kids;
            const int grid = (int)std::min<int64_t>(2048, std::max<int64_t>(1, (waves + 3) / 4));
            if (small)
                hipLaunchKernelGGL(k_child_boxes<16>, dim3(grid), dim3(kBlock), 0, s, nv,
                                   (const int32_t*)t.counters.p, c.x.p, c.y.p);
            else
                hipLaunchKernelGGL(k_child_boxes<64>, dim3(grid), dim3(kBlock), 0, s, nv,
                                   (const int32_t*)t.counters.p, c.x.p, c.y.p);
        }
        if (nseg)
            hipLaunchKernelGGL(k_seg_step, dim3(nblocks(nseg)), dim3(kBlock), 0, s, nv, c.segs.p, nseg, seg_node.p);
    };
    // Elements of the root whose nodes fit first.  Roots of a batch differ: 64 of
    // 14k to 400k elements, taken when the largest one's nodes fitted, gave 25k
    // subtrees of a few elements each (a tree 23 ms, now 13).
    int64_t start = n;
    for (int q = 0; nroots > 1 && q < nroots; q++) {
        const int64_t m = c.sim_off_h[q + 1] - c.sim_off_h[q];
        if (m > 0) start = std::min(start, m);
    }
    int depth = 0;
    for (; (start >> depth) > kSubElems; depth++) launch_level(depth);
    int32_t* hc = c.lev_counters;   // pinned
    for (;; depth++) {
        const int grid = (int)std::min<int64_t>(2 * c.n_cu, (int64_t)nroots << std::min(depth, 20));
        hipLaunchKernelGGL(k_subtree, dim3(grid), dim3(kSubThreads), 0, s, nv, t.counters.p, cap, min_node, max_node,
                           enode.p, c.x.p, c.y.p, c.id.p, (const vvhd_seg*)c.segs.p, nseg, seg_node.p, t.sub_lev.p,
                           t.sub_nlev.p, sub_cap);
        VVHD_HIP(hipMemcpyAsync(hc, t.counters.p, 10 * sizeof(int32_t), hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipMemcpyAsync(hc + 16, t.lev_d.p, (depth + 1) * sizeof(int2), hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipStreamSynchronize(s));
        if (hc[4] != 0 || depth >= kMaxLevels - 1) break;   // refused below
        if (hc[6] == 0) break;                              // the level's nodes are all decided
        hipLaunchKernelGGL(k_level_begin, dim3(1), dim3(64), 0, s, t.counters.p);
        launch_level(depth);
    }
    // tree order of the remaining fields (also where the build is refused: the
    // positions have been moved)
    hipLaunchKernelGGL(k_gather, dim3(nblocks(nvort)), dim3(kBlock), 0, s, c.id.p, nvort, c.g.p, c.vx.p, c.vy.p,
                       c.ie.p, c.g2.p, c.vx2.p, c.vy2.p, c.ie2.p);
    swap_buf(c.g, c.g2);
    swap_buf(c.vx, c.vx2);
    swap_buf(c.vy, c.vy2);
    swap_buf(c.ie, c.ie2);
    VVHD_CHECK(hc[4] != 1, VVHD_ENOMEM, "tree_build: node capacity exceeded");
    VVHD_CHECK(hc[4] == 0 && depth < kMaxLevels - 1, VVHD_EUNSUPPORTED, "tree_build: tree deeper than supported");
    t.nnodes = hc[0];
    t.nleaves_h = hc[1];
    t.max_depth = hc[5];
    t.nsub = std::min(hc[7], sub_cap);
    // node ranges of the levels over the whole list
    std::vector<std::pair<int, int>>& levels = t.levels;
    levels.clear();
    for (int d = 0; d <= depth; d++) levels.push_back({hc[16 + 2 * d], hc[17 + 2 * d]});
    const int nl = t.nleaves_h;

    if (perm_out && nvort) VVHD_HIP(hipMemcpyAsync(perm_out, c.id.p, (size_t)nvort * 4, hipMemcpyDeviceToHost, s));
    // the heat and streak lists in their new order
    for (int q = 0; q < 2; q++) {
        PList& L = q == 0 ? c.heat : c.streak;
        const int base = q == 0 ? t.hbase : t.sbase, m = q == 0 ? nh : nst;
        if (!m) continue;
        hipLaunchKernelGGL(k_gather_list, dim3(nblocks(m)), dim3(kBlock), 0, s, c.id.p + base, m, base, c.x.p + base,
                           c.y.p + base, L.g.p, L.vx.p, L.vy.p, L.ie.p, L.x2.p, L.y2.p, L.g2.p, L.vx2.p, L.vy2.p,
                           L.ie2.p);
        L.swap_buffers();
    }

    // leaf counts and monopoles bottom-up, DFS ranks top-down
    const CMView cm = cm_view(t);
    if (t.nsub)
        hipLaunchKernelGGL(k_up_subs, dim3(t.nsub), dim3(kBlock), 0, s, nv, cm, (const int2*)t.sub_lev.p,
                           (const int32_t*)t.sub_nlev.p, c.x.p, c.y.p, c.g.p, t.nleaves.p);
    for_level_runs(t, true, [&](int l0, int l1, int grid) {
        hipLaunchKernelGGL(k_up_levels, dim3(grid), dim3(kPassThreads), 0, s, nv, cm, (const int2*)t.lev_d.p, l0, l1,
                           c.x.p, c.y.p, c.g.p, t.nleaves.p);
    }, kPassNodes, kPassThreads);
    int32_t* first = t.arrive.p;
    t.root_first.grow(nroots + 1);
    hipLaunchKernelGGL(k_root_first, dim3(1), dim3(1), 0, s, t.nleaves.p, nroots, first, t.root_first.p, t.pre.p);
    for_level_runs(t, false, [&](int l0, int l1, int grid) {
        hipLaunchKernelGGL(k_down_levels, dim3(grid), dim3(kPassThreads), 0, s, nv, (const int2*)t.lev_d.p, l0, l1,
                           t.nleaves.p, first, t.leaf_rank.p, t.leaf_node.p, t.vleaf.p, t.pre.p);
    }, kPassNodes, kPassThreads);
    if (t.nsub)
        hipLaunchKernelGGL(k_down_subs, dim3(t.nsub), dim3(kBlock), 0, s, nv, (const int2*)t.sub_lev.p,
                           (const int32_t*)t.sub_nlev.p, t.nleaves.p, first, t.leaf_rank.p, t.leaf_node.p, t.vleaf.p,
                           t.pre.p);
    // leaf -> simulation and the list builder's leaf groups (64 leaves of one root)
    t.leaf_sim.grow(nl + 1);
    if (nroots == 1) {
        t.ngroups = (nl + kWave - 1) / kWave;
        t.groups.grow(3 * (size_t)t.ngroups + 3);
        if (nl)
            hipLaunchKernelGGL(k_one_root_leaves, dim3(nblocks(nl)), dim3(kBlock), 0, s, nl, t.leaf_sim.p, t.groups.p);
    } else {
        std::vector<int32_t> rf(nroots + 1), grp;
        VVHD_HIP(hipMemcpyAsync(rf.data(), t.root_first.p, (nroots + 1) * 4, hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipStreamSynchronize(s));
        if (nl)
            hipLaunchKernelGGL(k_leaf_sim, dim3(nblocks(nl)), dim3(kBlock), 0, s, (const int32_t*)t.root_first.p,
                               nroots, nl, t.leaf_sim.p);
        for (int r = 0; r < nroots; r++)
            for (int f = rf[r]; f < rf[r + 1]; f += kWave) grp.insert(grp.end(), {f, std::min(kWave, rf[r + 1] - f), r});
        t.ngroups = (int)grp.size() / 3;
        t.groups.grow(grp.size() + 3);
        if (!grp.empty())
            VVHD_HIP(hipMemcpyAsync(t.groups.p, grp.data(), grp.size() * 4, hipMemcpyHostToDevice, s));
    }
    // segments per leaf
    t.seg_off.grow(nl + 1);
    t.seg_leaf.grow(nseg + 1);
    t.seg_list.grow(nseg + 1);
    if (nseg) {
        // segments of every leaf in their own order (the stable partition of
        // the segment list, TSortedTree.cpp:139-148): a stable radix sort of
        // the segment numbers by leaf
        t.seg_keys.grow(nseg + 1);
        t.seg_ids.grow(nseg + 1);
        hipLaunchKernelGGL(k_seg_leaf, dim3(nblocks(nseg)), dim3(kBlock), 0, s, seg_node.p, t.leaf_rank.p, nseg,
                           t.seg_leaf.p, t.seg_ids.p);
        int bits = 1;
        while (bits < 31 && (1 << bits) <= nl) bits++;
        size_t bytes = 0;
        VVHD_HIP(rocprim::radix_sort_pairs(nullptr, bytes, t.seg_leaf.p, t.seg_keys.p, t.seg_ids.p, t.seg_list.p,
                                           (unsigned)nseg, 0, bits, s));
        c.tmp.grow(bytes + 16);
        VVHD_HIP(rocprim::radix_sort_pairs(c.tmp.p, bytes, t.seg_leaf.p, t.seg_keys.p, t.seg_ids.p, t.seg_list.p,
                                           (unsigned)nseg, 0, bits, s));
        hipLaunchKernelGGL(k_seg_off, dim3(nblocks(nl + 1)), dim3(kBlock), 0, s, t.seg_leaf.p, t.seg_list.p, nseg, nl,
                           t.seg_off.p);
    } else {
        VVHD_HIP(hipMemsetAsync(t.seg_off.p, 0, (size_t)(nl + 1) * 8, s));
    }
    tree_lists(c);
    pack_boxes(c);
    t.built = true;
}

void pack_boxes(Ctx& c) {
    TreeArrays& t = c.t;
    t.pbox.grow(std::max(t.nnodes, 1));
    if (t.nnodes)
        hipLaunchKernelGGL(k_pack_boxes, dim3(nblocks(t.nnodes)), dim3(kBlock), 0, c.stream, view(t), t.nnodes,
                           t.pbox.p);
}

void tree_lists(Ctx& c) {
    TreeArrays& t = c.t;
    const int nl = t.nleaves_h;
    NodeView nv = view(t);
    hipStream_t s = c.stream;
    t.cnt_near.grow(nl + 1);
    t.cnt_far.grow(nl + 1);
    t.near_off.grow(nl + 1);
    t.far_off.grow(nl + 1);
    t.trav.grow((size_t)t.nnodes * sizeof(TravNode));
    TravNode* tn = reinterpret_cast<TravNode*>(t.trav.p);
    t.log.most.grow(2);
    t.log.totals.grow(kTotals);
    t.cmk.grow(4 * (size_t)t.nnodes + 1);
    hipLaunchKernelGGL(k_trav_nodes, dim3(nblocks(t.nnodes)), dim3(kBlock), 0, s, nv, t.nnodes, t.pre.p, t.nleaves.p,
                       tn, t.log.most.p, cm_view(t), t.cmk.p);
    const double fc = (double)t.far_criteria;
    // subtrees walked by waves of their own: a walk over the top of the tree
    // has about 2 nnodes / item_nodes steps, one of an item at most item_nodes
    const int item_nodes = std::min(512, std::max(32, (int)(1.4 * std::sqrt((double)t.nnodes))));
    const int ng = t.ngroups;
    // a wave each, or what a launch may hold of them (its threads are a 32-bit
    // number): with room as counted the kernels over items go round the rest
    auto wave_grid = [](int64_t waves) {
        return dim3((unsigned)std::clamp<int64_t>((waves + kBlock / kWave - 1) / (kBlock / kWave), 1, (1 << 24) - 1));
    };
    ListLogBufs& b = t.log;
    // The same room for every group, as the last walk needed it, unless one
    // group among many needed far more than the others (a leaf spread wide
    // around the rest is near to all of them) and it comes to more than 128
    // MiB: the floors then, which most groups stay under.  Where they do not
    // do, the counts of the first walk over the groups give every group the
    // room that it needs in a second (55 us at 1M, against 400 us for the
    // items' walk).  With the widest group's room for all, ten strays around 4M
    // vortices took 24 GiB, and around 8M the launches of 12020 x 6211 waves
    // were larger than a grid may be.
    // (Room of no use costs, too: 150 us at 4M for nine idle items a group.)
    constexpr int64_t kRecFloor = 512, kItemFloor = 64, kNodeFloor = 6144;   // of a group
    auto room = [](int ng, int64_t most, int64_t all, int64_t floor, int64_t small) {
        const int64_t r = std::max(floor, most);
        return r * ng <= std::max(small, 4 * all + floor * ng) ? r : floor;
    };
    // what successive walks need stays where it does not fall by a fifth
    auto follow = [](int64_t& most, int64_t now) {
        if (now > most || 5 * now < 4 * most) most = now;
    };
    // The log takes 0.5 to 0.7 KB a vortex.  Where that is more than an eighth of
    // the memory free (some 50M vortices, or little memory left), the groups are
    // walked in parts, once for the counts and once more for the lists.  In one
    // part the tree of 96M vortices took 264 GiB, so 156; 150M did not fit.
    auto need = [&]() {
        return ng * (20 * room(ng, b.last_recs, b.last_all_recs, kRecFloor, 1 << 22) +
                     1048 * room(ng, b.last_items, b.last_all_items, kItemFloor, 1 << 17) +
                     20 * std::max(kNodeFloor, b.last_nodes));
    };
    auto parts_of = [&]() {
        const int64_t want = need(), have = b.bytes();
        if (want <= (1 << 30) || want <= have) return 1;
        size_t free_b = 0, all_b = 0;
        VVHD_HIP(hipMemGetInfo(&free_b, &all_b));
        const int64_t may = std::max<int64_t>(1 << 29, ((int64_t)free_b + have) / 8);
        return (int)std::min<int64_t>((want + may - 1) / may, ng);
    };
    int parts = parts_of();
    auto first_of = [&](int k) { return (int)((int64_t)t.ngroups * k / parts); };
    // The walk of the groups of part k: their logs, which a replay reads, and
    // their leaves' counts; where it is the only part also the lists' offsets and
    // lengths.  plan: where the counts ask for more parts, only their number.
    struct Walk {
        ListLog G;
        const int32_t* groups;
        int ng;
        bool exact;
        int64_t nnear, nfar;
        int parts;
    };
    auto scan_counts = [&]() {
        if (nl <= 65536) {
            hipLaunchKernelGGL(k_scan_block, dim3(2), dim3(kScanThreads), 0, s, (const int32_t*)t.cnt_near.p,
                               t.near_off.p, (const int32_t*)t.cnt_far.p, t.far_off.p, nl);
        } else {
            scan_i32_to_i64(c, t.cnt_near.p, t.near_off.p, nl);
            scan_i32_to_i64(c, t.cnt_far.p, t.far_off.p, nl);
        }
    };
    auto walk = [&](int k, bool plan) {
        const int g0 = first_of(k), ng = first_of(k + 1) - g0;
        const bool all = parts == 1;
        Walk W{};
        W.parts = parts;
        W.groups = (const int32_t*)t.groups.p + 3 * (size_t)g0;
        W.ng = ng;
        int64_t R, S, recs, items;   // room of a group, and in all
        auto same_room = [&]() {
            R = room(ng, b.last_recs, b.last_all_recs, kRecFloor, 1 << 22);
            S = room(ng, b.last_items, b.last_all_items, kItemFloor, 1 << 17);
            S = std::min<int64_t>(S, (1 << 25) / std::max(ng, 1));   // a wave each in one launch
            recs = R * ng;
            items = S * ng;
        };
        same_room();
        // the items' records: what the criteria in use need, or what was counted
        int64_t nodes = ng * kNodeFloor;
        for (;;) {
            VVHD_CHECK(items < (1 << 30), VVHD_ENOMEM, "tree_build: too many parts of the list walk");
            b.grow(ng, recs, items, nodes);
            W.G = ListLog{(int)R, (int)S, W.exact ? b.tbase.p : nullptr, W.exact ? b.ibase.p : nullptr, (int)items,
                          (int64_t)b.rid.cap, b.tid.p, b.tfar.p, b.tnear.p, b.nrec.p, b.nitem.p, b.gnodes.p, b.gbase.p,
                          b.item.p, b.item_mask.p, b.item_n.p, b.item_grp.p, b.lanes.p, b.after.p, b.rid.p, b.rfar.p,
                          b.rnear.p, b.most.p};
            if (ng)
                hipLaunchKernelGGL(k_list_top, wave_grid(ng), dim3(kBlock), 0, s, nv, (const TravNode*)tn,
                                   (const int32_t*)t.pre.p, W.groups, ng, t.leaf_node.p, fc, item_nodes, W.G);
            // (one block scans 65536 counts in about 12 us)
            if (ng <= 65536)
                hipLaunchKernelGGL(k_scan_block, dim3(1), dim3(kScanThreads), 0, s, (const int32_t*)b.gnodes.p,
                                   b.gbase.p, (const int32_t*)nullptr, (int64_t*)nullptr, ng);
            else
                scan_i32_to_i64(c, b.gnodes.p, b.gbase.p, ng);
            if (ng) {
                hipLaunchKernelGGL(W.exact ? k_list_items<true> : k_list_items<false>, wave_grid(items), dim3(kBlock), 0,
                                   s, nv, (const TravNode*)tn, W.groups, ng, t.leaf_node.p, fc, W.G);
                hipLaunchKernelGGL(k_list_sums, wave_grid(ng), dim3(kBlock), 0, s, W.groups, ng, W.G, t.cnt_near.p,
                                   t.cnt_far.p);
            }
            if (all) scan_counts();
            // lengths of the near and the far lists (of all groups), the items'
            // nodes, out of room, then most and all of the records and the items
            int64_t tot[kTotals];
            hipLaunchKernelGGL(k_list_totals, dim3(1),
                               dim3(std::clamp((ng + 255) / 256 * kWave, kWave, kTotalsThreads)), 0, s,
                               (const int64_t*)t.near_off.p + nl, (const int64_t*)t.far_off.p + nl,
                               (const int64_t*)b.gbase.p + ng, W.G, ng, b.totals.p);
            VVHD_HIP(hipGetLastError());   // no lengths from a launch that was refused
            VVHD_HIP(hipMemcpyAsync(tot, b.totals.p, sizeof(tot), hipMemcpyDeviceToHost, s));
            VVHD_HIP(hipStreamSynchronize(s));
            follow(b.last_recs, tot[4]);
            follow(b.last_items, tot[5]);
            b.last_all_recs = tot[6];
            b.last_all_items = tot[7];
            b.last_nodes = tot[2] / std::max(ng, 1);
            nodes = std::max(nodes, tot[2]);
            if (plan && (tot[3] || tot[2] > W.G.cap)) {
                W.parts = std::max(parts, parts_of());
                if (W.parts > parts) return W;
            }
            if (tot[3]) {
                same_room();
                W.exact = R < tot[4] || S < tot[5];
                if (W.exact) {
                    scan_i32_to_i64(c, b.nrec.p, b.tbase.p, ng);
                    scan_i32_to_i64(c, b.nitem.p, b.ibase.p, ng);
                    recs = tot[6];
                    items = tot[7];
                }
                continue;
            }
            if (tot[2] > W.G.cap) continue;
            W.nnear = tot[0];
            W.nfar = tot[1];
            return W;
        }
    };
    auto replay = [&](const Walk& W) {
        if (W.ng)
            hipLaunchKernelGGL(W.exact ? k_list_replay<true> : k_list_replay<false>, wave_grid((int64_t)W.G.slots + W.ng),
                               dim3(kBlock), 0, s, W.groups, W.ng, W.G, (const int64_t*)t.near_off.p,
                               (const int64_t*)t.far_off.p, t.near_list.p, t.far_list.p);
    };
    Walk last{};
    for (int k = 0; k < parts; k++) {
        last = walk(k, true);
        if (last.parts == parts) continue;
        parts = last.parts;   // from the first one, with smaller ones
        if (b.bytes() / 5 > need() / (4 * parts)) b.release_walk();
        k = -1;
    }
    bool again = false;   // the last part, too, in smaller ones
    if (parts > 1) {
        scan_counts();
        int64_t ends[2];
        VVHD_HIP(hipMemcpyAsync(&ends[0], t.near_off.p + nl, 8, hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipMemcpyAsync(&ends[1], t.far_off.p + nl, 8, hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipStreamSynchronize(s));
        last.nnear = ends[0];
        last.nfar = ends[1];
        size_t free_b = 0, all_b = 0;
        VVHD_HIP(hipMemGetInfo(&free_b, &all_b));
        again = 4 * (ends[0] + ends[1]) + (1 << 30) > (int64_t)free_b && t.far_list.cap <= (size_t)ends[1];
        if (again) b.release_walk();   // the lists first
    }
    t.nnear = last.nnear;
    t.nfar = last.nfar;
    t.near_list.grow(t.nnear + 1);
    t.far_list.grow(t.nfar + 1);
    if (again)
        parts = std::max(parts, parts_of());
    else
        replay(last);
    for (int k = 0; k < parts - !again; k++) replay(walk(k, false));
}

}  // namespace vvhd
