// epsilon.hip -- MEpsilonFast::CalcEpsilonFast (MEpsilonFast.cpp:11-63) on
// the GPU, with the reference's sequential merge semantics.
//
// The reference visits targets leaf by leaf in DFS order, i.e. in array
// order, and for each searches the two nearest vortices (g != 0, not itself)
// of its near leaves; ties go to the first found.  Because leaves in DFS
// order hold increasing array ranges, "first found" is "smaller index", so
// the result is the top-2 under the order (d^2, index): order independent,
// hence computable in parallel.  Distances are FP64 with the reference's
// operation order (no contraction), so indices are bit-exact.
//
// A merge (:111-126) mutates the target and zeroes its partner; every later
// target sees the mutated state.  Pass 1 computes every target on the
// unmodified state and flags the targets that would merge.  When flags exist,
// the sequential outcome is found as a fixed point, in parallel (merge_rounds
// below): the visit of target i depends only on the merges of targets before
// it, so each round evaluates every target whose surroundings the last round
// changed against the merges assumed so far, seen as of i, until no merge
// changes.  After k rounds every target whose chain of dependencies is
// shorter than k holds its sequential result, and a state that a round leaves
// unchanged is the sequential one.  Where chains are long, the targets left
// are visited one by one in order (k_merge_in_order).
//
// Pass 1 prunes near leaves by box distance: leaves touching the target leaf
// are scanned first, then only leaves whose box distance does not exceed the
// largest second-neighbour distance found.  Box distances are computed with
// the same monotone rounded operations, so pruning never drops a candidate.

#include "common.hpp"
#include "near_flat.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

#pragma clang fp contract(off)

namespace vvhd {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
inline int nblocks(int64_t n, int b = kBlock) { return (int)std::max<int64_t>(1, (n + b - 1) / b); }

__device__ inline double sgn(double x) { return (x > 0) ? 1 : ((x < 0) ? -1 : 0); }

// Top-2 state under the order (d, index); index -1 marks an empty slot whose
// distance is DBL_MAX (the reference's initial res1/res2).
struct Top2 {
    double d1, d2;
    int i1, i2;
};

__device__ inline bool less_di(double d, int j, double dc, int ic) {
    return d < dc || (d == dc && ic >= 0 && j < ic);
}

__device__ inline void top2_insert(Top2& t, double d, int j) {
    if (less_di(d, j, t.d1, t.i1)) {
        t.d2 = t.d1;
        t.i2 = t.i1;
        t.d1 = d;
        t.i1 = j;
    } else if (less_di(d, j, t.d2, t.i2)) {
        t.d2 = d;
        t.i2 = j;
    }
}

__device__ inline void top2_merge(Top2& t, const Top2& o) {
    if (o.i1 >= 0) top2_insert(t, o.d1, o.i1);
    if (o.i2 >= 0) top2_insert(t, o.d2, o.i2);
}

__device__ inline Top2 top2_shfl_xor(const Top2& t, int mask) {
    Top2 o;
    o.d1 = __shfl_xor(t.d1, mask, kWave);
    o.d2 = __shfl_xor(t.d2, mask, kWave);
    o.i1 = __shfl_xor(t.i1, mask, kWave);
    o.i2 = __shfl_xor(t.i2, mask, kWave);
    return o;
}

__device__ inline Top2 top2_empty() { return Top2{DBL_MAX, DBL_MAX, -1, -1}; }

// (lv->r - lobj->r).abs2() of MEpsilonFast.cpp:141
__device__ inline double dist2(double tx, double ty, double sx, double sy) {
    const double dx = tx - sx, dy = ty - sy;
    return dx * dx + dy * dy;
}

// nearestBodySegment (MEpsilonFast.cpp:214-253) for every leaf centre, then
// the merge criterion and the epsilon floor (:29-47), one wave per leaf.  The
// bodies searched are those of the leaf's simulation, [sim_body[s],
// sim_body[s+1]).  Among the segments of the near leaves the reference keeps
// the first nearest in list order: the lanes take the near entries in turn
// and the first of equal distances wins.  Without one it walks the bodies'
// segments, skipping nine after each that is no nearer: the lanes compute 64
// distances at a time and the walk reads them from the lanes.  (One thread
// per leaf, every load waiting for the one before: 210-640 us a call.)
__global__ __launch_bounds__(kBlock) void k_leaf_criteria(TreeDev T, const vvhd_seg* segs, const int32_t* body_range,
                                                          const int32_t* sim_body, const int32_t* leaf_sim, int merge,
                                                          double* crit_out, double* restr_out) {
    const int l = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    if (l >= T.nleaf) return;
    const int lane = lane_id();
    const int sim = leaf_sim[l];
    const int b0 = sim_body[sim], b1 = sim_body[sim + 1];
    if (b0 == b1) {   // no segment in the simulation: criterion 0 (or NaN), floor 0
        if (lane == 0) {
            crit_out[l] = merge ? 0.0 : __builtin_nan("");
            restr_out[l] = 0;
        }
        return;
    }
    const int L = T.leaf_node[l];
    const double px = T.nx[L], py = T.ny[L];
    int att = -1;
    double res = DBL_MAX;
    int64_t where = INT64_MAX;   // near entry of the candidate
    for (int64_t e = T.near_off[l] + lane; e < T.near_off[l + 1]; e += kWave) {
        const int m = T.leaf_rank[T.near_list[e]];
        const int64_t q1 = T.seg_off[m + 1];
        for (int64_t q = T.seg_off[m]; q < q1; q++) {
            const int s = T.seg_list[q];
            const double d2 = dist2(px, py, segs[s].x, segs[s].y);
            if (d2 < res) {
                res = d2;
                att = s;
                where = e;
            }
        }
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const double d = __shfl_xor(res, o, kWave);
        const int a = __shfl_xor(att, o, kWave);
        const int64_t w = __shfl_xor(where, o, kWave);
        if (a >= 0 && (d < res || (d == res && w < where))) {
            res = d;
            att = a;
            where = w;
        }
    }
    if (att < 0) {
        res = DBL_MAX;
        for (int b = b0; b < b1; b++) {
            const int f = body_range[2 * b], cnt = body_range[2 * b + 1];
            for (int k = 0; k < cnt;) {
                const int k0 = k, s = f + min(k0 + lane, cnt - 1);
                const double mine = dist2(px, py, segs[s].x, segs[s].y);
                while (k < min(k0 + kWave, cnt)) {
                    const double d2 = __shfl(mine, k - k0, kWave);
                    if (d2 < res) {
                        res = d2;
                        att = f + k;
                        k++;
                    } else {
                        k += 10;   // the reference's "speed up" skip
                    }
                }
            }
        }
    }
    if (lane != 0) return;
    double crit;
    if (merge) {
        if (att >= 0) {
            const double dlx = segs[att].dlx, dly = segs[att].dly;
            const double ddx = px - segs[att].x, ddy = py - segs[att].y;
            crit = 0.16 * (dlx * dlx + dly * dly) * (1. + sqrt(ddx * ddx + ddy * ddy));
        } else {
            crit = 0;
        }
    } else {
        crit = __builtin_nan("");
    }
    double restr = 0;
    if (att >= 0) {
        const double dlx = segs[att].dlx, dly = segs[att].dly;
        restr = sqrt(dlx * dlx + dly * dly) * (1.0 / 3.0);
    }
    crit_out[l] = crit;
    restr_out[l] = restr;
}

constexpr int kStageE = 256;   // staged sources of a wave (pass 1)

// Pass 1: top-2 of every target on the unmodified state, one wave per leaf
// and chunk of up to 16 targets.  The sources (g != 0) of the selected near
// leaves are staged in LDS, FP64, and lane (target t = l % ntc, slot
// s = l / ntc) runs over every nslot-th of them; the slots' top-2s combine
// afterwards (the top-2 under (d^2, index) does not depend on the order).
// First the leaves touching the target leaf, then those whose box lies
// within the largest second-neighbour distance found, without the sources
// that are farther than it from the target leaf's box.
// Bound by the latency of the staging loads.  A leaf per block: four leaves of
// unequal work in one held 32 KB of LDS until the last had finished, and each
// staged source was found by a search over the entries' offsets.
__global__ __launch_bounds__(kWave) void k_eps_top2(TreeDev T, const double* x, const double* y, const double* g,
                                                     int merge, const double* leaf_crit, int32_t* nn1, int32_t* nn2,
                                                     double* d1o, double* d2o, uint8_t* eflag, int32_t* ecount,
                                                     int32_t* flag_list) {
    __shared__ double sx[kStageE], sy[kStageE];
    __shared__ int sj[kStageE], sidx[kStageE];   // sidx: the vortices being staged
    const int l = xcd_block(blockIdx.x, gridDim.x);
    if (l >= T.nleaf) return;
    const int lane = lane_id();
    const int L = T.leaf_node[l];
    const int v0 = T.v0[L], v1 = T.v1[L];
    const double crit = leaf_crit[l];
    const double4 box = T.pbox[L];
    const int64_t e0 = T.near_off[l], e1 = T.near_off[l + 1];
    for (int base = v0 + 16 * (int)blockIdx.y; base < v1; base += 16 * (int)gridDim.y) {
        const int ntc = min(16, v1 - base);
        const int nslot = kWave / ntc;
        const int t = lane % ntc, slot = lane / ntc;
        const int i = base + t;
        const double tx = x[i], ty = y[i], tg = g[i];
        const bool active = tg != 0 && slot < nslot;
        Top2 st = top2_empty();
        auto compute = [&](int nsrc) {
            wave_sync();
            if (active) {
                auto one = [&](int j, double px, double py) {
                    if (j != i) top2_insert(st, dist2(tx, ty, px, py), j);
                };
                int k = slot;
                for (; k + 3 * nslot < nsrc; k += 4 * nslot) {
                    int j[4];
                    double px[4], py[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        j[u] = sj[k + u * nslot];
                        px[u] = sx[k + u * nslot];
                        py[u] = sy[k + u * nslot];
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++) one(j[u], px[u], py[u]);
                }
                for (; k < nsrc; k += nslot) one(sj[k], sx[k], sy[k]);
            }
            wave_sync();
        };
        // sources of the near leaves with lo < box distance <= hi
        auto stage_scan = [&](double lo, double hi) {
            int fill = 0;
            for (int64_t eb = e0; eb < e1; eb += kWave) {
                const int64_t e = eb + lane;
                int cnt = 0, j0 = 0;
                if (e < e1) {
                    const int M = T.near_list[e];
                    const double bd = box_dist2p(T, L, M);
                    if (bd > lo && bd <= hi) {
                        j0 = T.v0[M];
                        cnt = T.v1[M] - j0;
                    }
                }
                const int incl = wave_incl_scan(cnt);
                const int off = incl - cnt;
                const int tot = __shfl(incl, kWave - 1, kWave);
                if (tot == 0) continue;
                for (int done = 0; done < tot;) {
                    const int take = min(tot - done, kStageE - fill);
                    // each lane lists the vortices of its leaf that fall in this chunk
                    for (int k = max(off, done); k < min(off + cnt, done + take); k++) sidx[k - done] = j0 + (k - off);
                    wave_sync();
                    for (int q0 = 0; q0 < take; q0 += kWave) {
                        const int q = q0 + lane;
                        int j = 0;
                        double px = 0, py = 0;
                        bool on = false;
                        if (q < take) {
                            j = sidx[q];
                            px = x[j];
                            py = y[j];
                            const double bx = fmax(0.0, fmax(box.x - px, px - box.z));
                            const double by = fmax(0.0, fmax(box.y - py, py - box.w));
                            on = g[j] != 0 && (hi <= 0.0 || !(bx * bx + by * by > hi));
                        }
                        const uint64_t m = __ballot(on);
                        if (on) {
                            const int k = fill + __popcll(m & ((1ull << lane) - 1));
                            sx[k] = px;
                            sy[k] = py;
                            sj[k] = j;
                        }
                        fill += __popcll(m);
                    }
                    done += take;
                    if (fill == kStageE) {
                        compute(fill);
                        fill = 0;
                    }
                    wave_sync();   // the next chunk rewrites the index list
                }
            }
            if (fill) compute(fill);
        };
        auto combine = [&](Top2 s) {
            Top2 c = top2_empty();
            for (int q = 0; q < nslot; q++) {
                Top2 o;
                const int src = t + ntc * q;
                o.d1 = __shfl(s.d1, src, kWave);
                o.d2 = __shfl(s.d2, src, kWave);
                o.i1 = __shfl(s.i1, src, kWave);
                o.i2 = __shfl(s.i2, src, kWave);
                top2_merge(c, o);
            }
            return c;
        };
        stage_scan(-1.0, 0.0);
        const Top2 c1 = combine(st);
        double bound = (tg != 0) ? (c1.i2 >= 0 ? c1.d2 : INFINITY) : -INFINITY;
        bound = wave_max(bound);
        if (bound > 0) stage_scan(0.0, bound);
        const Top2 fin = combine(st);
        if (lane < ntc) {
            uint8_t f = 0;
            int n1 = -1, n2 = -1;
            if (tg != 0) {
                f = 1;
                n1 = fin.i1;
                n2 = fin.i2;
                if (n1 >= 0 && n2 >= 0 && !isnan(crit)) {
                    const double s1 = sgn(g[n1]), s2 = sgn(g[n2]), si = sgn(tg);
                    if ((fin.d1 < crit) || ((s1 == s2) && (s1 != si))) {
                        f |= 2;
                        flag_list[atomicAdd(&ecount[0], 1)] = i;
                    }
                }
            }
            nn1[i] = n1;
            nn2[i] = n2;
            d1o[i] = fin.d1;
            d2o[i] = fin.d2;
            eflag[i] = f;
        }
    }
}

// Squared distance from a point to a node's box (0 inside); never exceeds
// the computed squared distance to any point of the box.
__device__ inline double point_box_dist2(const TreeDev& T, int M, double px, double py) {
    const double dx = fmax(0.0, fmax(double_from_ord(T.blx[M]) - px, px - double_from_ord(T.trx[M])));
    const double dy = fmax(0.0, fmax(double_from_ord(T.bly[M]) - py, py - double_from_ord(T.try_[M])));
    return dx * dx + dy * dy;
}

__device__ inline Top2 wave_top2(Top2 st) {
    for (int o = kWave / 2; o > 0; o >>= 1) top2_merge(st, top2_shfl_xor(st, o));
    return st;
}

// Second-neighbour distance as an ordered integer (NaN counts as DBL_MAX).
__device__ inline uint64_t d2_key(double d2) { return ord_from_double(isnan(d2) ? DBL_MAX : d2); }

// Upper bound of the second-neighbour distance over the searched targets of
// every leaf (-1 for a leaf without one): a merge farther from the leaf's box
// than this changes none of its targets.  And the leaves' boxes in their order
// (lbox: four arrays), which the rounds read and grow.  16 lanes a leaf: a lane alone spent
// 20 us on the leaves of 3k vortices, one load after another.
constexpr int kMaxLanes = 16;
__global__ __launch_bounds__(kBlock) void k_leaf_maxd2(TreeDev T, const int32_t* r0, const int32_t* r1, int base, const double* d2a,
                             const uint8_t* eflag, uint64_t* maxd2, uint64_t* lbox) {
    const int l = blockIdx.x * (kBlock / kMaxLanes) + threadIdx.x / kMaxLanes, sub = threadIdx.x % kMaxLanes;
    if (l >= T.nleaf) return;
    const int L = T.leaf_node[l];
    uint64_t m = ord_from_double(-1.0);
    if (d2a)
        for (int i = r0[L] - base + sub; i < r1[L] - base; i += kMaxLanes)
            if (eflag[i] & 1) m = max(m, d2_key(d2a[i]));
    for (int o = kMaxLanes / 2; o > 0; o >>= 1) m = max(m, (uint64_t)__shfl_xor((unsigned long long)m, o, kMaxLanes));
    if (sub == 0) maxd2[l] = m;
    if (sub < 4) lbox[(size_t)sub * T.nleaf + l] = sub == 0 ? T.blx[L] : sub == 1 ? T.bly[L] : sub == 2 ? T.trx[L] : T.try_[L];
}

// The same bound and box over every kChunk leaves (cbound: least x, least y,
// most x, most y, bound; five arrays).
constexpr int kChunk = kBlock;
__global__ __launch_bounds__(kBlock) void k_chunk_bounds(int nleaf, const uint64_t* maxd2, const uint64_t* lbox,
                                                         uint64_t* cbound) {
    __shared__ uint64_t s_part[kWavesPerBlock][5];
    const int l = min(blockIdx.x * kChunk + (int)threadIdx.x, nleaf - 1), w = threadIdx.x / kWave;
    uint64_t v[5];
    for (int k = 0; k < 5; k++) v[k] = k < 4 ? lbox[(size_t)k * nleaf + l] : maxd2[l];
    for (int o = kWave / 2; o > 0; o >>= 1)
        for (int k = 0; k < 5; k++) {
            const uint64_t u = __shfl_xor((unsigned long long)v[k], o, kWave);
            v[k] = k < 2 ? min(v[k], u) : max(v[k], u);
        }
    if (lane_id() == 0)
        for (int k = 0; k < 5; k++) s_part[w][k] = v[k];
    __syncthreads();
    const int k = threadIdx.x;
    if (k >= 5) return;
    uint64_t r = s_part[0][k];
    for (int q = 1; q < kWavesPerBlock; q++) r = k < 2 ? min(r, s_part[q][k]) : max(r, s_part[q][k]);
    cbound[(size_t)k * gridDim.x + blockIdx.x] = r;
}

// The list being merged (the vortices, or the heat particles) and the state
// of the rounds.  Elements are numbered within the list; r0/r1 minus base are
// a node's range, vleaf[base + i] the leaf of element i.
//   info[i]  {partner, death}: the element that i merges with at its visit
//            (-1: none; -2: none now, but once), and the smallest target that
//            absorbs i (INT_MAX: none).  Target t sees i when death >= t.
//   rec[i]   position and circulation of i after its merge: what targets
//            after i see while info[i].x >= 0
//   fd2[i]   second-neighbour distance of i before its merge
//   cand     a changed element's next record {x, y, g, partner}
struct MergeArgs {
    TreeDev T;
    const double *x, *y, *g;
    const int32_t *r0, *r1;
    int base, n;
    int heat;              // epsh: the distance criterion only
    const double* crit;    // per leaf
    int32_t *nn1, *nn2;
    double *d1, *d2;
    uint8_t* eflag;
    uint64_t *maxd2, *lbox, *cbound;
    int nchunk;
    int2* info;
    double4 *rec, *cand;
    double* fd2;
    int32_t *stamp, *list0, *list1, *chg, *chg_p, *ever;
    double4* cbox;         // per changed element: box of every position its change involves
    int32_t* ctr;          // [0..1] targets to evaluate, [2..3] changed elements, [4] elements with a record
    uint64_t *blx, *bly, *trx, *try_;
    const int32_t *leaf_sim, *root_first;
};

constexpr int kMergeTab = 512;   // candidates staged per wave

// What target i sees of element j (j != i).
struct Seen {
    double x, y, g;
};
__device__ inline Seen seen_of(const MergeArgs& A, int j, int i, int2 f) {
    if (j < i && f.x >= 0) {
        const double4 r = A.rec[j];
        return Seen{r.x, r.y, r.z};
    }
    return Seen{A.x[j], A.y[j], A.g[j]};
}

// The two nearest of target i among what it sees in its near leaves, at
// (px, py), without itself and excl: the leaves touching its own first, then
// those whose box lies within the second-neighbour distance found.  G waves
// (1, or all of the block) share the list; all lanes get the result.
// Latency-bound: the entries of 256 list places, their boxes and ranges load
// together, and the candidates of all of them are listed in LDS, so that a
// search is about four dependent loads.
template <int G>
__device__ Top2 seen_top2(const MergeArgs& A, int l, int L, int i, int excl, double px, double py, int* tab,
                          Top2* parts) {
    const TreeDev& T = A.T;
    const int lane = lane_id();
    const int64_t e0 = T.near_off[l], e1 = T.near_off[l + 1];
    constexpr int kPer = 4;
    auto scan = [&](bool touching, double bound) {
        Top2 st = top2_empty();
        const int w = G == 1 ? 0 : threadIdx.x / kWave;
        // waves take places of the list in turn, or share the candidates of the
        // only ones (a wide leaf's neighbours may be few and wide)
        const bool share = G > 1 && e1 - e0 <= kPer * kWave;
        const int q0 = share ? w * kWave : 0, qstep = share ? G * kWave : kWave;
        for (int64_t eb = share ? e0 : e0 + (int64_t)w * kPer * kWave; eb < e1; eb += (int64_t)G * kPer * kWave) {
            int M[kPer], j0[kPer], cnt[kPer], mine = 0;
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const int64_t e = eb + k * kWave + lane;
                M[k] = e < e1 ? T.near_list[e] : -1;
            }
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const int m = M[k] >= 0 ? M[k] : L;
                const double bd = box_dist2(T, L, m);
                const bool take = M[k] >= 0 && (touching ? bd <= 0.0 : bd > 0.0 && point_box_dist2(T, m, px, py) <= bound);
                j0[k] = A.r0[m] - A.base;
                cnt[k] = take ? A.r1[m] - A.base - j0[k] : 0;
                mine += cnt[k];
            }
            const int incl = wave_incl_scan(mine);
            const int total = __shfl(incl, kWave - 1, kWave);
            for (int done = 0; done < total; done += kMergeTab) {
                int o = incl - mine - done;
#pragma unroll
                for (int k = 0; k < kPer; k++) {
                    if (cnt[k] <= kWide)
                        for (int t = max(0, -o); t < cnt[k] && o + t < kMergeTab; t++) tab[o + t] = j0[k] + t;
                    for (uint64_t wide = __ballot(cnt[k] > kWide); wide; wide &= wide - 1)
                        wave_write_range(j0[k], cnt[k], o, (int)__builtin_ctzll(wide), tab, kMergeTab);
                    o += cnt[k];
                }
                wave_sync();
                const int m = min(kMergeTab, total - done);
                for (int q = q0 + lane; q < m; q += qstep) {
                    const int j = tab[q];
                    if (j == i || j == excl) continue;
                    const int2 f = A.info[j];
                    if (f.y < i) continue;
                    const Seen v = seen_of(A, j, i, f);
                    if (v.g != 0) top2_insert(st, dist2(px, py, v.x, v.y), j);
                }
                wave_sync();
            }
        }
        st = wave_top2(st);
        if (G > 1) {
            __syncthreads();   // parts of the search before are read
            if (lane == 0) parts[w] = st;
            __syncthreads();
            st = parts[0];
            for (int q = 1; q < G; q++) top2_merge(st, parts[q]);
        }
        return st;
    };
    Top2 c = scan(true, 0.0);
    top2_merge(c, scan(false, c.i2 >= 0 ? c.d2 : INFINITY));
    return c;
}

// Elements start without a merge.
__global__ void k_merge_init(MergeArgs A) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.n) return;
    A.info[i] = make_int2(-1, INT32_MAX);
    A.stamp[i] = 0;
    A.ever[i] = -1;
    if (A.heat) {   // no parallel pass before the rounds: every particle is a target of the first
        A.list0[i] = i;
        A.d2[i] = -1.;
    }
}

// Entries that a block collects for a list in global memory: one claim of the
// list's counter a block (12 ns each, 8000 and more of them a round where every
// wave claimed its own).  Entries past the room go to the list at once.
struct BlockList {
    static constexpr int kRoom = 512;
    int n, base;
    int32_t at[kRoom];
    __device__ void begin() {   // all threads
        if (threadIdx.x == 0) n = 0;
        __syncthreads();
    }
    __device__ void push(int32_t v, int32_t* list, int32_t* count) {
        const int k = atomicAdd(&n, 1);
        if (k < kRoom)
            at[k] = v;
        else
            list[atomicAdd(count, 1)] = v;
    }
    __device__ void end(int32_t* list, int32_t* count) {   // all threads
        __syncthreads();
        const int m = min(n, kRoom);
        if (m == 0) return;
        if (threadIdx.x == 0) base = atomicAdd(count, m);
        __syncthreads();
        for (int k = threadIdx.x; k < m; k += blockDim.x) list[base + k] = at[k];
    }
};

// Raises *a to key: by an atomic, or where the block's one writer is the only
// one that touches it by a store, which the block's later loads see.
template <bool kAlone>
__device__ inline void raise_key(uint64_t* a, uint64_t key) {
    if (kAlone) {
        if (key > *a) *a = key;
    } else {
        atomicMax((unsigned long long*)a, (unsigned long long)key);
    }
}

// Target i is visited as the reference does when the merges of the targets
// before it are those assumed now.  Its search results are written in place
// (only the marking pass reads them), its merge to cand; true where that is
// not the assumed one (the same on all lanes).  G waves share the search.
template <int G, bool kAlone>
__device__ bool merge_visit(const MergeArgs& A, int i, int* tab, Top2* parts) {
    const TreeDev& T = A.T;
    const double gi = A.g[i];
    const int2 own = A.info[i];
    const int l = T.vleaf[A.base + i], L = T.leaf_node[l];
    Top2 st = top2_empty();
    int partner = -1;
    double4 rec = make_double4(0, 0, 0, 0);
    const bool alive = gi != 0 && own.y >= i;
    double first_d2 = -1.;
    if (alive) {
        double px = A.x[i], py = A.y[i];
        st = seen_top2<G>(A, l, L, i, -1, px, py, tab, parts);
        first_d2 = st.d2;
        const double crit = A.crit[l];
        if (st.i1 >= 0 && st.i2 >= 0 && !isnan(crit)) {
            const Seen a = seen_of(A, st.i1, i, A.info[st.i1]), b = seen_of(A, st.i2, i, A.info[st.i2]);
            const double s1 = sgn(a.g), s2 = sgn(b.g), si = sgn(gi);
            if ((st.d1 < crit) || (!A.heat && (s1 == s2) && (s1 != si))) {
                // MergeVortexes (:111-126), then the search without merging
                partner = st.i1;
                if (si == s1) {
                    const double inv = 1. / (gi + a.g);
                    const double nx = (px * gi + a.x * a.g) * inv;
                    const double ny = (py * gi + a.y * a.g) * inv;
                    px = nx;
                    py = ny;
                } else if (fabs(gi) < fabs(a.g)) {
                    px = a.x;
                    py = a.y;
                }
                rec = make_double4(px, py, gi + a.g, 0);
                st = seen_top2<G>(A, l, L, i, partner, px, py, tab, parts);
            }
        }
    }
    bool changed = partner != max(own.x, -1);
    if (!changed && partner >= 0) {
        const double4 o = A.rec[i];
        changed = __double_as_longlong(o.x) != __double_as_longlong(rec.x) ||
                  __double_as_longlong(o.y) != __double_as_longlong(rec.y) ||
                  __double_as_longlong(o.z) != __double_as_longlong(rec.z);
    }
    if (lane_id() == 0 && (G == 1 || threadIdx.x / kWave == 0)) {
        A.nn1[i] = st.i1;
        A.nn2[i] = st.i2;
        A.d1[i] = st.d1;
        A.d2[i] = alive ? st.d2 : -1.;
        A.fd2[i] = first_d2;
        A.eflag[i] = alive ? 1 : 0;
        if (alive) {
            const uint64_t key = max(d2_key(st.d2), d2_key(first_d2));
            raise_key<kAlone>(&A.maxd2[l], key);
            // (leaves of several simulations share a chunk)
            raise_key<false>(&A.cbound[4 * (size_t)A.nchunk + l / kChunk], key);
        }
        if (changed) {
            rec.w = (double)partner;
            A.cand[i] = rec;
        }
    }
    return changed;
}

// One round, first part: every listed target is visited, those whose merge
// differs go to the list of changes.  A wave takes a target, or while
// there are no more targets than blocks a whole block: the near list of a wide
// leaf at a cluster's rim runs to thousands of leaves (4M vortices: 310 us a
// round with a wave each, 64 with a block).
constexpr int kEvalThreads = 512, kEvalWaves = kEvalThreads / kWave, kEvalBlocks = 512;
template <int G>
__device__ void merge_eval(const MergeArgs& A, int parity, int nd, int (*s_tab)[kMergeTab], Top2* parts,
                           BlockList& changes) {
    const int w = threadIdx.x / kWave;
    const int32_t* list = parity ? A.list1 : A.list0;
    const int k0 = G == 1 ? blockIdx.x * kEvalWaves + w : blockIdx.x;
    for (int k = k0; k < nd; k += G == 1 ? gridDim.x * kEvalWaves : gridDim.x) {
        const int i = list[k];
        if (merge_visit<G, false>(A, i, s_tab[w], parts) && lane_id() == 0 && (G == 1 || w == 0))
            changes.push(i, A.chg, &A.ctr[2 + parity]);
    }
}

__global__ __launch_bounds__(kEvalThreads) void k_merge_eval(MergeArgs A, int parity) {
    __shared__ int s_tab[kEvalWaves][kMergeTab];
    __shared__ Top2 s_parts[kEvalWaves];
    __shared__ BlockList s_changes;
    const int nd = A.ctr[parity];
    s_changes.begin();
    if (nd <= (int)gridDim.x)
        merge_eval<kEvalWaves>(A, parity, nd, s_tab, s_parts, s_changes);
    else
        merge_eval<1>(A, parity, nd, s_tab, s_parts, s_changes);
    s_changes.end(A.chg, &A.ctr[2 + parity]);
}

// Second part: the changed records take effect, the deaths follow from all
// records, and every change gets the box of the positions it involves (the
// element's own before and after, and its old and new partner's).  Node boxes
// grow by the new positions, so that box distances stay lower bounds.  Three
// phases, each over all changes before the next; thread tid of stride.
__device__ inline void grow_box(double4& b, double px, double py) {
    b.x = fmin(b.x, px);
    b.y = fmin(b.y, py);
    b.z = fmax(b.z, px);
    b.w = fmax(b.w, py);
}

// The leaf of element q holds (px, py) too: its boxes grow (mostly inside
// already: the leaf's copy tells for the node, too).
template <bool kAlone>
__device__ inline void grow_leaf(const MergeArgs& A, int q, double px, double py) {
    const int lq = A.T.vleaf[A.base + q], Lq = A.T.leaf_node[lq], nl = A.T.nleaf;
    const size_t ck = lq / kChunk, nk = A.nchunk;
    auto least = [](uint64_t* a, uint64_t key, bool alone) {
        if (key >= *a) return false;
        if (alone)
            *a = key;
        else
            atomicMin((unsigned long long*)a, (unsigned long long)key);
        return true;
    };
    auto most = [](uint64_t* a, uint64_t key, bool alone) {
        if (key <= *a) return false;
        if (alone)
            *a = key;
        else
            atomicMax((unsigned long long*)a, (unsigned long long)key);
        return true;
    };
    for (int k = 0; k < 2; k++) {
        const double v = k == 0 ? px : py;
        if (isnan(v)) continue;
        const uint64_t key = ord_from_double(v);
        if (least(&A.lbox[k * (size_t)nl + lq], key, kAlone)) {
            least(k == 0 ? &A.blx[Lq] : &A.bly[Lq], key, kAlone);
            atomicMin((unsigned long long*)&A.cbound[k * nk + ck], (unsigned long long)key);
        }
        if (most(&A.lbox[(2 + k) * (size_t)nl + lq], key, kAlone)) {
            most(k == 0 ? &A.trx[Lq] : &A.try_[Lq], key, kAlone);
            atomicMax((unsigned long long*)&A.cbound[(2 + k) * nk + ck], (unsigned long long)key);
        }
    }
}

template <int kPhase>
__device__ void merge_apply(const MergeArgs& A, int parity, int tid, int stride) {
    const int nc = A.ctr[2 + parity];
    if (kPhase == 0) {
        for (int e = tid; e < nc; e += stride) {
            const int q = A.chg[e], p = A.info[q].x;
            double4 b = make_double4(A.x[q], A.y[q], A.x[q], A.y[q]);
            A.chg_p[e] = p;
            if (p >= 0) {
                const double4 r = A.rec[q];
                grow_box(b, r.x, r.y);
                grow_box(b, A.x[p], A.y[p]);
                A.info[p].y = INT32_MAX;
            }
            A.cbox[e] = b;
        }
    } else if (kPhase == 1) {
        for (int e = tid; e < nc; e += stride) {
            const int q = A.chg[e];
            const double4 r = A.cand[q];
            const int p = (int)r.w;
            if (A.info[q].x == -1) A.ever[atomicAdd(&A.ctr[4], 1)] = q;
            A.info[q].x = p >= 0 ? p : -2;
            A.rec[q] = r;
            if (p >= 0) {
                double4 b = A.cbox[e];
                grow_box(b, r.x, r.y);
                grow_box(b, A.x[p], A.y[p]);
                A.cbox[e] = b;
                grow_leaf<false>(A, q, r.x, r.y);
            }
        }
    } else {
        const int ne = A.ctr[4];
        for (int k = tid; k < ne; k += stride) {
            const int q = A.ever[k], p = A.info[q].x;
            if (p >= 0) atomicMin(&A.info[p].y, q);
        }
        // a partner that has merged itself is seen at its merged position too
        for (int e = tid; e < nc; e += stride) {
            const int q = A.chg[e];
            double4 b = A.cbox[e];
            for (int which = 0; which < 2; which++) {
                const int p = which ? A.chg_p[e] : A.info[q].x;
                if (p < 0 || A.info[p].x < 0) continue;
                const double4 r = A.rec[p];
                grow_box(b, r.x, r.y);
            }
            A.cbox[e] = b;
        }
        if (tid == 0) {
            A.ctr[parity] = 0;
            A.ctr[2 + (parity ^ 1)] = 0;
        }
    }
}

// All phases in one workgroup: 12 us for up to a few hundred changes.
constexpr int kMergeThreads = 1024;
__global__ __launch_bounds__(kMergeThreads) void k_merge_apply(MergeArgs A, int parity) {
    merge_apply<0>(A, parity, threadIdx.x, kMergeThreads);
    __threadfence();
    __syncthreads();
    merge_apply<1>(A, parity, threadIdx.x, kMergeThreads);
    __threadfence();
    __syncthreads();
    merge_apply<2>(A, parity, threadIdx.x, kMergeThreads);
}

// A phase a launch, over the chip.
template <int kPhase>
__global__ __launch_bounds__(kBlock) void k_merge_apply_part(MergeArgs A, int parity) {
    merge_apply<kPhase>(A, parity, blockIdx.x * kBlock + threadIdx.x, gridDim.x * kBlock);
}

// Does a change in the box b reach target i: before its own merge or after?
__device__ inline bool change_reaches(const MergeArgs& A, const double4& b, int i) {
    auto reach = [&](double px, double py, double d2) {
        const double dx = fmax(0.0, fmax(b.x - px, px - b.z)), dy = fmax(0.0, fmax(b.y - py, py - b.w));
        return !(dx * dx + dy * dy > d2);
    };
    if (!(A.eflag[i] & 1)) return false;
    if (A.info[i].x < 0) return reach(A.x[i], A.y[i], A.d2[i]);
    const double4 r = A.rec[i];
    return reach(A.x[i], A.y[i], A.fd2[i]) || reach(r.x, r.y, A.d2[i]);
}

// The targets after a changed element q whose second-neighbour distance
// reaches the change's box b have to be visited again (those it does not reach
// cannot take or lose a neighbour by it), and so have its old and new partner
// p0 and p1, which it kills or revives: push(target) for each, by any thread.
// A block per change: each wave tests the chunks of leaves from the element's
// on (leaves before it hold no later target), a lane each; the block's first
// threads the leaves of a chunk that may be reached; and their targets a lane
// each.  tab: the wave's.
// Testing every leaf for every change took 120 us a round in the batch of 16
// cylinders, 14 us behind one in 100k vortices; now 18 and 8.5.
// kRaised: other blocks raise the chunks' bounds meanwhile, by atomics.  Ranges
// of more than kWide targets go to wide(j0, cnt), which says whether it takes them.
template <bool kRaised, typename Push, typename Wide>
__device__ inline void mark_change(const MergeArgs& A, int q, const double4& b, int p0, int p1, int* tab, Push push,
                                   Wide wide) {
    const TreeDev& T = A.T;
    const int lane = lane_id();
    auto far = [&](uint64_t blx, uint64_t bly, uint64_t trx, uint64_t try_, double m) {
        const double dx = fmax(0.0, fmax(b.x - double_from_ord(trx), double_from_ord(blx) - b.z));
        const double dy = fmax(0.0, fmax(b.y - double_from_ord(try_), double_from_ord(bly) - b.w));
        return dx * dx + dy * dy > m;
    };
    const int lq = T.vleaf[A.base + q];
    const int lend = A.root_first[A.leaf_sim[lq] + 1];
    if (threadIdx.x == 0) {
        if (p0 > q) push(p0);
        if (p1 > q) push(p1);
    }
    auto leaves = [&](int l) {
        const double m = l >= lq && l < lend ? double_from_ord(A.maxd2[l]) : -1.0;
        int j0 = 0, cnt = 0;
        if (!(m < 0)) {
            const uint64_t* lb = A.lbox + l;
            const size_t nl = T.nleaf;
            if (!far(lb[0], lb[nl], lb[2 * nl], lb[3 * nl], m)) {
                const int L = T.leaf_node[l];
                j0 = max(A.r0[L] - A.base, q + 1);
                cnt = max(0, A.r1[L] - A.base - j0);
                if (cnt > kWide && wide(j0, cnt)) cnt = 0;
            }
        }
        wave_lay_out(j0, cnt, tab, [&](int n) {
            for (int k = lane; k < n; k += kWave)
                if (change_reaches(A, b, tab[k])) push(tab[k]);
        });
    };
    const int ck1 = (lend - 1) / kChunk;
    for (int c0 = lq / kChunk; c0 <= ck1; c0 += kWave) {
        bool may = false;
        if (c0 + lane <= ck1) {
            uint64_t cb[5];
            for (int k = 0; k < 5; k++) {
                const uint64_t* p = A.cbound + k * (size_t)A.nchunk + c0 + lane;
                cb[k] = kRaised ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
            }
            const double m = double_from_ord(cb[4]);
            may = !(m < 0) && !far(cb[0], cb[1], cb[2], cb[3], m);
        }
        for (uint64_t mask = __ballot(may); mask; mask &= mask - 1)
            if (threadIdx.x < kChunk) leaves((c0 + (int)__builtin_ctzll(mask)) * kChunk + threadIdx.x);
    }
}

// Third part of a round: what the changes reach is listed for the next one.
__global__ __launch_bounds__(kBlock) void k_merge_mark(MergeArgs A, int parity, int tag) {
    __shared__ int s_tab[kWavesPerBlock][kNearTab];
    __shared__ BlockList s_next;
    const int nc = A.ctr[2 + parity];
    int32_t* list = parity ? A.list0 : A.list1;
    s_next.begin();
    for (int e = blockIdx.x; e < nc; e += gridDim.x) {
        const int q = A.chg[e];
        mark_change<false>(A, q, A.cbox[e], A.chg_p[e], A.info[q].x, s_tab[threadIdx.x / kWave], [&](int i) {
            if (atomicExch(&A.stamp[i], tag) != tag) s_next.push(i, list, &A.ctr[parity ^ 1]);
        }, [](int, int) { return false; });
    }
    s_next.end(list, &A.ctr[parity ^ 1]);
}

// The targets still to be visited (stamp == tag) one after another in their
// order, a block per simulation: every target is visited once, when all before
// it are settled.  For chains of merges that wait for each other one by one,
// where each round settles a single one and visits all behind it in vain.
// next: the block's first element to look at; a launch visits kInOrder targets
// of a simulation at most, *left then counts the simulations that have more.
// What is written here is read by the same block only (stores, and barriers
// that wait for them), but for the chunk bounds and the list of elements that
// have a record, of which an entry of another simulation does nothing.
constexpr int kInOrder = 2048;
__global__ __launch_bounds__(kEvalThreads) void k_merge_in_order(MergeArgs A, int tag, int32_t* next, int32_t* left) {
    __shared__ int s_tab[kEvalWaves][kNearTab];
    __shared__ Top2 s_parts[kEvalWaves];
    __shared__ int s_first[kEvalWaves], s_death[2], s_nwide;
    __shared__ int2 s_wide[kChunk];   // ranges of targets that all threads share
    __shared__ double4 s_box;
    static_assert(kNearTab >= kMergeTab && kEvalThreads >= kChunk, "tables of the searches and leaves of a chunk");
    const int sim = blockIdx.x, t = threadIdx.x, w = t / kWave, lane = lane_id();
    const int end = A.r1[sim] - A.base;
    auto sync = [] {
        __threadfence_block();
        __syncthreads();
    };
    int cur = next[sim];
    for (int visits = 0; cur < end && visits < kInOrder;) {
        // the first one listed from cur on
        constexpr int kPer = 4;
        int first = INT32_MAX;
        for (int k = kPer - 1; k >= 0; k--) {
            const int i = cur + k * kEvalThreads + t;
            const uint64_t m = __ballot(i < end && A.stamp[i] == tag);
            if (m) first = i - lane + (int)__builtin_ctzll(m);
        }
        if (lane == 0) s_first[w] = first;
        __syncthreads();
        for (int q = 0; q < kEvalWaves; q++) first = min(first, s_first[q]);
        if (first == INT32_MAX) {
            cur += kPer * kEvalThreads;
            __syncthreads();
            continue;
        }
        const int i = first;
        visits++;
        cur = i + 1;
        const int p0 = A.info[i].x;
        const bool changed = merge_visit<kEvalWaves, true>(A, i, s_tab[w], s_parts);
        sync();
        if (!changed) continue;
        // the record takes effect (see merge_apply)
        const double4 r = A.cand[i];
        const int p1 = (int)r.w;
        if (t == 0) {
            double4 b = make_double4(A.x[i], A.y[i], A.x[i], A.y[i]);
            if (p0 >= 0) {
                const double4 o = A.rec[i];
                grow_box(b, o.x, o.y);
                grow_box(b, A.x[p0], A.y[p0]);
            }
            if (p0 == -1) A.ever[atomicAdd(&A.ctr[4], 1)] = i;
            A.info[i].x = p1 >= 0 ? p1 : -2;
            A.rec[i] = r;
            if (p1 >= 0) {
                grow_box(b, r.x, r.y);
                grow_box(b, A.x[p1], A.y[p1]);
                grow_leaf<true>(A, i, r.x, r.y);
            }
            for (int p : {p0, p1})
                if (p >= 0 && A.info[p].x >= 0) {
                    const double4 o = A.rec[p];
                    grow_box(b, o.x, o.y);
                }
            s_box = b;
            s_death[0] = s_death[1] = INT32_MAX;
            s_nwide = 0;
        }
        sync();
        // deaths of the old and the new partner
        const int ne = __hip_atomic_load(&A.ctr[4], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int k = t; k < ne; k += kEvalThreads) {
            const int q = A.ever[k], p = q >= 0 ? A.info[q].x : -1;
            if (p < 0) continue;
            if (p == p0) atomicMin(&s_death[0], q);
            if (p == p1) atomicMin(&s_death[1], q);
        }
        __syncthreads();
        if (t == 0) {
            if (p0 >= 0) A.info[p0].y = s_death[0];
            if (p1 >= 0) A.info[p1].y = s_death[1];
        }
        auto push = [&](int k) { A.stamp[k] = tag; };
        mark_change<true>(A, i, s_box, p0, p1, s_tab[w], push, [&](int j0, int cnt) {
            const int k = atomicAdd(&s_nwide, 1);
            if (k < kChunk) s_wide[k] = make_int2(j0, cnt);
            return k < kChunk;
        });
        __syncthreads();
        for (int r = 0; r < min(s_nwide, kChunk); r++)
            for (int k = t; k < s_wide[r].y; k += kEvalThreads)
                if (change_reaches(A, s_box, s_wide[r].x + k)) push(s_wide[r].x + k);
        sync();
    }
    if (t == 0) {
        next[sim] = cur;
        if (cur < end) atomicAdd(left, 1);
    }
}

// The first element of every simulation.
__global__ void k_merge_first(MergeArgs A, int nsim, int32_t* next) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nsim) next[s] = A.r0[s] - A.base;
}

// The converged merges written to the list, one workgroup: every merging
// element takes its record, then every partner loses its circulation.
__global__ __launch_bounds__(kMergeThreads) void k_merge_finish(MergeArgs A, double* x, double* y, double* g,
                                                                int32_t* merged) {
    __shared__ int s_n;
    const int ne = A.ctr[4], tid = threadIdx.x;
    if (tid == 0) s_n = 0;
    __syncthreads();
    int cnt = 0;
    for (int k = tid; k < ne; k += kMergeThreads) {
        const int q = A.ever[k];
        if (A.info[q].x < 0) continue;
        const double4 r = A.rec[q];
        x[q] = r.x;
        y[q] = r.y;
        g[q] = r.z;
        cnt++;
    }
    atomicAdd(&s_n, cnt);
    __threadfence();
    __syncthreads();
    for (int k = tid; k < ne; k += kMergeThreads) {
        const int p = A.info[A.ever[k]].x;
        if (p >= 0) g[p] = 0;
    }
    if (tid == 0) *merged = s_n;
}

// Applies _1_eps = 1/max(eps, floor) to every processed target (:49-54) and
// packs the FP32 {g, eps^2} copy the pair kernels read.
__global__ void k_eps_apply(const TreeDev T, const double* g, double* ie, int64_t n, const int32_t* nn1,
                            const int32_t* nn2, const double* d1a, const double* d2a, const uint8_t* eflag,
                            const double* leaf_restr, float2* src_ge) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double iv = ie[i];
    if (eflag[i] & 1) {
        double eps;
        if (nn1[i] < 0)
            eps = DBL_MIN;
        else if (nn2[i] < 0)
            eps = sqrt(d1a[i]);
        else
            eps = sqrt(d2a[i]);
        const double r = leaf_restr[T.vleaf[i]];
        iv = 1.0 / ((eps < r) ? r : eps);
        ie[i] = iv;
    }
    const double gi = g[i];
    if (gi != 0) {
        const double e = 1. / iv;
        src_ge[i] = make_float2((float)gi, (float)(e * e));
    } else {
        src_ge[i] = make_float2(0.f, 1.f);
    }
}

__global__ void k_pack(const double* g, const double* ie, int64_t n, float2* src_ge) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double gi = g[i];
    if (gi != 0) {
        const double e = 1. / ie[i];
        src_ge[i] = make_float2((float)gi, (float)(e * e));
    } else {
        src_ge[i] = make_float2(0.f, 1.f);
    }
}

}  // namespace

void pack_sources(Ctx& c) {
    if (c.n)
        hipLaunchKernelGGL(k_pack, dim3(nblocks(c.n)), dim3(kBlock), 0, c.stream, c.g.p, c.ie.p, c.n, c.src_ge.p);
}

namespace {

// Finds the sequential merges of the list in A (see MergeArgs) and writes
// them to x, y, g; the number goes to *merged on the device.  The first
// round's targets are in list0, their count in ctr[0].  Rounds are queued a
// few at a time and end when one leaves nothing to visit: at most one per
// element, in practice the longest chain of merges that wait for each other
// (three to about ten).  One workgroup committing merge after merge took
// about 45 us each (5.8 ms a step for a cylinder wake of 3k vortices); a
// round of all of them takes about 25 us.
// left: the targets listed for the first round.
constexpr int kApplyOne = 2048;
// A round takes about 25 us and 1/16 us a target, a visit in order 10 to 18.
// Rounds are given up for the order when they have taken about a third of what
// the targets left would take in it; most lists have settled long before.  A
// line of 2000 merges: 350 ms in rounds alone, 38 so (121 where one workgroup
// committed merge after merge); 300 round a body 14.2, 3.5 (6.1).
constexpr int64_t kInOrderShare = 3, kInOrderAfter = 16;
void merge_rounds(Ctx& c, MergeArgs A, int32_t left, double* x, double* y, double* g, int32_t* merged) {
    hipStream_t s = c.stream;
    hipLaunchKernelGGL(k_chunk_bounds, dim3(A.nchunk), dim3(kBlock), 0, s, A.T.nleaf, (const uint64_t*)A.maxd2,
                       (const uint64_t*)A.lbox, A.cbound);
    int64_t spent = 0;
    for (int64_t round = 0; left > 0; ) {
        VVHD_CHECK(round <= (int64_t)A.n + 8, VVHD_EHIP, "epsilon: the merges do not settle");
        for (int k = 0; k < 4; k++, round++) {
            const int par = (int)(round & 1);
            hipLaunchKernelGGL(k_merge_eval, dim3(kEvalBlocks), dim3(kEvalThreads), 0, s, A, par);
            if (left <= kApplyOne) {
                hipLaunchKernelGGL(k_merge_apply, dim3(1), dim3(kMergeThreads), 0, s, A, par);
            } else {
                hipLaunchKernelGGL(k_merge_apply_part<0>, dim3(256), dim3(kBlock), 0, s, A, par);
                hipLaunchKernelGGL(k_merge_apply_part<1>, dim3(256), dim3(kBlock), 0, s, A, par);
                hipLaunchKernelGGL(k_merge_apply_part<2>, dim3(256), dim3(kBlock), 0, s, A, par);
            }
            hipLaunchKernelGGL(k_merge_mark, dim3(1024), dim3(kBlock), 0, s, A, par, (int)round + 1);
        }
        VVHD_HIP(hipMemcpyAsync(&left, A.ctr + (round & 1), 4, hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipStreamSynchronize(s));
        spent += 4 * (25 + (int64_t)left / 16);
        if (round < kInOrderAfter || spent < kInOrderShare * (int64_t)left) continue;
        // the rounds do not pay: the rest in order
        c.mg.next.grow(c.nsim + 1);
        int32_t* more = c.mg.next.p + c.nsim;
        hipLaunchKernelGGL(k_merge_first, dim3(nblocks(c.nsim)), dim3(kBlock), 0, s, A, c.nsim, c.mg.next.p);
        while (left > 0) {
            VVHD_HIP(hipMemsetAsync(more, 0, 4, s));
            hipLaunchKernelGGL(k_merge_in_order, dim3(c.nsim), dim3(kEvalThreads), 0, s, A, (int)round, c.mg.next.p,
                               more);
            VVHD_HIP(hipMemcpyAsync(&left, more, 4, hipMemcpyDeviceToHost, s));
            VVHD_HIP(hipStreamSynchronize(s));
        }
    }
    hipLaunchKernelGGL(k_merge_finish, dim3(1), dim3(kMergeThreads), 0, s, A, x, y, g, merged);
}

// Buffers of the rounds for a list of n elements.
MergeArgs merge_args(Ctx& c, const double* x, const double* y, const double* g, const int32_t* r0, const int32_t* r1,
                     int base, int64_t n, int heat, int32_t* nn1, int32_t* nn2, double* d1, double* d2,
                     uint8_t* eflag, int32_t* list0) {
    MergeBufs& b = c.mg;
    b.info.grow(n);
    b.rec.grow(n);
    b.cand.grow(n);
    b.cbox.grow(n);
    b.fd2.grow(n);
    for (auto* p : {&b.stamp, &b.list, &b.chg, &b.chg_p, &b.ever}) p->grow(n);
    b.maxd2.grow(c.t.nleaves_h + 1);
    b.lbox.grow(4 * (size_t)c.t.nleaves_h + 1);
    const int nchunk = nblocks(c.t.nleaves_h, kChunk);
    b.cbound.grow(5 * (size_t)nchunk);
    TreeArrays& t = c.t;
    return MergeArgs{tree_dev(t), x, y, g, r0, r1, base, (int)n, heat, c.leaf_crit.p, nn1, nn2, d1, d2, eflag,
                     b.maxd2.p, b.lbox.p, b.cbound.p, nchunk, b.info.p, b.rec.p, b.cand.p, b.fd2.p, b.stamp.p, list0, b.list.p, b.chg.p, b.chg_p.p,
                     b.ever.p, b.cbox.p, c.ecount.p, t.blx.p, t.bly.p, t.trx.p, t.try_.p, t.leaf_sim.p,
                     t.root_first.p};
}

}  // namespace

// ecount: [0..4] the rounds' counters ([0] pass 1's flags), [5] merges.
void epsilon(Ctx& c, int merge, int32_t* nn1_out, int32_t* nn2_out, int32_t* merged_out) {
    const int64_t n = c.n;
    const TreeDev T = tree_dev(c.t);
    const int nl = T.nleaf;
    hipStream_t s = c.stream;
    c.nn1.grow(n + 1);
    c.nn2.grow(n + 1);
    c.d1.grow(n + 1);
    c.d2.grow(n + 1);
    c.eflag.grow(n + 1);
    c.flag_list.grow(n + 1);
    c.ecount.grow(8);
    c.leaf_crit.grow(nl + 1);
    c.leaf_restr.grow(nl + 1);
    VVHD_HIP(hipMemsetAsync(c.ecount.p, 0, 8 * 4, s));
    hipLaunchKernelGGL(k_leaf_criteria, dim3(nblocks(nl, kWavesPerBlock)), dim3(kBlock), 0, s, T, c.segs.p, c.body_range.p,
                       (const int32_t*)c.sim_body.p, (const int32_t*)c.t.leaf_sim.p,
                       merge, c.leaf_crit.p, c.leaf_restr.p);
    if (nl > 0)
        hipLaunchKernelGGL(k_eps_top2, dim3(nl, leaf_parts(nl)), dim3(kWave), 0, s, T, c.x.p,
                           c.y.p, c.g.p, merge, c.leaf_crit.p, c.nn1.p, c.nn2.p, c.d1.p, c.d2.p, c.eflag.p,
                           c.ecount.p, c.flag_list.p);
    int32_t flags = 0, merged = 0;
    VVHD_HIP(hipMemcpyAsync(&flags, c.ecount.p, 4, hipMemcpyDeviceToHost, s));
    VVHD_HIP(hipStreamSynchronize(s));
    if (flags > 0) {
        const MergeArgs A = merge_args(c, c.x.p, c.y.p, c.g.p, T.v0, T.v1, 0, n, 0, c.nn1.p, c.nn2.p, c.d1.p, c.d2.p,
                                       c.eflag.p, c.flag_list.p);
        hipLaunchKernelGGL(k_merge_init, dim3(nblocks(n)), dim3(kBlock), 0, s, A);
        hipLaunchKernelGGL(k_leaf_maxd2, dim3(nblocks(nl, kBlock / kMaxLanes)), dim3(kBlock), 0, s, T, A.r0, A.r1, 0,
                           (const double*)c.d2.p, (const uint8_t*)c.eflag.p, A.maxd2, A.lbox);
        merge_rounds(c, A, flags, c.x.p, c.y.p, c.g.p, c.ecount.p + 5);
    }
    hipLaunchKernelGGL(k_eps_apply, dim3(nblocks(n)), dim3(kBlock), 0, s, T, c.g.p, c.ie.p, n, c.nn1.p, c.nn2.p,
                       c.d1.p, c.d2.p, c.eflag.p, c.leaf_restr.p, c.src_ge.p);
    if (flags > 0) {
        VVHD_HIP(hipMemcpyAsync(&merged, c.ecount.p + 5, 4, hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipStreamSynchronize(s));
    }
    if (nn1_out && n) VVHD_HIP(hipMemcpyAsync(nn1_out, c.nn1.p, (size_t)n * 4, hipMemcpyDeviceToHost, s));
    if (nn2_out && n) VVHD_HIP(hipMemcpyAsync(nn2_out, c.nn2.p, (size_t)n * 4, hipMemcpyDeviceToHost, s));
    if (flags > 0) pack_boxes(c);   // merges grew leaf boxes
    const int heat_merged = heat_epsilon(c, merge);   // epsh on the heat list (MEpsilonFast.cpp:53-60)
    if (merged_out) *merged_out = merged + heat_merged;
}

// _1_eps = 1 / max(eps, floor) of the heat particles (MEpsilonFast.cpp:55-60).
__global__ void k_heat_eps_apply(const int32_t* vleaf, const int32_t* nn1, const int32_t* nn2, const double* d1,
                                 const double* d2, const uint8_t* eflag, const double* restr, double* hie, int64_t nh) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nh || !(eflag[j] & 1)) return;
    const double e = nn1[j] < 0 ? DBL_MIN : (nn2[j] < 0 ? sqrt(d1[j]) : sqrt(d2[j]));
    const double r = restr[vleaf[j]];
    hie[j] = 1.0 / ((e < r) ? r : e);   // std::max(e, r)
}

// epsh (MEpsilonFast.cpp:175-212) on the heat list: the same rounds, every
// particle a target of the first (without merging the criterion is NaN and
// the first round is all there is).
int heat_epsilon(Ctx& c, int merge) {
    const int64_t nh = c.heat.n;
    if (nh == 0) return 0;
    const TreeDev T = tree_dev(c.t);
    hipStream_t s = c.stream;
    MergeBufs& b = c.mg;
    for (auto* p : {&b.hn1, &b.hn2, &b.hlist}) p->grow(nh);
    for (auto* p : {&b.hd1, &b.hd2}) p->grow(nh);
    b.hflag.grow(nh);
    const MergeArgs A = merge_args(c, c.heat.x.p, c.heat.y.p, c.heat.g.p, T.h0, T.h1, T.hbase, nh, 1, b.hn1.p,
                                   b.hn2.p, b.hd1.p, b.hd2.p, b.hflag.p, b.hlist.p);
    const int32_t start[8] = {(int32_t)nh, 0, 0, 0, 0, 0, 0, 0};
    VVHD_HIP(hipMemcpyAsync(c.ecount.p, start, sizeof(start), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_merge_init, dim3(nblocks(nh)), dim3(kBlock), 0, s, A);
    hipLaunchKernelGGL(k_leaf_maxd2, dim3(nblocks(T.nleaf, kBlock / kMaxLanes)), dim3(kBlock), 0, s, T, A.r0, A.r1, A.base,
                       (const double*)nullptr, (const uint8_t*)nullptr, A.maxd2, A.lbox);
    merge_rounds(c, A, (int32_t)nh, c.heat.x.p, c.heat.y.p, c.heat.g.p, c.ecount.p + 5);
    hipLaunchKernelGGL(k_heat_eps_apply, dim3(nblocks(nh)), dim3(kBlock), 0, s, T.vleaf + T.hbase,
                       (const int32_t*)b.hn1.p, (const int32_t*)b.hn2.p, (const double*)b.hd1.p,
                       (const double*)b.hd2.p, (const uint8_t*)b.hflag.p, (const double*)c.leaf_restr.p, c.heat.ie.p,
                       nh);
    int32_t merged = 0;
    if (merge) {
        VVHD_HIP(hipMemcpyAsync(&merged, c.ecount.p + 5, 4, hipMemcpyDeviceToHost, s));
        VVHD_HIP(hipStreamSynchronize(s));
    }
    VVHD_HIP(hipGetLastError());
    return merged;
}

}  // namespace vvhd
