// near_flat.hpp -- the elements of a list of leaves as one sequence for a wave.
#pragma once
#include "common.hpp"

namespace vvhd {

// Elements in a wave's table, 4 KiB: 16 leaves of the usual 16 elements fill a
// quarter of it, and blocks of four waves still fill a CU (10 x 16 KiB).
constexpr int kNearTab = 1024;

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The elements [j0, j0 + cnt) of every lane's range, in lane order: some of
// them at a time in tab[0..m), then chunk(m).
template <typename Chunk>
__device__ inline void wave_lay_out(int j0, int cnt, int* tab, Chunk chunk) {
    const int incl = wave_incl_scan(cnt);
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    for (int done = 0; done < total; done += kNearTab) {
        const int o = incl - cnt - done;
        for (int t = max(0, -o); t < cnt && o + t < kNearTab; t++) tab[o + t] = j0 + t;
        wave_sync();
        chunk(min(kNearTab, total - done));
        wave_sync();
    }
}

// The same for the ranges that range(list[e], j0, cnt) gives for e in [e0, e1).
// A leaf has about 12 elements: taken leaf by leaf, four of five lanes idle,
// and every leaf waits for its own chain of loads (list, range, element).  Here
// 64 entries are looked up at once, a lane each, and their elements laid out in
// LDS.
template <typename Range, typename Chunk>
__device__ inline void wave_lay_out(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, Chunk chunk) {
    const int lane = lane_id();
    for (int64_t eb = e0; eb < e1; eb += kWave) {
        int j0 = 0, cnt = 0;
        if (eb + lane < e1) range(list[eb + lane], j0, cnt);
        wave_lay_out(j0, cnt, tab, chunk);
    }
}

// f(j) for every element, one per lane, where their order does not matter.
template <typename Range, typename F>
__device__ inline void wave_flat(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, F f) {
    wave_lay_out(list, e0, e1, tab, range, [&](int m) {
#pragma unroll 2
        for (int q = lane_id(); q < m; q += kWave) f(tab[q]);
    });
}

// f(j, on) for 64 elements at a time, in order, on all lanes; on where the
// lane has an element.
template <typename Range, typename F>
__device__ inline void wave_flat_all(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, F f) {
    wave_lay_out(list, e0, e1, tab, range, [&](int m) {
        for (int q = lane_id(); q - lane_id() < m; q += kWave) f(q < m ? tab[q] : 0, q < m);
    });
}

// acc + buf[0] + buf[1] + ... + buf[n - 1], one after another, from LDS; every
// lane computes it, so that the reads are broadcasts and run ahead of the adds.
__device__ inline double ordered_add(double acc, const double* buf, int n) {
    int q = 0;
    for (; q + 8 <= n; q += 8) {
        double t[8];
#pragma unroll
        for (int u = 0; u < 8; u++) t[u] = buf[q + u];
#pragma unroll
        for (int u = 0; u < 8; u++) acc += t[u];
    }
    for (; q < n; q++) acc += buf[q];
    return acc;
}

}  // namespace vvhd
