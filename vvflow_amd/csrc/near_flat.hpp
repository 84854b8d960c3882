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
// them at a time in tab[0..m), then chunk(m).  A lane writes its own range; one
// of more than kWide elements is written by all lanes, range after range (a
// leaf that the least node size keeps whole may hold thousands).
constexpr int kWide = 32;

// The part of lane b's range [j0, j0 + cnt) that falls in tab[0..room), its
// first element at tab[o] (before the table where o < 0).
__device__ inline void wave_write_range(int j0, int cnt, int o, int b, int* tab, int room) {
    const int ob = __builtin_amdgcn_readlane(o, b), j = __builtin_amdgcn_readlane(j0, b) - ob;
    const int end = min(ob + __builtin_amdgcn_readlane(cnt, b), room);
    for (int t = max(0, ob) + lane_id(); t < end; t += kWave) tab[t] = j + t;
}

template <typename Chunk>
__device__ inline void wave_lay_out(int j0, int cnt, int* tab, Chunk chunk) {
    const int incl = wave_incl_scan(cnt);
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    const uint64_t wide = __ballot(cnt > kWide);
    for (int done = 0; done < total; done += kNearTab) {
        const int o = incl - cnt - done;
        if (cnt <= kWide)
            for (int t = max(0, -o); t < cnt && o + t < kNearTab; t++) tab[o + t] = j0 + t;
        for (uint64_t w = wide; w; w &= w - 1)
            wave_write_range(j0, cnt, o, (int)__builtin_ctzll(w), tab, kNearTab);
        wave_sync();
        chunk(min(kNearTab, total - done));
        wave_sync();
    }
}

// The same for the ranges that range(list[e], j0, cnt) gives for e in [e0, e1).
// A leaf has about 12 elements: taken leaf by leaf, four of five lanes idle,
// and every leaf waits for its own chain of loads (list, range, element).  Here
// 64 entries are looked up at once, a lane each, and their elements laid out in
// LDS.  Ranges of more than kDirect elements go to direct(j0, j0 + cnt) instead.
template <int kDirect, typename Range, typename Chunk, typename Direct>
__device__ inline void wave_lay_out(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, Chunk chunk,
                                    Direct direct) {
    const int lane = lane_id();
    for (int64_t eb = e0; eb < e1; eb += kWave) {
        int j0 = 0, cnt = 0;
        if (eb + lane < e1) range(list[eb + lane], j0, cnt);
        if (kDirect) {
            for (uint64_t w = __ballot(cnt > kDirect); w; w &= w - 1) {
                const int b = (int)__builtin_ctzll(w), j = __builtin_amdgcn_readlane(j0, b);
                direct(j, j + __builtin_amdgcn_readlane(cnt, b));
            }
            if (cnt > kDirect) cnt = 0;
        }
        wave_lay_out(j0, cnt, tab, chunk);
    }
}

// f(j) for every element, one per lane, where their order does not matter.
// Ranges of thousands of elements fill the lanes by themselves: read through
// the table they took a fifth longer.
template <typename Range, typename F>
__device__ inline void wave_flat(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, F f) {
    wave_lay_out<512>(list, e0, e1, tab, range,
                      [&](int m) {
#pragma unroll 2
                          for (int q = lane_id(); q < m; q += kWave) f(tab[q]);
                      },
                      [&](int j, int end) {
                          for (j += lane_id(); j < end; j += kWave) f(j);
                      });
}

// f(j, on) for 64 elements at a time, in order, on all lanes; on where the
// lane has an element.
template <typename Range, typename F>
__device__ inline void wave_flat_all(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, F f) {
    wave_lay_out<0>(list, e0, e1, tab, range,
                    [&](int m) {
                        for (int q = lane_id(); q - lane_id() < m; q += kWave) f(q < m ? tab[q] : 0, q < m);
                    },
                    [](int, int) {});
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
