// near_flat.hpp -- the elements of a list of leaves as one sequence for a wave.
#pragma once
#include "common.hpp"

namespace vvhd {

// Elements in a wave's table, 4 KiB: 16 leaves of the usual 16 elements fill a
// quarter of it, and blocks of four waves still fill a CU (10 x 16 KiB).
constexpr int kNearTab = 1024;

// Calls f(j) for the elements j of the ranges that range(list[e], j0, count)
// gives for e in [e0, e1), one element per lane.  A leaf has about 12
// elements: taken leaf by leaf, four of five lanes idle, and every leaf waits
// for its own chain of loads (list, range, element).  Here 64 entries are
// looked up at once, a lane each, and their elements laid out in LDS.
template <typename Range, typename F>
__device__ inline void wave_flat(const int32_t* list, int64_t e0, int64_t e1, int* tab, Range range, F f) {
    const int lane = lane_id();
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    for (int64_t eb = e0; eb < e1; eb += kWave) {
        int j0 = 0, cnt = 0;
        if (eb + lane < e1) range(list[eb + lane], j0, cnt);
        const int incl = wave_incl_scan(cnt);
        const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
        for (int done = 0; done < total; done += kNearTab) {
            const int o = incl - cnt - done;
            for (int t = max(0, -o); t < cnt && o + t < kNearTab; t++) tab[o + t] = j0 + t;
            wave_sync();
            const int m = min(kNearTab, total - done);
#pragma unroll 2
            for (int q = lane; q < m; q += kWave) f(tab[q]);
            wave_sync();
        }
    }
}

}  // namespace vvhd
