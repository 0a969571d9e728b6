// Host side of stream.hpp: cuts a schedule into phases and levels.
#pragma once

#include <algorithm>

#include "launch.hpp"

namespace bf {

constexpr int kStreamMaxLogN = 12;

// Fills phases and levels of the schedule's first NS stages for `waves` wavefronts.  saves: nsaves stage numbers in front of which the
// tile is stored, to the plane of the same number.  False when the schedule does not fit the tables
// or the rows the workgroup.
inline bool plan_stream(const Schedule &sc, int NS, int elem, int waves, const int *saves, int nsaves, StreamArgs &a)
{
    const int L = sc.log_n;
    const int nbits = 8 + (waves == 16 ? 4 : waves == 8 ? 3 : 2);
    if (!sc.base4 || L < 2 || L > nbits || NS < 1 || NS > kStreamMaxLevels || nsaves > kStreamMaxSaves) return false;
    auto saved_behind = [&](int t) {
        for (int k = 0; k < nsaves; ++k)
            if (saves[k] == t + 1) return k + 1;
        return 0;
    };
    const int max_lo = std::min(L - 1, nbits - 4);   // (register bits past the row are row bits)
    // end of the run of stages from t on that lie on the register bits lo .. lo + 3
    auto run = [&](int t, int lo) {
        for (; t < NS; ++t) {
            const StageInfo s = stage_info(sc, t);
            if (s.log_stride < lo || s.log_stride + s.radix4 > lo + 3) break;
            if (s.radix4 && ((s.log_stride - lo) & 1)) break;
        }
        return t;
    };
    a.log_n = L;
    a.nlevels = 0;
    int nphases = 0;
    for (int t = 0; t < NS;) {
        int best = 0, end = t;
        for (int lo = 0; lo <= max_lo; ++lo)
            if (run(t, lo) > end) {
                best = lo;
                end = run(t, lo);
            }
        if (end == t || nphases == kStreamMaxPhases) return false;
        StreamPhase &p = a.phase[nphases];
        p.reg = (unsigned)best;
        p.places = 0;
        // Lane bits 2..5: the lowest four index bits that are free and adjacent.  Low ones make the
        // saved planes' stores contiguous; adjacent ones land in different LDS banks.
        bool used[16] = {};
        for (int b = 0; b < 4; ++b) used[best + b] = true;
        int lane = -1;
        for (int b = 0; b + 3 < nbits && lane < 0; ++b)
            if (!used[b] && !used[b + 1] && !used[b + 2] && !used[b + 3]) lane = b;
        for (int k = 0, b = 0; k < nbits - 4; ++k) {
            if (k < 4 && lane >= 0) b = lane + k;
            else for (b = 0; used[b];) ++b;
            p.places |= (unsigned)b << (4 * k);
            used[b] = true;
        }
        if (nphases > 0) a.level[a.nlevels - 1].bits |= (unsigned)(nphases + 1) << 16;
        ++nphases;
        for (; t < end; ++t) {
            StreamLevel &l = a.level[a.nlevels++];
            const StageInfo s = stage_info(sc, t);
            const int off = s.log_stride - best, save = saved_behind(t);
            l.off = (unsigned)(s.tw_off * elem);
            l.bits = StreamLevel::pack(s.log_stride, s.radix4, off >> 1, off & 1, save, 0);
            if (save && best != 0 && p.lane(0) != 0) return false;
        }
    }
    return true;
}

}  // namespace bf
