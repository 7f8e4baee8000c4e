// qt_plan.h -- points per device batch of the sweep, and whether the first pass's
// products stay resident.  Host arithmetic only.
#pragma once
#include <algorithm>
#include <cstddef>

namespace qt {

struct BatchPlan {
    int B = 1;          // points per batch
    bool keep = false;  // the first pass's coupling products stay for the second
};

// npts points of blocks up to nmax on a device with `total` bytes of memory, of
// which `avail` can be had (free, or held by the workspace already);
// bytes(B, keep) is the workspace of B points.  fixed > 0 sets B, extra > 0
// bounds the two things below that are there for speed alone.
//
// Without either, B is 128 points (fewer where they don't fit 0.8 of avail).
//
// More points: a product of n x n blocks is ceil(n / 64)^2 workgroups a member and
// the device takes 512 at once, so blocks of up to 128 need more members to fill
// it: up to 1024 workgroups (n = 64, 256 points: 256 members take the sweep of
// 32 slabs from 23.8 to 12.9 ms).  The workspace is held until the library is
// finished, so they stop at a sixteenth of the memory (1024 points of 64 x 32
// slabs take a twenty-fifth).
//
// Kept products take about half as much again.  They stay where 32 points with them
// fit the device, a rule on device and shape only, so that a point's results
// do not depend on its company; but a call that has not got the memory now runs
// without them (its results then differ by rounding): where the workspace does
// not fit, or where it leaves less than 32 points, from which on the device is
// not filled.
//
// The points are dealt evenly: a batch is padded to B by repeating a point.
template <class Bytes>
BatchPlan plan_batch(int npts, int nmax, size_t avail, size_t total, size_t extra, int fixed, Bytes bytes) {
    const size_t budget = (size_t)(0.80 * (double)avail), kept = extra > 0 ? std::min(extra, budget) : budget;
    const size_t wide = std::min(kept, total / 16);
    const int tiles = ((nmax + 63) / 64) * ((nmax + 63) / 64);
    const int base = std::min(npts, 128), most = std::min(npts, std::max(128, 1024 / tiles));
    auto points = [&](bool keep) {
        if (fixed > 0) return std::min(npts, fixed);
        int B = most;
        while (B > base && bytes(B, keep) > wide) B = B * 3 / 4;
        B = std::max(B, base);
        while (B > 1 && bytes(B, keep) > budget) B = B * 3 / 4;
        return std::max(B, 1);
    };
    BatchPlan p;
    p.keep = bytes(32, true) <= (size_t)(0.80 * (double)total);
    p.B = points(p.keep);
    if (p.keep && (bytes(p.B, true) > kept || (fixed <= 0 && p.B < std::min(npts, 32)))) {
        p.keep = false;
        p.B = points(false);
    }
    if (fixed <= 0) {
        const int parts = (npts + p.B - 1) / p.B;
        p.B = (npts + parts - 1) / parts;
    }
    return p;
}

}  // namespace qt
