// deep2d.hip -- the shape and width of a 2D or 3D method's passes.
#include "deep2d.hpp"
#include "deep3d.hpp"

namespace cilreg {

DeepPlan plan_deep(int nx, int ny, int rlo, int rhi, const DeepIterCost (&cost)[kDeepShapeCount], int words, int most,
                   int rows_per_thread) {
    constexpr double kCus = 256, kBytesPerUs = 4.5e6;
    DeepPlan best{};
    double best_us = 1e300;
    for (int s = 0; s < kDeepShapeCount; ++s) {
        const DeepShapeCost& c = kDeepShapes[s];
        if (c.r > rows_per_thread) continue;
        const int h = 64 * c.nw / c.lx * c.r;
        for (int w = 1; w <= most; ++w) {
            const int lo = rlo * w, hi = rhi * w;
            // what the inner edges leave of a region (the low ones have none along y)
            const bool rows = h < 32 ? ny <= h : w == 1 || h - lo - hi >= 4;
            if (!rows || (w > 1 && c.lx - lo - hi < 8)) break;
            const Deep2D g = make_deep(nx, ny, c.lx, h, lo, hi);
            // workgroups per CU: whole rounds while few, then about the mean
            const double per = g.nblocks / kCus, load = per <= 4 ? ceil(per) : per + 0.5;
            const double it = load * cost[s].shared_us > cost[s].alone_us ? load * cost[s].shared_us : cost[s].alone_us;
            // reads cover the regions' overlap, writes do not
            const double bytes = 4.0 * words * 0.5 * ((double)g.nblocks * c.lx * h + (double)nx * ny);
            const double us = (c.base_us + w * it + 0.4 * bytes / kBytesPerUs) / w;
            if (us < best_us) {
                best_us = us;
                best = DeepPlan{s, w, g};
            }
        }
    }
    return best;
}

// Time of a pass: rounds of resident workgroups, each marching its chunk and the
// planes it repeats at the chunk's ends, one step per plane.  Every solve pays
// for this search: 256 planes 17 -> 3.4 us on the host by trying each chunk depth
// once instead of every number of chunks.
Deep3Plan plan_deep3(int nx, int ny, int nz, int rlo, int rhi, const Deep3Cost (&cost)[kDeep3Shapes], size_t bytes,
                     int most, int zchunk) {
    constexpr double kLaunchUs = 4.0, kAloneStep = 0.75;
    const bool stream = bytes * nx * ny * nz > kDeep3CacheBytes;
    Deep3Plan best{};
    double best_us = 1e300;
    for (int s = 0; s < kDeep3Shapes; ++s) {
        const Deep3Shape& sh = kDeep3Shapes_[s];
        const int h = sh.nw * sh.r;
        for (int t = 1; t <= most && t <= kDeep3Max; ++t) {
            const int lo = rlo * t, hi = rhi * t;
            if (h - lo - hi < 4) break;
            const long long regions = make_deep3(nx, ny, nz, 64, h, lo, hi, nz).nblocks;
            const double step = stream ? cost[s].stream_us[t - 1] : cost[s].cached_us[t - 1];
            // each chunk depth once: the smallest number of chunks that has it
            for (int c = 1, zc; c <= nz; c = zc > 1 ? (nz + zc - 2) / (zc - 1) : nz + 1) {
                zc = zchunk > 0 ? zchunk : (nz + c - 1) / c;
                const int n = (nz + zc - 1) / zc;
                // a last round of half the workgroups that fit steps faster
                const long long rem = regions * n % sh.slots;
                const double rounds = (double)(regions * n / sh.slots) +
                                      (rem == 0 ? 0.0 : rem <= sh.slots - 256 ? kAloneStep : 1.0);
                const double us = (kLaunchUs + rounds * step * (zc + (n > 1 ? lo + hi : t))) / t;
                if (us < best_us * (1 - 1e-9)) {
                    best_us = us;
                    best = Deep3Plan{s, t, make_deep3(nx, ny, nz, 64, h, lo, hi, zc)};
                }
                if (zchunk > 0) break;
            }
        }
    }
    return best;
}

}  // namespace cilreg
