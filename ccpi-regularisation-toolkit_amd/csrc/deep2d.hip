// deep2d.hip -- the shape and width of a 2D method's passes.
#include "deep2d.hpp"

namespace cilreg {

DeepPlan plan_deep(int nx, int ny, int rlo, int rhi, const DeepIterCost (&cost)[kDeepShapeCount], int words, int most) {
    constexpr double kCus = 256, kBytesPerUs = 4.5e6;
    DeepPlan best{};
    double best_us = 1e300;
    for (int s = 0; s < kDeepShapeCount; ++s) {
        const DeepShapeCost& c = kDeepShapes[s];
        const int h = 64 * c.nw / c.lx * c.r;
        for (int w = 1; w <= most; ++w) {
            const int lo = rlo * w, hi = rhi * w;
            if (w > 1 && (c.lx - lo - hi < 8 || h - lo - hi < 4)) break;
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

}  // namespace cilreg
