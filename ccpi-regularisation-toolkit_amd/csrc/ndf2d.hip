// ndf2d.hip -- NDF (linear and nonlinear diffusion) on a 2D image, many
// iterations per launch (the algorithm and its reference citations: top of
// diffusion.hip; the passes: deep2d.hpp).
#include "solvers.hpp"
#include "ndf_flux.hpp"
#include "deep2d.hpp"

namespace cilreg {

namespace {

struct NdfPar { float lambda, sigma, tau; };
using NdfDeepArgs = DeepArgs<float, 1, NdfPar>;   // state: u

// Registers per point: u, f.  One exchange an iteration (u of a group's first
// and last rows).  Each edge's flux is evaluated once, as in ndf_shared_body,
// but at a group's first row, whose upper flux is cheaper to evaluate again
// than to wait for.  Bound by VALU issue (the fluxes' IEEE divisions), for small
// images by the launch: Huber 256^2 3.3 -> 1.0 us per iteration, 512^2 4.1 -> 1.6,
// 1024^2 7.8 -> 3.5, 2048^2 27 -> 9.8 (before: one iteration per launch).
template <class Sh, int PEN>
__global__ __launch_bounds__(64 * Sh::NW) void ndf_deep_kernel(NdfDeepArgs a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R;
    const DeepPos<Sh> p(a.g);
    __shared__ DeepRow<Sh> ua, ub;
    __shared__ DeepRed<Sh> red;
    float u[R], f[R];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t e = p.elem(r);
        f[r] = a.f[e];
        u[r] = a.cold ? f[r] : ((const float*)a.in[0])[e];
    }
    const bool xfirst = p.x == 0, xlast = p.x == p.nx - 1;
    const float lam = a.par.lambda, sigma = a.par.sigma, tau = a.par.tau;
    int nchk = 0;
    for (int it = 0; it < a.nit; ++it) {
        const int b = it & 1;
        ua.put(p, b, u[0]);
        ub.put(p, b, u[R - 1]);
        __syncthreads();
        const float below = ua.below(p, b), above = ub.above(p, b);
        float e[R], w[R], n[R], s[R];   // differences to x + 1, x - 1, y + 1, y - 1
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            float ul = deep_left(u[r]), ur = deep_right(u[r]);
            float dn = r + 1 < R ? u[r + 1 < R ? r + 1 : r] : below, up = r > 0 ? u[r > 0 ? r - 1 : 0] : above;
            if (p.xedge) {
                deep_keep_branch();
                const float l = ul, q = ur;
                ul = xfirst ? q : l;
                ur = xlast ? l : q;
            }
            if (p.yedge) {
                deep_keep_branch();
                const float l = up, q = dn;
                up = p.y + r == 0 ? q : l;
                dn = p.y + r == p.ny - 1 ? l : q;
            }
            e[r] = ur - u[r];
            w[r] = ul - u[r];
            n[r] = dn - u[r];
            s[r] = up - u[r];
        }
        if constexpr (PEN != 0) {
            #pragma unroll
            for (int r = 0; r < R; ++r) {
                const float fe = ndf_flux<PEN>(e[r], sigma), fl = deep_left(fe);
                w[r] = xfirst ? fe : ndf_flux_mirror<PEN>(w[r], fl, sigma);
                e[r] = fe;
                n[r] = ndf_flux<PEN>(n[r], sigma);
                s[r] = r == 0 ? ndf_flux<PEN>(s[r], sigma) : ndf_flux_mirror<PEN>(s[r], n[r > 0 ? r - 1 : 0], sigma);
            }
        }
        double sd = 0.0, su = 0.0;
        const bool check = (a.check >> it) & 1u;
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const float t = e[r] + w[r] + n[r] + s[r];
            const float un = u[r] + tau * (lam * t - (u[r] - f[r]));
            if (check && p.out(r)) {
                const float df = un - u[r];
                sd += (double)df * (double)df;
                su += (double)un * (double)un;
            }
            u[r] = un;
        }
        if (check) {
            deep_check<Sh>(red, sd, su, nchk);
            ++nchk;
        }
    }
    #pragma unroll
    for (int r = 0; r < R; ++r)
        if (p.out(r)) {
            const size_t e = p.elem(r);
            if (a.write_state) ((float*)a.out[0])[e] = u[r];
            if (a.write_res) a.res[e] = u[r];
        }
    deep_store_checks<Sh>(red, nchk, a.partials, a.g.nblocks, p.lin);
}

struct NdfDeep : DeepMethod {
    using Args = NdfDeepArgs;
    static constexpr int NF = 1, rlo = 1, rhi = 1, words = 3;
    static constexpr DeepIterCost cost[kDeepShapeCount] = {{0.5, 0.4}, {0.7, 0.65}, {1.1, 1.05}, {0.75, 0.55}, {0.45, 0.115},
                                                              {0.50, 0.17}};
    static constexpr bool seeded = false;
    NdfPar par;
    int penalty;
    size_t field_size(int) const { return sizeof(float); }
    void prepare(Args& a, int, int, bool) const { a.par = par; }
    template <class Sh, int PEN>
    void go(const Args& a, hipStream_t s) const {
        hipLaunchKernelGGL((ndf_deep_kernel<Sh, PEN>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
    }
    template <class Sh>
    void launch(const Args& a, hipStream_t s) const {
        switch (penalty) {
            case 1: go<Sh, 1>(a, s); break;
            case 2: go<Sh, 2>(a, s); break;
            case 3: go<Sh, 3>(a, s); break;
            case 4: go<Sh, 4>(a, s); break;
            case 5: go<Sh, 5>(a, s); break;
            default: go<Sh, 0>(a, s); break;
        }
    }
    void load(int, void*, const WarmState&, size_t, hipStream_t) const {}
    void store(int, const void*, const WarmState&, size_t, hipStream_t) const {}
};

}  // namespace

int ndf_solve_2d(const float* d_f, float* d_out, float lambda, float sigma, int iter, float tau, int penalty,
                 float epsil, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re) {
    NdfDeep m;
    m.par = NdfPar{lambda, sigma, tau};
    m.penalty = penalty;
    return deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, nullptr);
}

}  // namespace cilreg
