// rof2d.hip -- ROF-TV on a 2D image, many iterations per launch (the
// algorithm and its reference citations: top of rof.hip; the passes:
// deep2d.hpp).
#include "solvers.hpp"
#include "rof_kernels.hpp"
#include "deep2d.hpp"

namespace cilreg {

namespace {

struct RofPar { float lambda, tau; };
using RofDeepArgs = DeepArgs<float, 1, RofPar>;   // state: u

// The fluxes D1 (along y) and D2 (along x) of N points from u there (uc) and
// its mirrored neighbours: the values of rof_flux_math<2>.  In-range points
// take sqrt_in and div_in; one test sends a wave with any other point (as in
// rof_flux_math) to rof_flux_ref.
template <int N>
__device__ inline void rof2d_fluxes(const float (&uc)[N], const float (&ul)[N], const float (&ur)[N],
                                    const float (&uu)[N], const float (&ud)[N], float (&d1)[N], float (&d2)[N]) {
    float x1[N], x2[N], prod = 0.0f, sq = 0.0f;
    uint32_t key = ~0u;
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        const float fi = ur[r] - uc[r], bi = uc[r] - ul[r], fj = ud[r] - uc[r], bj = uc[r] - uu[r];
        const float mi = __builtin_amdgcn_fmed3f(fi, bi, 0.f), mj = __builtin_amdgcn_fmed3f(fj, bj, 0.f);
        const float s1 = fj * fj + mi * mi, s2 = fi * fi + mj * mj;
        prod = __builtin_fmaf(fi, bi, prod);
        prod = __builtin_fmaf(fj, bj, prod);
        sq = sq + s1;
        sq = sq + s2;
        key = min_key(key, min_key(tiny_key(fi), tiny_key(fj)));
        x1[r] = (float)((double)s1 + 1.0e-8);
        x2[r] = (float)((double)s2 + 1.0e-8);
        d1[r] = fj;
        d2[r] = fi;
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(rof_odd(prod, sq) || key < kTinyKey) != 0, 0)) {
        #pragma unroll
        for (int r = 0; r < N; ++r) {
            float d3;
            rof_flux_ref<2, float>(uc[r], ur[r], ul[r], ud[r], uu[r], 0.f, 0.f, d1[r], d2[r], d3, 1.0e-8);
        }
        return;
    }
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        const float b1 = sqrt_in(x1[r]), b2 = sqrt_in(x2[r]);
        d1[r] = div_in(d1[r], b1, rcp_in(b1));
        d2[r] = div_in(d2[r], b2, rcp_in(b2));
    }
}

// Bound by VALU issue (about 60 instructions per point and iteration, a third
// of them in two square roots and two quotients): 256^2 3.4 -> 1.3 us per
// iteration, 512^2 3.4 -> 1.8, 1024^2 8.5 -> 4.0, 2048^2 27 -> 11.8 (before:
// two iterations per launch through LDS below 2^20 pixels, one above).  Three
// columns and rows are lost per iteration (two for the other methods), which
// is what limits the pass at large sizes.
//
// Registers per point: u, f and (transient) the fluxes.  Two exchanges an
// iteration: u of a group's first and last row, then D1 of its last row (with
// one row per group also the row below's, the mirrored neighbour of row 0).
// 64 VGPRs keep two 1024-thread workgroups on a CU (68 without the cap; four
// spilled): 1024^2 4.7 -> 4.0 us per iteration.
template <class Sh>
constexpr int rof_deep_waves() { return Sh::R == 4 ? 8 : 1; }
template <class Sh>
__global__ __launch_bounds__(64 * Sh::NW) __attribute__((amdgpu_waves_per_eu(rof_deep_waves<Sh>())))
void rof_deep_kernel(RofDeepArgs a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R;
    using T = float;
    const DeepPos<Sh> p(a.g);
    __shared__ DeepRow<Sh> upu, dnu, dnd;
    __shared__ DeepRed<Sh> red;

    T u[R], f[R];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t e = p.elem(r);
        f[r] = a.f[e];
        u[r] = a.cold ? f[r] : ((const T*)a.in[0])[e];
    }
    const bool xfirst = p.x == 0, xlast = p.x == p.nx - 1;
    const T lam = a.par.lambda, tau = a.par.tau;
    int nchk = 0;
    for (int it = 0; it < a.nit; ++it) {
        const int b = it & 1;
        upu.put(p, b, u[0]);
        dnu.put(p, b, u[R - 1]);
        __syncthreads();
        const T ub = upu.below(p, b), ua = dnu.above(p, b);
        T ul[R], ur[R], uu[R], ud[R], d1[R], d2[R];
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const T l = deep_left(u[r]), q = deep_right(u[r]);
            ul[r] = l;
            ur[r] = q;
            if (p.xedge) {
                deep_keep_branch();
                ul[r] = xfirst ? q : l;
                ur[r] = xlast ? l : q;
                if (R == 1 && p.nx == 1) ul[r] = ur[r] = u[r];   // the mirror of a single column is itself
            }
            const T dn = r + 1 < R ? u[r + 1 < R ? r + 1 : r] : ub, up = r > 0 ? u[r > 0 ? r - 1 : 0] : ua;
            uu[r] = up;
            ud[r] = dn;
            if (p.yedge) {
                deep_keep_branch();
                uu[r] = p.y + r == 0 ? dn : up;
                ud[r] = p.y + r == p.ny - 1 ? up : dn;
                if (R == 1 && p.ny == 1) uu[r] = ud[r] = u[r];
            }
        }
        rof2d_fluxes(u, ul, ur, uu, ud, d1, d2);
        dnd.put(p, b, d1[R - 1]);
        __syncthreads();
        const T da = dnd.above(p, b), db = R == 1 ? dnd.below(p, b) : (T)0;
        double sd = 0.0, su = 0.0;
        const bool check = (a.check >> it) & 1u;
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const T l = deep_left(d2[r]), q = deep_right(d2[r]);
            T d2m = l;
            if (p.xedge) {
                deep_keep_branch();
                d2m = xfirst ? q : l;
                if (R == 1 && p.nx == 1) d2m = d2[r];
            }
            T d1m = r > 0 ? d1[r > 0 ? r - 1 : 0] : da;
            if (r == 0 && p.yedge) {
                deep_keep_branch();
                d1m = p.y == 0 ? (R > 1 ? d1[R > 1 ? 1 : 0] : db) : d1m;
                if (R == 1 && p.ny == 1) d1m = d1[0];
            }
            const T dv = (d1[r] - d1m) + (d2[r] - d2m);
            const T un = u[r] + tau * (lam * dv - (u[r] - f[r]));
            if (check && p.out(r)) {
                const T df = un - u[r];
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
            if (a.write_state) ((T*)a.out[0])[e] = u[r];
            if (a.write_res) a.res[e] = u[r];
        }
    deep_store_checks<Sh>(red, nchk, a.partials, a.g.nblocks, p.lin);
}

struct RofDeep : DeepMethod {
    using Args = RofDeepArgs;
    // D1, D2 at the low neighbours read u two columns / rows away
    static constexpr int NF = 1, rlo = 2, rhi = 1, words = 3;
    static constexpr DeepIterCost cost[kDeepShapeCount] = {{0.75, 0.61}, {1.12, 1.00}, {1.95, 1.70}, {1.30, 0.86}, {0.60, 0.11},
                                                              {0.70, 0.18}};
    static constexpr bool seeded = false;
    // a single column or row mirrors onto itself, which only the kernels of one
    // row per thread provide for (in the others it costs two more spilled registers)
    static int most_rows(int nx, int ny) { return nx > 1 && ny > 1 ? 4 : 1; }
    RofPar par;
    size_t field_size(int) const { return sizeof(float); }
    void prepare(Args& a, int, int, bool) const { a.par = par; }
    template <class Sh>
    void launch(const Args& a, hipStream_t s) const {
        hipLaunchKernelGGL((rof_deep_kernel<Sh>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
    }
    void load(int, void*, const WarmState&, size_t, hipStream_t) const {}
    void store(int, const void*, const WarmState&, size_t, hipStream_t) const {}
};

}  // namespace

int rof_solve_2d(const float* d_f, float* d_out, float lambda, int iter, float tau, float epsil, int nx, int ny,
                 const Opts& opts, hipStream_t s, int* iters_done, float* re) {
    RofDeep m;
    m.par.lambda = lambda;
    m.par.tau = tau;
    return deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, nullptr);
}

}  // namespace cilreg
