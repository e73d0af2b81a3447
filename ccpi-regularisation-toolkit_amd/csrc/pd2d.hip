// pd2d.hip -- PD-TV on a 2D image, many iterations per launch (the algorithm
// and its reference citations: top of pd.hip; the passes: deep2d.hpp).
#include "solvers.hpp"
#include "deep2d.hpp"

namespace cilreg {

namespace {

struct PdPar {
    float sigma, tau, lt;
    double c, rlo, rhi;  // 1 + lt, bounds of its reciprocal
    int nonneg, plain;   // plain: the result is U before extrapolation (a stop), else u_bar
};
// state: u_bar, P (2 components)
using PdDeepArgs = DeepArgs<float, 3, PdPar>;

// Bound by VALU issue and, for small images, by the launch: 256^2 3.5 -> 0.94
// us per iteration, 512^2 4.2 -> 1.5, 1024^2 7.6 -> 3.3, 2048^2 31.6 -> 9.9
// (before: one iteration per launch).
//
// Registers per point: u_bar, P, f.  Two exchanges an iteration: u_bar of a
// group's first and last row (the forward difference, mirrored at the image's
// last row), then the new P2 of its last row.
template <class Sh, typename S, bool ISO>
__global__ __launch_bounds__(64 * Sh::NW) void pd_deep_kernel(PdDeepArgs a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R;
    using T = float;
    const DeepPos<Sh> p(a.g);
    __shared__ DeepRow<Sh> upu, dnu, dnq;
    __shared__ DeepRed<Sh> red;

    T u[R], q1[R], q2[R], q3[R], f[R], un[R];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t e = p.elem(r);
        f[r] = a.f[e];
        u[r] = a.cold ? f[r] : ((const T*)a.in[0])[e];
        q1[r] = a.cold ? (T)0 : ldT<T>((const S*)a.in[1], e);
        q2[r] = a.cold ? (T)0 : ldT<T>((const S*)a.in[2], e);
        q3[r] = 0;
        un[r] = 0;
    }
    const bool xlast = p.x == p.nx - 1, nonneg = a.par.nonneg;
    const T sigma = a.par.sigma, tau = a.par.tau, lt = a.par.lt;
    int nchk = 0;
    for (int it = 0; it < a.nit; ++it) {
        const int b = it & 1;
        upu.put(p, b, u[0]);
        dnu.put(p, b, u[R - 1]);
        __syncthreads();
        const T ub = upu.below(p, b), ua = dnu.above(p, b);
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const T ur = deep_right(u[r]), ul = deep_left(u[r]);
            T ux = ur;
            if (p.xedge) {
                deep_keep_branch();
                ux = xlast ? ul : ur;
            }
            const T dn = r + 1 < R ? u[r + 1 < R ? r + 1 : r] : ub, up = r > 0 ? u[r > 0 ? r - 1 : 0] : ua;
            T uy = dn;
            if (p.yedge) {
                deep_keep_branch();
                uy = (p.y + r == p.ny - 1) ? up : dn;
            }
            q1[r] = q1[r] + sigma * (ux - u[r]);
            q2[r] = q2[r] + sigma * (uy - u[r]);
        }
        project_unit_n<2, T, ISO>(q1, q2, q3);
        dnq.put(p, b, q2[R - 1]);
        __syncthreads();
        const T qa = dnq.above(p, b);
        const T above = p.grp > 0 ? qa : (T)0;   // P2(-1) = 0 at the image's first row; elsewhere an edge
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            if (nonneg) u[r] = u[r] < (T)0 ? (T)0 : u[r];
            // -(q - 0) is -q: no select at the first column and row
            const T dv = -(q1[r] - deep_left0(p, q1[r])) + -(q2[r] - (r > 0 ? q2[r > 0 ? r - 1 : 0] : above));
            un[r] = u[r] - tau * dv + lt * f[r];
        }
        Mixed<T>::pd_div_n(un, a.par.c, a.par.rlo, a.par.rhi);
        if ((a.check >> it) & 1u) {
            double sd = 0.0, su = 0.0;
            #pragma unroll
            for (int r = 0; r < R; ++r)
                if (p.out(r)) {
                    const T df = un[r] - u[r];
                    sd += (double)df * (double)df;
                    su += (double)un[r] * (double)un[r];
                }
            deep_check<Sh>(red, sd, su, nchk);
            ++nchk;
        }
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            u[r] = un[r] + (un[r] - u[r]);
            q1[r] = through_storage<T, S>(q1[r]);
            q2[r] = through_storage<T, S>(q2[r]);
        }
    }
    #pragma unroll
    for (int r = 0; r < R; ++r)
        if (p.out(r)) {
            const size_t e = p.elem(r);
            if (a.write_state) {
                ((T*)a.out[0])[e] = u[r];
                stT<T>((S*)a.out[1], e, q1[r]);
                stT<T>((S*)a.out[2], e, q2[r]);
            }
            if (a.write_res) a.res[e] = a.par.plain ? un[r] : u[r];
        }
    deep_store_checks<Sh>(red, nchk, a.partials, a.g.nblocks, p.lin);
}

template <typename S>
struct PdDeep : DeepMethod {
    using Args = PdDeepArgs;
    static constexpr int NF = 3, rlo = 1, rhi = 1, words = 7;
    static constexpr DeepIterCost cost[kDeepShapeCount] = {{0.53, 0.48}, {0.85, 0.82}, {1.40, 1.70}, {0.85, 0.70}, {0.50, 0.09},
                                                              {0.55, 0.12}};
    static constexpr bool seeded = false;
    PdPar par;
    bool iso;
    size_t field_size(int i) const { return i == 0 ? sizeof(float) : sizeof(S); }
    void prepare(Args& a, int, int, bool stop) const {
        a.par = par;
        a.par.plain = stop;
    }
    template <class Sh>
    void launch(const Args& a, hipStream_t s) const {
        if (iso) hipLaunchKernelGGL((pd_deep_kernel<Sh, S, true>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
        else hipLaunchKernelGGL((pd_deep_kernel<Sh, S, false>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
    }
    // caller state channels: u_bar, P1, P2, P3
    void load(int i, void* dst, const WarmState& ws, size_t n, hipStream_t s) const {
        if (i == 0) state_in<float>((float*)dst, ws.d_state, n, s);
        else state_in<S>((S*)dst, ws.d_state + (size_t)i * n, n, s);
    }
    void store(int i, const void* src, const WarmState& ws, size_t n, hipStream_t s) const {
        if (i == 0) state_out<float>(ws.d_state, (const float*)src, n, s);
        else state_out<S>(ws.d_state + (size_t)i * n, (const S*)src, n, s);
    }
};

}  // namespace

template <typename S>
int pd_solve_2d(const float* d_f, float* d_out, float lambda, int iter, float epsil, float lipschitz, int method,
                int nonneg, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                const WarmState* ws) {
    PdDeep<S> m;
    // step sizes in float (PD_TV_core.c:50-53)
    m.par.tau = lambda * 0.1f;
    m.par.sigma = (float)(1.0 / (double)(lipschitz * m.par.tau));
    m.par.lt = m.par.tau / lambda;
    m.par.c = 1.0 + (double)m.par.lt;
    m.par.rlo = 1.0 / m.par.c * (1.0 - 0x1p-50);
    m.par.rhi = 1.0 / m.par.c * (1.0 + 0x1p-50);
    m.par.nonneg = nonneg != 0;
    m.par.plain = 0;
    m.iso = method == 0;
    return deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, ws);
}

template int pd_solve_2d<float>(const float*, float*, float, int, float, float, int, int, int, int, const Opts&,
                                hipStream_t, int*, float*, const WarmState*);
template int pd_solve_2d<bf16_t>(const float*, float*, float, int, float, float, int, int, int, int, const Opts&,
                                 hipStream_t, int*, float*, const WarmState*);
template int pd_solve_2d<_Float16>(const float*, float*, float, int, float, float, int, int, int, int, const Opts&,
                                   hipStream_t, int*, float*, const WarmState*);

}  // namespace cilreg
