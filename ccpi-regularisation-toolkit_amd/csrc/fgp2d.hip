// fgp2d.hip -- FGP-TV on a 2D image, many iterations per launch (the
// algorithm and its reference citations: top of fgp.hip; the passes:
// deep2d.hpp).
#include "solvers.hpp"
#include "deep2d.hpp"

namespace cilreg {

namespace {

struct FgpPar {
    float lambda, step, mult[kDeepMax];   // mult[i]: of the pass's iteration i
    int nonneg;
    const float* B[2];                    // FGP-dTV only
};
// state: P_k (2 components), P_{k-1} (2)
using FgpDeepArgs = DeepArgs<float, 4, FgpPar>;

// Bound by VALU issue (about 50 instructions per point and iteration) and, for
// small images, by the launch: 256^2 3.6 -> 0.92 us per iteration, 512^2 4.6
// -> 1.3, 1024^2 8.7 -> 2.8, 2048^2 28 -> 8.1 (before: two iterations per
// launch through LDS below 2^20 pixels, one above).
//
// Registers per point: P_k, P_{k-1}, f and (transient) R_k, D_k; a seeded
// check reads D_{k-1} from res, where the pass's last D is written: each point
// that matters is read and written by one thread.  Row groups exchange R_k
// once per iteration -- R2 of a group's last row downwards, R1 and R2 of its
// first row upwards -- and every group evaluates D_k of the row below its last
// one itself (8 operations) instead of waiting for it, so one barrier an
// iteration suffices.
//
// DIR: FGP-dTV (top of dtv.hip).  R_k and the gradient of D_k are projected
// onto the line orthogonal to the reference's normalised gradient B; a pass
// loads B once.  256^2 3.3 -> 1.0 us per iteration, 512^2 4.1 -> 1.5, 1024^2 9.2
// -> 4.0, 2048^2 35 -> 13.7 (before: one iteration per launch).
template <class Sh, typename S, bool ISO, bool DIR>
__global__ __launch_bounds__(64 * Sh::NW) void fgp_deep_kernel(FgpDeepArgs a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R;
    using T = float;
    const DeepPos<Sh> p(a.g);
    __shared__ DeepRow<Sh> up1, up2, dn2;
    __shared__ DeepRed<Sh> red;

    T c1[R], c2[R], m1[R], m2[R], f[R + 1], dprev[R];   // P_k, P_{k-1}, f (and the row below), D_{k-1}
    #pragma unroll
    for (int r = 0; r <= R; ++r) f[r] = a.f[p.elem(r)];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t e = p.elem(r);
        c1[r] = c2[r] = m1[r] = m2[r] = dprev[r] = 0;
        if (!a.cold) {
            c1[r] = ldT<T>((const S*)a.in[0], e);
            c2[r] = ldT<T>((const S*)a.in[1], e);
            m1[r] = ldT<T>((const S*)a.in[2], e);
            m2[r] = ldT<T>((const S*)a.in[3], e);
        }
        if (a.check & 1u) dprev[r] = a.res[e];
    }
    T bx[R], by[R];
    if (DIR) {
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const size_t e = p.elem(r);
            bx[r] = a.par.B[0][e];
            by[r] = a.par.B[1][e];
        }
    }
    // v less its component along B (FGP_dTV_core.c:210-223)
    auto orthogonal = [&](T& v1, T& v2, int r) {
        const T ip = v1 * bx[r] + v2 * by[r];
        v1 = v1 - ip * bx[r];
        v2 = v2 - ip * by[r];
    };
    const bool xlast = p.x == p.nx - 1;
    const T lam = a.par.lambda, step = a.par.step;
    const bool nonneg = a.par.nonneg;
    int nchk = 0;
    for (int it = 0; it < a.nit; ++it) {
        const T m = a.par.mult[it];
        const int b = it & 1;
        T r1[R], r2[R], d[R + 1];
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            r1[r] = c1[r] + m * (c1[r] - m1[r]);
            r2[r] = c2[r] + m * (c2[r] - m2[r]);
            if (DIR) orthogonal(r1[r], r2[r], r);
        }
        up1.put(p, b, r1[0]);
        up2.put(p, b, r2[0]);
        dn2.put(p, b, r2[R - 1]);
        __syncthreads();
        const T n1 = up1.below(p, b), n2 = up2.below(p, b);
        const T ab = dn2.above(p, b);
        const T above = p.grp > 0 ? ab : (T)0;   // group 0: the image's first row, or an edge
        #pragma unroll
        for (int r = 0; r <= R; ++r) {
            const T q1 = r < R ? r1[r < R ? r : 0] : n1, q2 = r < R ? r2[r < R ? r : 0] : n2;
            const T b1 = deep_left0(p, q1);
            const T b2 = r == 0 ? above : r2[r > 0 ? r - 1 : 0];
            d[r] = f[r] - lam * (q1 + q2 - b1 - b2);
        }
        if (nonneg) {
            #pragma unroll
            for (int r = 0; r <= R; ++r) d[r] = d[r] < (T)0 ? (T)0 : d[r];
        }
        if ((a.check >> it) & 1u) {
            double sd = 0.0, su = 0.0;
            #pragma unroll
            for (int r = 0; r < R; ++r)
                if (p.out(r)) {
                    const T df = d[r] - dprev[r];
                    sd += (double)df * (double)df;
                    su += (double)d[r] * (double)d[r];
                }
            deep_check<Sh>(red, sd, su, nchk);
            ++nchk;
        }
        T p1[R], p2[R], p3[R];
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const T dx = deep_right(d[r]);
            T g1 = d[r] - dx, g2 = d[r] - d[r + 1];
            if (p.xedge) {
                deep_keep_branch();
                g1 = xlast ? (T)0 : g1;
            }
            if (p.yedge) {
                deep_keep_branch();
                g2 = (p.y + r == p.ny - 1) ? (T)0 : g2;
            }
            if (DIR) orthogonal(g1, g2, r);
            p1[r] = r1[r] + step * g1;
            p2[r] = r2[r] + step * g2;
            p3[r] = 0;
        }
        project_unit_n<2, T, ISO>(p1, p2, p3);
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            m1[r] = c1[r];
            m2[r] = c2[r];
            c1[r] = through_storage<T, S>(p1[r]);
            c2[r] = through_storage<T, S>(p2[r]);
            dprev[r] = d[r];
        }
    }
    #pragma unroll
    for (int r = 0; r < R; ++r)
        if (p.out(r)) {
            const size_t e = p.elem(r);
            if (a.write_state) {
                stT<T>((S*)a.out[0], e, c1[r]);
                stT<T>((S*)a.out[1], e, c2[r]);
                stT<T>((S*)a.out[2], e, m1[r]);
                stT<T>((S*)a.out[3], e, m2[r]);
            }
            if (a.write_res) a.res[e] = dprev[r];
        }
    deep_store_checks<Sh>(red, nchk, a.partials, a.g.nblocks, p.lin);
}

template <typename S, bool DIR = false>
struct FgpDeep : DeepMethod {
    using Args = FgpDeepArgs;
    static constexpr int NF = 4, rlo = 1, rhi = 1, words = DIR ? 11 : 9;
    static constexpr DeepIterCost cost[kDeepShapeCount] = {{0.52, 0.42}, {0.70, 0.72}, {1.08, 1.15}, {0.72, 0.50}, {0.50, 0.085},
                                                              {0.55, 0.12}};
    static constexpr bool seeded = true;
    float lambda, step;
    int nonneg;
    bool iso;
    std::vector<float> mult;
    const float* B[2] = {nullptr, nullptr};
    size_t field_size(int) const { return sizeof(S); }
    void prepare(Args& a, int k, int nk, bool) const {
        a.par.lambda = lambda;
        a.par.step = step;
        a.par.nonneg = nonneg;
        a.par.B[0] = B[0];
        a.par.B[1] = B[1];
        for (int i = 0; i < kDeepMax; ++i) a.par.mult[i] = i < nk ? mult[k + i] : 0.0f;
    }
    template <class Sh>
    void launch(const Args& a, hipStream_t s) const {
        if (iso) hipLaunchKernelGGL((fgp_deep_kernel<Sh, S, true, DIR>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
        else hipLaunchKernelGGL((fgp_deep_kernel<Sh, S, false, DIR>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
    }
    // caller state channels: P1, P2, P3, then the previous P1, P2, P3
    static size_t channel(int i) { return i < 2 ? i : 3 + (i - 2); }
    void load(int i, void* dst, const WarmState& ws, size_t n, hipStream_t s) const {
        state_in<S>((S*)dst, ws.d_state + channel(i) * n, n, s);
    }
    void store(int i, const void* src, const WarmState& ws, size_t n, hipStream_t s) const {
        state_out<S>(ws.d_state + channel(i) * n, (const S*)src, n, s);
    }
};

}  // namespace

template <typename S>
int fgp_solve_2d(const float* d_f, float* d_out, float lambda, int iter, float epsil, int method, int nonneg, int nx,
                 int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws) {
    FgpDeep<S> m;
    m.lambda = lambda;
    m.step = 1.0f / (8.0f * lambda);
    m.nonneg = nonneg != 0;
    m.iso = method == 0;
    std::vector<float> tks;
    fgp_multipliers(iter, ws, m.mult, tks);
    int last = 0;
    if (deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, ws, &last) != 0) return -1;
    if (ws) {
        ws->tstate[0] = tks[last + 1];
        ws->tstate[1] = m.mult[last + 1];
    }
    return 0;
}

// FGP-dTV; refgrad queues the kernel that computes B, mult holds the t_k sequence's factors.
int dtv_solve_2d(const float* d_f, const RefGrad& refgrad, float* d_out, float lambda, int iter, float epsil,
                 int method, int nonneg, int nx, int ny, const std::vector<float>& mult, const Opts& opts,
                 hipStream_t s, int* iters_done, float* re) {
    FgpDeep<float, true> m;
    m.lambda = lambda;
    m.step = 1.0f / (8.0f * lambda);
    m.nonneg = nonneg != 0;
    m.iso = method == 0;
    m.mult = mult;
    const DeepExtra b{2, [&](float* const (&B)[3]) {
        m.B[0] = B[0];
        m.B[1] = B[1];
        refgrad({B[0], B[1], B[1]});   // two components
    }};
    return deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, nullptr, nullptr, &b);
}

template int fgp_solve_2d<float>(const float*, float*, float, int, float, int, int, int, int, const Opts&, hipStream_t,
                                 int*, float*, const WarmState*);
template int fgp_solve_2d<bf16_t>(const float*, float*, float, int, float, int, int, int, int, const Opts&,
                                  hipStream_t, int*, float*, const WarmState*);
template int fgp_solve_2d<_Float16>(const float*, float*, float, int, float, int, int, int, int, const Opts&,
                                    hipStream_t, int*, float*, const WarmState*);

}  // namespace cilreg
