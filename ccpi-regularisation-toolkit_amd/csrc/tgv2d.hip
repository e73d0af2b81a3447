// tgv2d.hip -- TGV on a 2D image, many iterations per launch (the algorithm
// and its reference citations: top of tgv.hip; the passes: deep2d.hpp).
#include "solvers.hpp"
#include "tgv_kernels.hpp"
#include "deep2d.hpp"

namespace cilreg {

namespace {

struct TgvPar {
    float lambda, tau, alpha1, alpha0;
    float ra1, ra0;        // 1 / alpha1, 1 / alpha0
    float lt, rlt;         // lambda + tau and its reciprocal
    float lim1, lim0;      // |P|^2, |Q|^2 above which the norm's quotient leaves div_in's range
    int fast;              // alpha1, alpha0, lambda + tau in range of div_in
};
// state: u_bar, v_bar (2 components), P (2), Q11, Q22, Q12
using TgvDeepArgs = DeepArgs<float, 8, TgvPar>;

// alpha-ball projection of N points: v_i / max(|v| / alpha, 1) for the NC
// components, ss their (weighted) sum of squares.  |v| / alpha > 1 decides as
// in the reference: below 2^-90 the sum is raised to it, where the quotient is
// far under 1 (fast: alpha >= 2^-30).  A point inside the ball divides by 1,
// which leaves it as it is.  A wave with a sum above lim or NaN (a point that
// holds an infinity beside a NaN keeps it: the reference scales nothing there,
// and div_in would turn it into a NaN), or with a component in (0, 2^-100) that
// is really divided, takes the reference's expressions.  One test serves the N
// sums: their total is NaN if one is, and above lim if one is.
template <int NC, int N>
__device__ inline bool tgv2d_ball(float (&v)[NC][N], const float (&ss)[N], float alpha, float ra, float lim,
                                  bool fast) {
    float n[N], total = 0.0f;
    bool odd = !fast;
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        total = total + ss[r];
        const float w = sqrt_in(__builtin_fmaxf(ss[r], 0x1p-90f));
        const float m = div_in(w, alpha, ra);
        n[r] = __builtin_fmaxf(m, 1.0f);
        uint32_t key = tiny_key(v[0][r]);
        #pragma unroll
        for (int c = 1; c < NC; ++c) key = min_key(key, tiny_key(v[c][r]));
        odd = odd || (key < kTinyKey && m > 1.0f);
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd || !(total <= lim)) != 0, 0)) {
        #pragma unroll
        for (int r = 0; r < N; ++r) {
            const float m = sqrtf(ss[r]) / alpha;
            if (m > 1.0f) {
                #pragma unroll
                for (int c = 0; c < NC; ++c) v[c][r] = v[c][r] / m;
            }
        }
        return false;
    }
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        const float rn = rcp_in(n[r]);
        #pragma unroll
        for (int c = 0; c < NC; ++c) v[c][r] = div_in(v[c][r], n[r], rn);
    }
    return true;
}

// Bound by VALU issue, above 1024^2 also by its 68 B per point and pass:
// 256^2 4.3 -> 1.7 us per iteration, 512^2 5.7 -> 2.7, 1024^2 18.5 -> 7.5,
// 2048^2 60 -> 24 (before: one iteration per launch).
//
// Registers per point: u_bar, v_bar, P, Q, f.  Two exchanges an iteration:
// u_bar and v_bar of a group's first row, then the new P2, Q22 and Q12 of its
// last row.
// 80 VGPRs keep three 512-thread workgroups on a CU (92 without the cap; four
// spilled): 2048^2 25.5 -> 24.1 us per iteration.
template <class Sh>
constexpr int tgv_deep_waves() { return Sh::R == 4 && Sh::NW == 8 ? 6 : 1; }
template <class Sh, typename S>
__global__ __launch_bounds__(64 * Sh::NW) __attribute__((amdgpu_waves_per_eu(tgv_deep_waves<Sh>())))
void tgv_deep_kernel(TgvDeepArgs a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R;
    using T = float;
    const DeepPos<Sh> p(a.g);
    __shared__ DeepRow<Sh> uu, uv1, uv2, dp2, dq22, dq12;
    __shared__ DeepRed<Sh> red;

    T u[R], v1[R], v2[R], P[2][R], Q[3][R], f[R];   // Q: Q11, Q22, Q12
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t e = p.elem(r);
        f[r] = a.f[e];
        u[r] = f[r];
        v1[r] = v2[r] = P[0][r] = P[1][r] = Q[0][r] = Q[1][r] = Q[2][r] = 0;
        if (!a.cold) {
            u[r] = ((const T*)a.in[0])[e];
            v1[r] = ldT<T>((const S*)a.in[1], e);
            v2[r] = ldT<T>((const S*)a.in[2], e);
            P[0][r] = ldT<T>((const S*)a.in[3], e);
            P[1][r] = ldT<T>((const S*)a.in[4], e);
            Q[0][r] = ldT<T>((const S*)a.in[5], e);
            Q[1][r] = ldT<T>((const S*)a.in[6], e);
            Q[2][r] = ldT<T>((const S*)a.in[7], e);
        }
    }
    const bool xlast = p.x == p.nx - 1, xneg = xlast && p.x > 0;
    const TgvPar& k = a.par;
    const T tau = k.tau, sigma = k.tau;
    int nchk = 0;
    for (int it = 0; it < a.nit; ++it) {
        const int b = it & 1;
        uu.put(p, b, u[0]);
        uv1.put(p, b, v1[0]);
        uv2.put(p, b, v2[0]);
        __syncthreads();
        const T ub = uu.below(p, b), v1b = uv1.below(p, b), v2b = uv2.below(p, b);
        T np[R], nq[R];
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const int rd = r + 1 < R ? r + 1 : r;
            const T ux = deep_right(u[r]), v1x = deep_right(v1[r]), v2x = deep_right(v2[r]);
            const T uy = r + 1 < R ? u[rd] : ub, v1y = r + 1 < R ? v1[rd] : v1b, v2y = r + 1 < R ? v2[rd] : v2b;
            T e1 = (ux - u[r]) - v1[r], e2 = (uy - u[r]) - v2[r];
            T d11 = v1x - v1[r], d12 = v1y - v1[r], d21 = v2x - v2[r], d22 = v2y - v2[r];
            if (p.xedge) {
                deep_keep_branch();
                e1 = xlast ? -v1[r] : e1;
                d11 = xlast ? (T)0 : d11;
                d21 = xlast ? (T)0 : d21;
            }
            if (p.yedge) {
                deep_keep_branch();
                const bool yl = p.y + r == p.ny - 1;
                e2 = yl ? -v2[r] : e2;
                d12 = yl ? (T)0 : d12;
                d22 = yl ? (T)0 : d22;
            }
            P[0][r] = P[0][r] + sigma * e1;
            P[1][r] = P[1][r] + sigma * e2;
            Q[0][r] = Q[0][r] + sigma * d11;
            Q[1][r] = Q[1][r] + sigma * d22;
            Q[2][r] = Q[2][r] + sigma * ((T)0.5 * (d21 + d12));
            np[r] = P[0][r] * P[0][r] + P[1][r] * P[1][r];
            nq[r] = Q[0][r] * Q[0][r] + Q[1][r] * Q[1][r] + (T)2 * Q[2][r] * Q[2][r];
        }
        tgv2d_ball<2>(P, np, k.alpha1, k.ra1, k.lim1, k.fast);
        tgv2d_ball<3>(Q, nq, k.alpha0, k.ra0, k.lim0, k.fast);
        dp2.put(p, b, P[1][R - 1]);
        dq22.put(p, b, Q[1][R - 1]);
        dq12.put(p, b, Q[2][R - 1]);
        __syncthreads();
        // above the image's first row zero, which makes the backward
        // difference the value itself (elsewhere group 0's is an edge)
        const T p2l = dp2.above(p, b), q22l = dq22.above(p, b), q12l = dq12.above(p, b);
        const T p2a = p.grp > 0 ? p2l : (T)0, q22a = p.grp > 0 ? q22l : (T)0, q12a = p.grp > 0 ? q12l : (T)0;
        T num[R], q1[R];
        uint32_t key = ~0u;
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const int ru = r > 0 ? r - 1 : 0;
            const T p1x = deep_left0(p, P[0][r]), q11x = deep_left0(p, Q[0][r]), q12x = deep_left0(p, Q[2][r]);
            const T p2y = r > 0 ? P[1][ru] : p2a, q22y = r > 0 ? Q[1][ru] : q22a, q12y = r > 0 ? Q[2][ru] : q12a;
            T px = P[0][r] - p1x, py = P[1][r] - p2y, q11 = Q[0][r] - q11x, q12d = Q[2][r] - q12y;
            T q12 = Q[2][r] - q12x, q22 = Q[1][r] - q22y;
            if (p.xedge) {
                deep_keep_branch();
                px = xneg ? -p1x : px;
                q11 = xneg ? -q11x : q11;
                q12 = xneg ? -q12x : q12;
            }
            if (p.yedge) {
                deep_keep_branch();
                const bool yn = p.y + r == p.ny - 1 && p.y + r > 0;
                py = yn ? -p2y : py;
                q12d = yn ? -q12y : q12d;
                q22 = yn ? -q22y : q22;
            }
            const T dv = px + py, dq1 = q11 + q12d, dq2 = q12 + q22;
            num[r] = k.lambda * (u[r] + tau * dv) + tau * f[r];
            const T w1 = v1[r] + tau * (P[0][r] + dq1), w2 = v2[r] + tau * (P[1][r] + dq2);
            v1[r] = through_storage<T, S>((T)2 * w1 - v1[r]);
            v2[r] = through_storage<T, S>((T)2 * w2 - v2[r]);
            // in (0, 2^-100), or not below 2^60 (the key of such a dividend is replaced by the smallest)
            key = min_key(key, fabsf(num[r]) < 0x1p+60f ? tiny_key(num[r]) : 0u);
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!k.fast || key < kTinyKey) != 0, 0)) {
            #pragma unroll
            for (int r = 0; r < R; ++r) q1[r] = num[r] / k.lt;
        } else {
            #pragma unroll
            for (int r = 0; r < R; ++r) q1[r] = div_in(num[r], k.lt, k.rlt);
        }
        double sd = 0.0, su = 0.0;
        const bool check = (a.check >> it) & 1u;
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            const T un = (T)2 * q1[r] - u[r];
            if (check && p.out(r)) {
                const T df = un - u[r];
                sd += (double)df * (double)df;
                su += (double)un * (double)un;
            }
            u[r] = un;
            if (!std::is_same<S, float>::value) {
                #pragma unroll
                for (int c = 0; c < 2; ++c) P[c][r] = through_storage<T, S>(P[c][r]);
                #pragma unroll
                for (int c = 0; c < 3; ++c) Q[c][r] = through_storage<T, S>(Q[c][r]);
            }
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
            if (a.write_state) {
                ((T*)a.out[0])[e] = u[r];
                stT<T>((S*)a.out[1], e, v1[r]);
                stT<T>((S*)a.out[2], e, v2[r]);
                stT<T>((S*)a.out[3], e, P[0][r]);
                stT<T>((S*)a.out[4], e, P[1][r]);
                stT<T>((S*)a.out[5], e, Q[0][r]);
                stT<T>((S*)a.out[6], e, Q[1][r]);
                stT<T>((S*)a.out[7], e, Q[2][r]);
            }
            if (a.write_res) a.res[e] = u[r];
        }
    deep_store_checks<Sh>(red, nchk, a.partials, a.g.nblocks, p.lin);
}

template <typename S>
struct TgvDeep : DeepMethod {
    using Args = TgvDeepArgs;
    static constexpr int NF = 8, rlo = 1, rhi = 1, words = 17;
    static constexpr DeepIterCost cost[kDeepShapeCount] = {{1.22, 1.65}, {1.90, 2.20}, {3.50, 4.90}, {2.20, 1.40}, {0.90, 0.18},
                                                              {1.10, 0.30}};
    static constexpr bool seeded = false;
    TgvPar par;
    size_t field_size(int i) const { return i == 0 ? sizeof(float) : sizeof(S); }
    void prepare(Args& a, int, int, bool) const { a.par = par; }
    template <class Sh>
    void launch(const Args& a, hipStream_t s) const {
        hipLaunchKernelGGL((tgv_deep_kernel<Sh, S>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
    }
    // caller state channels: u_bar, V1..3, P1..3, Q11, Q22, Q12
    static size_t channel(int i) { return i < 3 ? i : i < 5 ? i + 1 : i + 2; }
    void load(int i, void* dst, const WarmState& ws, size_t n, hipStream_t s) const {
        if (i == 0) state_in<float>((float*)dst, ws.d_state, n, s);
        else state_in<S>((S*)dst, ws.d_state + channel(i) * n, n, s);
    }
    void store(int i, const void* src, const WarmState& ws, size_t n, hipStream_t s) const {
        if (i == 0) state_out<float>(ws.d_state, (const float*)src, n, s);
        else state_out<S>(ws.d_state + channel(i) * n, (const S*)src, n, s);
    }
};

}  // namespace

template <typename S>
int tgv_solve_2d(const float* d_f, float* d_out, float lambda, float alpha1, float alpha0, int iter, float L2,
                 float epsil, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                 const WarmState* ws) {
    TgvDeep<S> m;
    TgvPar& k = m.par;
    k.lambda = lambda;
    k.tau = (float)pow((double)L2, -0.5);   // TGV_core.c:54-55
    k.alpha1 = alpha1;
    k.alpha0 = alpha0;
    k.lt = lambda + k.tau;
    auto in = [](float v) { return v >= 0x1p-30f && v <= 0x1p+30f; };
    k.fast = in(alpha1) && in(alpha0) && in(k.lt) && k.lt <= 0x1p+26f;   // quotients by lt stay normal
    k.ra1 = 1.0f / alpha1;
    k.ra0 = 1.0f / alpha0;
    k.rlt = 1.0f / k.lt;
    // |v| / alpha at most 2^23: the quotients of components from 2^-100 up stay normal
    k.lim1 = k.fast ? (0x1p+23f * alpha1) * (0x1p+23f * alpha1) : 0.0f;
    k.lim0 = k.fast ? (0x1p+23f * alpha0) * (0x1p+23f * alpha0) : 0.0f;
    return deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, ws);
}

template int tgv_solve_2d<float>(const float*, float*, float, float, float, int, float, float, int, int, const Opts&,
                                 hipStream_t, int*, float*, const WarmState*);
template int tgv_solve_2d<bf16_t>(const float*, float*, float, float, float, int, float, float, int, int, const Opts&,
                                  hipStream_t, int*, float*, const WarmState*);
template int tgv_solve_2d<_Float16>(const float*, float*, float, float, float, int, float, float, int, int,
                                    const Opts&, hipStream_t, int*, float*, const WarmState*);

}  // namespace cilreg
