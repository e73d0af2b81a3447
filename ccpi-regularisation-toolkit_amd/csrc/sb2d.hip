// sb2d.hip -- SB-TV on a 2D image, many iterations per launch (the algorithm
// and its reference citations: top of sb.hip; the passes: deep2d.hpp).
#include "solvers.hpp"
#include "state.hpp"
#include "deep2d.hpp"

namespace cilreg {

namespace {

struct SbPar { float lam, mu, nc, thr; };   // as in SbArgs
// state: U, D (2 components), B (2)
using SbDeepArgs = DeepArgs<float, 5, SbPar>;

// The shrinkage of N points, d = shrink(v): in range (squared norm 0 or in
// [2^-90, 2^52], components 0 or from 2^-100 up, which keeps the quotients
// normal) by sqrt_in and div_in; a wave with any other point takes the
// reference's expressions.  Anisotropic: v / |v| is +-1 for finite v.
template <int N, bool ANISO>
__device__ inline void sb2d_shrink(const float (&v0)[N], const float (&v1)[N], float thr, float (&d0)[N],
                                   float (&d1)[N]) {
    bool odd = false;
    float w[N];
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        if (ANISO) {
            odd = odd || !(fabsf(v0[r]) < __builtin_inff()) || !(fabsf(v1[r]) < __builtin_inff());
        } else {
            w[r] = v0[r] * v0[r] + v1[r] * v1[r];
            odd = odd || !(w[r] <= 0x1p+52f) || (w[r] != 0.0f && w[r] < 0x1p-90f) ||
                  min_key(tiny_key(v0[r]), tiny_key(v1[r])) < kTinyKey;
        }
    }
    const bool slow = __builtin_amdgcn_ballot_w64(odd) != 0;
    if (ANISO) {
        #pragma unroll
        for (int r = 0; r < N; ++r) {
            float s0 = fabsf(v0[r]) - thr, s1 = fabsf(v1[r]) - thr;
            if (s0 < 0.0f) s0 = 0.0f;
            if (s1 < 0.0f) s1 = 0.0f;
            d0[r] = v0[r] != 0.0f ? __builtin_copysignf(s0, v0[r]) : 0.0f;
            d1[r] = v1[r] != 0.0f ? __builtin_copysignf(s1, v1[r]) : 0.0f;
            if (__builtin_expect(slow, 0)) {
                deep_keep_branch();
                d0[r] = v0[r] != 0.0f ? (v0[r] / fabsf(v0[r])) * s0 : 0.0f;
                d1[r] = v1[r] != 0.0f ? (v1[r] / fabsf(v1[r])) * s1 : 0.0f;
            }
        }
        return;
    }
    if (__builtin_expect(slow, 0)) {
        #pragma unroll
        for (int r = 0; r < N; ++r) {
            const float nrm = sqrtf(w[r]);
            float s = nrm - thr;
            if (s < 0.0f) s = 0.0f;
            d0[r] = nrm != 0.0f ? s * (v0[r] / nrm) : 0.0f;
            d1[r] = nrm != 0.0f ? s * (v1[r] / nrm) : 0.0f;
        }
        return;
    }
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        const float nrm = sqrt_in(__builtin_fmaxf(w[r], 0x1p-90f)), rn = rcp_in(nrm);
        float s = nrm - thr;
        if (s < 0.0f) s = 0.0f;
        d0[r] = w[r] != 0.0f ? s * div_in(v0[r], nrm, rn) : 0.0f;
        d1[r] = w[r] != 0.0f ? s * div_in(v1[r], nrm, rn) : 0.0f;
    }
}

// The mirrored neighbours of N points of one column: left, right, above and
// below (above / below: the rows of the neighbouring groups).
template <class Sh>
__device__ inline void sb2d_around(const DeepPos<Sh>& p, const float (&u)[Sh::R], float above, float below,
                                   float (&l)[Sh::R], float (&r)[Sh::R], float (&a)[Sh::R], float (&b)[Sh::R]) {
    constexpr int R = Sh::R;
    #pragma unroll
    for (int i = 0; i < R; ++i) {
        l[i] = deep_left(u[i]);
        r[i] = deep_right(u[i]);
        a[i] = i > 0 ? u[i > 0 ? i - 1 : 0] : above;
        b[i] = i + 1 < R ? u[i + 1 < R ? i + 1 : i] : below;
    }
    if (p.xedge) {
        deep_keep_branch();
        #pragma unroll
        for (int i = 0; i < R; ++i) {
            const float s = l[i], t = r[i];
            l[i] = p.x == 0 ? t : s;
            r[i] = p.x == p.nx - 1 ? s : t;
        }
    }
    if (p.yedge) {
        deep_keep_branch();
        #pragma unroll
        for (int i = 0; i < R; ++i) {
            const float s = a[i], t = b[i];
            a[i] = p.y + i == 0 ? t : s;
            b[i] = p.y + i == p.ny - 1 ? s : t;
        }
    }
}

// Registers per point: U, D, B, f.  Three exchanges an iteration: U0 (with D2
// and B2 of a group's last row), U1 and U2, each between row groups.
// Bound by VALU issue and the three barriers, above 1024^2 also by its 44 B
// per point and pass: 256^2 5.8 -> 2.1 us per iteration, 512^2 6.7 -> 3.3,
// 1024^2 20.7 -> 8.1, 2048^2 77 -> 25 (before: one fused launch per iteration).
template <class Sh, bool ANISO>
__global__ __launch_bounds__(64 * Sh::NW) void sb_deep_kernel(SbDeepArgs a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R;
    const DeepPos<Sh> p(a.g);
    __shared__ DeepRow<Sh> u0a, u0b, d2b, b2b, u1a, u1b, u2a, u2b;
    __shared__ DeepRed<Sh> red;

    float u[R], D1[R], D2[R], B1[R], B2[R], f[R];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t e = p.elem(r);
        f[r] = a.f[e];
        u[r] = f[r];
        D1[r] = D2[r] = B1[r] = B2[r] = 0.0f;
        if (!a.cold) {
            u[r] = ((const float*)a.in[0])[e];
            D1[r] = ((const float*)a.in[1])[e];
            D2[r] = ((const float*)a.in[2])[e];
            B1[r] = ((const float*)a.in[3])[e];
            B2[r] = ((const float*)a.in[4])[e];
        }
    }
    const float lam = a.par.lam, mu = a.par.mu, nc = a.par.nc;
    int nchk = 0;
    for (int it = 0; it < a.nit; ++it) {
        const int b = it & 1;
        float l[R], r[R], up[R], dn[R], db[R], u1[R], g1[R], g2[R];
        u0a.put(p, b, u[0]);
        u0b.put(p, b, u[R - 1]);
        d2b.put(p, b, D2[R - 1]);
        b2b.put(p, b, B2[R - 1]);
        __syncthreads();
        sb2d_around<Sh>(p, u, u0b.above(p, b), u0a.below(p, b), l, r, up, dn);
        // D and B at the mirrored x - 1 and y - 1
        float d1m[R], b1m[R], d2m[R], b2m[R];
        #pragma unroll
        for (int i = 0; i < R; ++i) {
            d1m[i] = deep_left(D1[i]);
            b1m[i] = deep_left(B1[i]);
            d2m[i] = i > 0 ? D2[i > 0 ? i - 1 : 0] : d2b.above(p, b);
            b2m[i] = i > 0 ? B2[i > 0 ? i - 1 : 0] : b2b.above(p, b);
        }
        if (p.xedge) {
            deep_keep_branch();
            #pragma unroll
            for (int i = 0; i < R; ++i) {
                const float s = deep_right(D1[i]), t = deep_right(B1[i]);
                d1m[i] = p.x == 0 ? s : d1m[i];
                b1m[i] = p.x == 0 ? t : b1m[i];
            }
        }
        if (p.yedge) {
            deep_keep_branch();
            const float s = R > 1 ? D2[R > 1 ? 1 : 0] : d2b.below(p, b), t = R > 1 ? B2[R > 1 ? 1 : 0] : b2b.below(p, b);
            d2m[0] = p.y == 0 ? s : d2m[0];
            b2m[0] = p.y == 0 ? t : b2m[0];
        }
        #pragma unroll
        for (int i = 0; i < R; ++i) {
            db[i] = d1m[i] - D1[i] + d2m[i] - D2[i] - b1m[i] + B1[i] - b2m[i] + B2[i];
            u1[i] = nc * ((db[i] + (r[i] + l[i] + dn[i] + up[i])) * lam + mu * f[i]);
        }
        u1a.put(p, b, u1[0]);
        u1b.put(p, b, u1[R - 1]);
        __syncthreads();
        sb2d_around<Sh>(p, u1, u1b.above(p, b), u1a.below(p, b), l, r, up, dn);
        #pragma unroll
        for (int i = 0; i < R; ++i) u[i] = nc * ((db[i] + (r[i] + l[i] + dn[i] + up[i])) * lam + mu * f[i]);
        u2a.put(p, b, u[0]);
        u2b.put(p, b, u[R - 1]);
        __syncthreads();
        sb2d_around<Sh>(p, u, u2b.above(p, b), u2a.below(p, b), l, r, up, dn);
        float v1[R], v2[R];
        #pragma unroll
        for (int i = 0; i < R; ++i) {
            g1[i] = r[i] - u[i];
            g2[i] = dn[i] - u[i];
            v1[i] = g1[i] + B1[i];
            v2[i] = g2[i] + B2[i];
        }
        sb2d_shrink<R, ANISO>(v1, v2, a.par.thr, D1, D2);
        #pragma unroll
        for (int i = 0; i < R; ++i) {
            B1[i] = B1[i] + (g1[i] - D1[i]);
            B2[i] = B2[i] + (g2[i] - D2[i]);
        }
        if ((a.check >> it) & 1u) {
            double sd = 0.0, su = 0.0;
            #pragma unroll
            for (int i = 0; i < R; ++i)
                if (p.out(i)) {
                    const float df = u[i] - u1[i];
                    sd += (double)df * (double)df;
                    su += (double)u[i] * (double)u[i];
                }
            deep_check<Sh>(red, sd, su, nchk);
            ++nchk;
        }
    }
    #pragma unroll
    for (int r = 0; r < R; ++r)
        if (p.out(r)) {
            const size_t e = p.elem(r);
            if (a.write_state) {
                ((float*)a.out[0])[e] = u[r];
                ((float*)a.out[1])[e] = D1[r];
                ((float*)a.out[2])[e] = D2[r];
                ((float*)a.out[3])[e] = B1[r];
                ((float*)a.out[4])[e] = B2[r];
            }
            if (a.write_res) a.res[e] = u[r];
        }
    deep_store_checks<Sh>(red, nchk, a.partials, a.g.nblocks, p.lin);
}

struct SbDeep : DeepMethod {
    using Args = SbDeepArgs;
    // two sweeps and a forward difference: two columns at low edges, three at high ones
    static constexpr int NF = 5, rlo = 2, rhi = 3, words = 11;
    static constexpr DeepIterCost cost[kDeepShapeCount] = {{1.0, 0.8}, {1.4, 1.4}, {2.2, 2.2}, {1.5, 1.1}, {0.8, 0.2},
                                                              {0.9, 0.3}};
    static constexpr bool seeded = false;
    SbPar par;
    bool aniso;
    size_t field_size(int) const { return sizeof(float); }
    void prepare(Args& a, int, int, bool) const { a.par = par; }
    template <class Sh>
    void launch(const Args& a, hipStream_t s) const {
        if (aniso) hipLaunchKernelGGL((sb_deep_kernel<Sh, true>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
        else hipLaunchKernelGGL((sb_deep_kernel<Sh, false>), dim3(a.g.nblocks), dim3(64 * Sh::NW), 0, s, a);
    }
    // caller state channels: U, D1, D2, D3, B1, B2, B3
    static size_t channel(int i) { return i < 3 ? i : 4 + (i - 3); }
    void load(int i, void* dst, const WarmState& ws, size_t n, hipStream_t s) const {
        state_in<float>((float*)dst, ws.d_state + channel(i) * n, n, s);
    }
    void store(int i, const void* src, const WarmState& ws, size_t n, hipStream_t s) const {
        state_out<float>(ws.d_state + channel(i) * n, (const float*)src, n, s);
    }
};

}  // namespace

int sb_solve_2d(const float* d_f, float* d_out, float lam, float mu, float nc, float thr, int iter, float epsil,
                int method, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                const WarmState* ws) {
    SbDeep m;
    m.par = SbPar{lam, mu, nc, thr};
    m.aniso = method == 1;
    return deep_solve(m, d_f, d_out, nx, ny, iter, epsil, opts, s, iters_done, re, ws);
}

}  // namespace cilreg
