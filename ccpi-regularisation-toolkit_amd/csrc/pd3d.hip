// pd3d.hip -- PD-TV on a volume, several iterations per pass (the algorithm
// and its reference citations: top of pd.hip; the passes: deep3d.hpp).
#include "solvers.hpp"
#include "deep3d.hpp"

namespace cilreg {

namespace {

struct Pd3Par {
    float sigma, tau, lt;
    double c, rlo, rhi;  // 1 + lt, bounds of its reciprocal
    int nonneg, plain;   // plain: the result is U before extrapolation (a stop), else u_bar
};
// state: u_bar, P (3 components)
using Pd3Args = Deep3Args<4, Pd3Par>;

// Per level and plane: u_bar of the level's plane closes the forward
// differences of the plane below it, whose new P follows; P2 of the group's
// last row goes to the group below (the level's one barrier) and the primal
// step gives u_bar of the next iteration, one plane behind.  u_bar of a
// group's first and last rows, read one plane later, needs no barrier.
//
// Bound by VALU issue and the barriers (a step of four levels takes 3.5 us on
// 16 waves whether its fields come from HBM or the last-level cache; about 115
// VALU instructions per level and wave; at 256^3 with T = 3 they fill 80% of the
// CUs' busy cycles, and a launch moves 46 B per voxel of the 36 it needs at 3.3
// TB/s); with T <= 2 and FP32 P, by HBM.  256^3 93 -> 73 us per iteration (bf16 90 ->
// 66, FP16 89 -> 65), 300^3 183 -> 106 (bf16 178 -> 95), 190 x 257 x 231 84 -> 47 (81 ->
// 40), 160^3 30 -> 20, 128^3 15.8 -> 15.3, 100^3 12.5 -> 10.3 (before: two iterations
// per pass on 64 x 8 tiles through LDS).
template <class Sh, int T, typename S, bool ISO, bool CHK>
__global__ __launch_bounds__(64 * Sh::NW, 4) void pd_deep3_kernel(Pd3Args a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R, G = Sh::G;
    const DeepPos3<Sh> p(a.g, xcd_logical_block((int)blockIdx.x, a.g.nblocks));
    __shared__ float rowQ[2][G][64];          // new P2 of a group's last row, exchange by exchange
    __shared__ float rowU[T][2][2][G][64];    // u_bar of its first and last row, by step parity
    __shared__ double acc[CHK ? 2 * T : 1][CHK ? 64 * Sh::NW : 1];
    __shared__ DeepRed<Sh> red;
    const int tid = (int)threadIdx.x;
    if (CHK) {
        #pragma unroll
        for (int c = 0; c < 2 * T; ++c) acc[c][tid] = 0.0;
    }
    // carried, per level, of its last plane: u_bar, P, f; of the plane before: u_bar, the new P3
    float cu[T][R] = {}, cp[T][R][3] = {}, cf[T][R] = {}, bu[T][R] = {}, bq[T][R] = {};
    typename PlaneIn<S>::Word lp[R][3];
    float lu[R], lf[R];   // level 0's next plane
    const bool xlast = p.x == p.nx - 1, nonneg = a.par.nonneg;
    const float sigma = a.par.sigma, tau = a.par.tau, lt = a.par.lt;
    uint32_t off[R], so[R];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        off[r] = 4u * (uint32_t)p.elem(r);
        so[r] = p.out(r) ? off[r] : kNoStore;
    }
    const int nz = p.nz, z0 = p.z0, z1 = p.z1;
    const int zs = z0 > T ? z0 - T : 0, ze = z1 + T - 1;
    const float* u_in = a.cold ? a.f : (const float*)a.in[0];   // u_bar = f at the start

    auto load = [&](int z) {
        const size_t zo = plane_offset(z < nz ? z : nz - 1, p.sxy);
        const PlaneIn<float> pu(u_in + zo, true, p.sxy), pf(a.f + zo, true, p.sxy);
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            lu[r] = pu.ld(off[r]);
            lf[r] = pf.ld(off[r]);
        }
        #pragma unroll
        for (int c = 0; c < 3; ++c) {
            const PlaneIn<S> pp((const S*)a.in[1 + c] + zo, !a.cold, p.sxy);
            #pragma unroll
            for (int r = 0; r < R; ++r) lp[r][c] = pp.word(off[r]);
        }
    };
    load(zs);
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        landed(lu[r]);
        landed(lf[r]);
        #pragma unroll
        for (int c = 0; c < 3; ++c) landed(lp[r][c]);
    }
    // one plane of every level per step, two steps per turn: what one carries on
    // lands in registers that the other has freed (T = 3 on 8 waves 4-6% faster;
    // deeper and checked passes would spill)
    constexpr int U = !CHK && T < 4 ? 2 : 1;
    for (int zu = zs, parity = 0; zu <= ze; zu += U, parity ^= U & 1) {
        #pragma unroll
        for (int h = 0; h < U; ++h) {
            const int zi = zu + h, b = U == 2 ? h : parity;
            if (h > 0 && zi > ze) break;
            float iu[R], ip[R][3], fi[R];   // the level's input at its plane: u_bar, P, f
            #pragma unroll
            for (int r = 0; r < R; ++r) {
                iu[r] = lu[r];
                fi[r] = lf[r];
                #pragma unroll
                for (int c = 0; c < 3; ++c) ip[r][c] = PlaneIn<S>::value(lp[r][c]);
            }
            load(zi + 1);
            #pragma unroll
            for (int i = 0; i < T; ++i) {
                const int zc = zi - i, zp = zc - 1, ex = (i + b * T) & 1;
                rowU[i][b][0][p.grp][p.lx] = iu[0];
                rowU[i][b][1][p.grp][p.lx] = iu[R - 1];
                // the dual step at plane zp
                const float ubl = rowU[i][b ^ 1][0][p.grp + 1 < G ? p.grp + 1 : p.grp][p.lx];
                float q1[R], q2[R], q3[R], ux[R], uy[R], uz[R];
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    ux[r] = deep_right(cu[i][r]);
                    uy[r] = r + 1 < R ? cu[i][r + 1 < R ? r + 1 : r] : ubl;
                    uz[r] = iu[r];
                }
                if (p.xedge) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float l = deep_left(cu[i][r]);
                        ux[r] = xlast ? l : ux[r];
                    }
                }
                if (p.yedge) {
                    deep_keep_branch();
                    const float uab = rowU[i][b ^ 1][1][p.grp > 0 ? p.grp - 1 : 0][p.lx];
                    #pragma unroll
                    for (int r = 0; r < R; ++r)
                        uy[r] = p.y + r == p.ny - 1 ? (r > 0 ? cu[i][r > 0 ? r - 1 : 0] : uab) : uy[r];
                }
                if (zp == nz - 1) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) uz[r] = bu[i][r];
                }
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    q1[r] = cp[i][r][0] + sigma * (ux[r] - cu[i][r]);
                    q2[r] = cp[i][r][1] + sigma * (uy[r] - cu[i][r]);
                    q3[r] = cp[i][r][2] + sigma * (uz[r] - cu[i][r]);
                }
                project_unit_n<3, float, ISO>(q1, q2, q3);
                rowQ[ex][p.grp][p.lx] = q2[R - 1];
                __syncthreads();
                const float qab = rowQ[ex][p.grp > 0 ? p.grp - 1 : 0][p.lx];
                const float above = p.grp > 0 ? qab : 0.0f;   // P2(-1) = 0 at the first row
                if (zp == 0) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) bq[i][r] = 0.0f;   // P3(-1) = 0
                }
                // the primal step at plane zp; -(q - 0) is -q
                float u0[R], un[R];
                #pragma unroll
                for (int r = 0; r < R; ++r) u0[r] = cu[i][r];
                if (nonneg) {
                    #pragma unroll
                    for (int r = 0; r < R; ++r) u0[r] = u0[r] < 0.0f ? 0.0f : u0[r];
                }
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float v1 = -(q1[r] - deep_left(q1[r])), v2 = -(q2[r] - (r > 0 ? q2[r > 0 ? r - 1 : 0] : above));
                    const float v3 = -(q3[r] - bq[i][r]);
                    const float dv = v1 + v2 + v3;
                    un[r] = u0[r] - tau * dv + lt * cf[i][r];
                }
                Mixed<float>::pd_div_n(un, a.par.c, a.par.rlo, a.par.rhi);
                const bool inz = zp >= z0 && zp < z1;
                if (CHK && inz && ((a.check >> i) & 1u)) {
                    double sd = 0.0, su = 0.0;
                    #pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (p.out(r)) {
                            const float df = un[r] - u0[r];
                            sd += (double)df * (double)df;
                            su += (double)un[r] * (double)un[r];
                        }
                    acc[2 * i][tid] += sd;
                    acc[2 * i + 1][tid] += su;
                }
                if (i == T - 1) {
                    const size_t zo = plane_offset(zp, p.sxy);
                    const PlaneOut<float> pr(a.res + zo, inz && a.write_res, p.sxy);
                    const PlaneOut<float> pu((float*)a.out[0] + zo, inz && a.write_state, p.sxy);
                    #pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float v = un[r] + (un[r] - u0[r]);
                        pu.st(so[r], v);
                        pr.st(so[r], a.par.plain ? un[r] : v);
                    }
                    #pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const PlaneOut<S> pp((S*)a.out[1 + c] + zo, inz && a.write_state, p.sxy);
                        #pragma unroll
                        for (int r = 0; r < R; ++r) pp.st(so[r], c == 0 ? q1[r] : c == 1 ? q2[r] : q3[r]);
                    }
                }
                if (zc == nz - 1) {   // the last plane's forward difference reads the plane below it
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) bu[i][r] = cu[i][r];
                }
                // carry this plane; the next level takes u_bar, P and f of plane zp
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float of = cf[i][r];
                    bq[i][r] = q3[r];
                    cu[i][r] = iu[r];
                    cf[i][r] = fi[r];
                    #pragma unroll
                    for (int c = 0; c < 3; ++c) cp[i][r][c] = ip[r][c];
                    iu[r] = un[r] + (un[r] - u0[r]);
                    ip[r][0] = through_storage<float, S>(q1[r]);
                    ip[r][1] = through_storage<float, S>(q2[r]);
                    ip[r][2] = through_storage<float, S>(q3[r]);
                    fi[r] = of;
                }
            }
        }
    }
    if (CHK) {
        int n = 0;
        #pragma unroll
        for (int i = 0; i < T; ++i)
            if ((a.check >> i) & 1u) {
                deep_check<Sh>(red, acc[2 * i][tid], acc[2 * i + 1][tid], n);
                ++n;
            }
        deep_store_checks<Sh>(red, n, a.partials, a.g.nblocks, p.lin);
    }
}

// A step's time (one plane of every level, microseconds) with T = 1..4 levels:
// when the fields stay in the last-level cache, and when they stream from HBM.
constexpr Deep3Cost kPd3Cost[kDeep3Shapes] = {
    {{1.55, 2.2, 2.9, 3.5}, {3.2, 3.35, 3.75, 4.15}},
    {{1.3, 1.95, 2.55, 3.15}, {3.4, 2.85, 2.75, 3.2}},
};
// with 16-bit P
constexpr Deep3Cost kPd3Cost16[kDeep3Shapes] = {
    {{1.55, 2.25, 3.0, 3.7}, {2.1, 2.5, 3.2, 4.0}},
    {{1.3, 2.1, 2.75, 3.4}, {2.3, 2.15, 2.75, 3.4}},
};

template <typename S>
struct Pd3 {
    using Args = Pd3Args;
    static constexpr int NF = 4, rlo = 1, rhi = 1, max = 4;
    static constexpr bool seeded = false;
    Pd3Par par;
    bool iso;
    int most(bool) const { return max; }
    size_t field_size(int i) const { return i == 0 ? sizeof(float) : sizeof(S); }
    const Deep3Cost (&cost() const)[kDeep3Shapes] { return sizeof(S) == 4 ? kPd3Cost : kPd3Cost16; }
    size_t bytes() const { return 6 * sizeof(S) + 12; }
    void prepare(Args& a, int, int, bool stop) const {
        a.par = par;
        a.par.plain = stop;
    }
    template <int T>
    void go(int shape, const Args& a, hipStream_t s) const {
        deep3_dispatch(shape, [&](auto sh) {
            using Sh = decltype(sh);
            const dim3 grid(a.g.nblocks), block(64 * Sh::NW);
            if (a.check) {
                if (iso) hipLaunchKernelGGL((pd_deep3_kernel<Sh, T, S, true, true>), grid, block, 0, s, a);
                else hipLaunchKernelGGL((pd_deep3_kernel<Sh, T, S, false, true>), grid, block, 0, s, a);
            } else {
                if (iso) hipLaunchKernelGGL((pd_deep3_kernel<Sh, T, S, true, false>), grid, block, 0, s, a);
                else hipLaunchKernelGGL((pd_deep3_kernel<Sh, T, S, false, false>), grid, block, 0, s, a);
            }
        });
    }
    void launch(int T, int shape, const Args& a, hipStream_t s) const {
        switch (T) {
            case 1: go<1>(shape, a, s); break;
            case 2: go<2>(shape, a, s); break;
            case 3: go<3>(shape, a, s); break;
            default: go<4>(shape, a, s); break;
        }
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
int pd_solve_3d(const float* d_f, float* d_out, float lambda, int iter, float epsil, float lipschitz, int method,
                int nonneg, int nx, int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                const WarmState* ws) {
    Pd3<S> m;
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
    return deep3_solve(m, d_f, d_out, nx, ny, nz, iter, epsil, opts, s, iters_done, re, ws);
}

template int pd_solve_3d<float>(const float*, float*, float, int, float, float, int, int, int, int, int, const Opts&,
                                hipStream_t, int*, float*, const WarmState*);
template int pd_solve_3d<bf16_t>(const float*, float*, float, int, float, float, int, int, int, int, int, const Opts&,
                                 hipStream_t, int*, float*, const WarmState*);
template int pd_solve_3d<_Float16>(const float*, float*, float, int, float, float, int, int, int, int, int,
                                   const Opts&, hipStream_t, int*, float*, const WarmState*);

}  // namespace cilreg
