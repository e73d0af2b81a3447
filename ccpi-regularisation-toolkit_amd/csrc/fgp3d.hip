// fgp3d.hip -- FGP-TV on a volume, several iterations per pass (the algorithm
// and its reference citations: top of fgp.hip; the passes: deep3d.hpp).
#include "solvers.hpp"
#include "deep3d.hpp"

namespace cilreg {

namespace {

struct Fgp3Par {
    float lambda, step, mult[kDeep3Max];   // mult[i]: of the pass's iteration i
    int nonneg;
    const float* B[3];     // FGP-dTV only
};
// state: P_k (3 components), P_{k-1} (3)
using Fgp3Args = Deep3Args<6, Fgp3Par>;

// v less its component along b (FGP_dTV_core.c:308-323)
__device__ inline void orthogonal(float& v1, float& v2, float& v3, const float (&b)[3]) {
    const float ip = v1 * b[0] + v2 * b[1] + v3 * b[2];
    v1 = v1 - ip * b[0];
    v2 = v2 - ip * b[1];
    v3 = v3 - ip * b[2];
}

// Per level and plane: R_i from the level's input (P_i, P_{i-1}), R2 of the
// group's last row to the group below, D_i from R_i and the carried R3 of the
// plane below, then P_{i+1} one plane behind from the carried R_i and D_i and
// from D_i here.  The next level's input is then complete: P_{i+1}, the carried
// P_i, f and D_i (for its check).  One barrier per level and plane; D_i of a
// group's first row, read by the group above one plane later, needs none.  The
// next plane's loads are issued a whole step ahead, and nothing else waits on
// memory.
//
// Bound by VALU issue, then by the traffic of overlapping regions: checked at
// 256^3 (T = 4, 64 x 16 columns) the VALU instructions fill 82% of the CUs' busy
// cycles at four each, and a launch reads 50 and writes 32 B per voxel at 3.1
// TB/s where it needs 32 and 28 (a region loads each point 2.3 times, most of it
// from L2, and the partial lines of two regions meet).  256^3 111 -> 86 us per
// iteration (bf16 91 -> 76, FP16 89 -> 74), 250^3 133 -> 80, 300^3 221 -> 129, 131 x
// 200 x 305 67 -> 43, 128^3 20.3 -> 16.0 (bf16 17.6 -> 16.6, FP16 17.4 -> 15.3), 100^3
// 14.3 -> 10.2 (before: two iterations per pass on 64 x 8 tiles, every stage
// through LDS).  T = 4 levels need 116-121 VGPRs: one 1024- or two 512-thread workgroups on a
// CU.  Also measured: a level two planes behind the one before (one barrier
// per plane for all levels, 15 instead of 8 values carried per row and level)
// 139 against 135 us at T = 2 and spills from T = 3 on; four rows per thread
// on 8 waves 104 us.
//
// DIR: FGP-dTV (top of dtv.hip).  R and the gradient of D are projected onto
// the plane orthogonal to the reference's normalised gradient B, which travels
// through the levels beside f; T = 3 fills the 128 VGPRs.  256^3 152 -> 120 us
// per iteration, 300^3 323 -> 189, 190 x 257 x 231 157 -> 74, 160^3 45 -> 29, 128^3
// 24.1 -> 19.4, 100^3 17.8 -> 13.0 (before: as for FGP).
template <class Sh, int T, typename S, bool ISO, bool CHK, bool DIR>
__global__ __launch_bounds__(64 * Sh::NW, 4) void fgp_deep3_kernel(Fgp3Args a) {
    if (solve_stopped(a.ctrl)) return;
    constexpr int R = Sh::R, G = Sh::G;
    const DeepPos3<Sh> p(a.g, xcd_logical_block((int)blockIdx.x, a.g.nblocks));
    __shared__ float rowR[2][G][64];          // R2 of a group's last row, exchange by exchange
    __shared__ float rowD[T][2][G][64];       // D_i of a group's first row, by step parity
    __shared__ double acc[CHK ? 2 * T : 1][CHK ? 64 * Sh::NW : 1];
    __shared__ DeepRed<Sh> red;
    const int tid = (int)threadIdx.x;
    if (CHK) {
        #pragma unroll
        for (int c = 0; c < 2 * T; ++c) acc[c][tid] = 0.0;
    }
    // carried from plane to plane, per level i (its last plane z_i): R_i, P_i, f, D_i
    float cr[T][R][3] = {}, cp[T][R][3] = {}, cf[T][R] = {}, cd[T][R] = {};
    float cb[DIR ? T : 1][R][3] = {}, lb[R][3];   // and B
    typename PlaneIn<S>::Word lp[R][3], lm[R][3];
    float lf[R], ld[R];   // level 0's next plane: P_k, P_{k-1}, f, D_{k-1}
    const bool xlast = p.x == p.nx - 1, nonneg = a.par.nonneg;
    const float lam = a.par.lambda, step = a.par.step;
    uint32_t off[R], so[R];
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        off[r] = 4u * (uint32_t)p.elem(r);
        so[r] = p.out(r) ? off[r] : kNoStore;
    }
    const int nz = p.nz, z0 = p.z0, z1 = p.z1;
    const int zs = z0 > T ? z0 - T : 0, ze = z1 + T - 1;

    auto load = [&](int z) {
        const size_t zo = plane_offset(z < nz ? z : nz - 1, p.sxy);
        const PlaneIn<float> pf(a.f + zo, true, p.sxy), pd(a.res + zo, CHK && (a.check & 1u), p.sxy);
        #pragma unroll
        for (int r = 0; r < R; ++r) {
            lf[r] = pf.ld(off[r]);
            ld[r] = CHK ? pd.ld(off[r]) : 0.0f;
        }
        if (DIR)
            #pragma unroll
            for (int c = 0; c < 3; ++c) {
                const PlaneIn<float> pb(a.par.B[c] + zo, true, p.sxy);
                #pragma unroll
                for (int r = 0; r < R; ++r) lb[r][c] = pb.ld(off[r]);
            }
        #pragma unroll
        for (int c = 0; c < 3; ++c) {
            const PlaneIn<S> pc((const S*)a.in[c] + zo, !a.cold, p.sxy), pm((const S*)a.in[3 + c] + zo, !a.cold, p.sxy);
            #pragma unroll
            for (int r = 0; r < R; ++r) {
                lp[r][c] = pc.word(off[r]);
                lm[r][c] = pm.word(off[r]);
            }
        }
    };
    load(zs);
    if (DIR)
        #pragma unroll
        for (int r = 0; r < R; ++r)
            #pragma unroll
            for (int c = 0; c < 3; ++c) landed(lb[r][c]);
    // the first plane's loads end here, so the loop's waits count its own
    #pragma unroll
    for (int r = 0; r < R; ++r) {
        landed(lf[r]);
        landed(ld[r]);
        #pragma unroll
        for (int c = 0; c < 3; ++c) {
            landed(lp[r][c]);
            landed(lm[r][c]);
        }
    }
    // one plane of every level per step, two steps per turn: what one carries on
    // lands in registers that the other has freed (T = 3 on 8 waves 4-6% faster;
    // deeper and checked passes would spill)
    constexpr int U = !CHK && T < (DIR ? 2 : 4) ? 2 : 1;
    for (int zu = zs, parity = 0; zu <= ze; zu += U, parity ^= U & 1) {
        #pragma unroll
        for (int h = 0; h < U; ++h) {
            const int zi = zu + h, b = U == 2 ? h : parity;
            if (h > 0 && zi > ze) break;
            float ip[R][3], im[R][3], fi[R], dp[R];   // the level's input: P_i, P_{i-1}, f, D_{i-1} at its plane
            #pragma unroll
            for (int r = 0; r < R; ++r) {
                fi[r] = lf[r];
                dp[r] = ld[r];
                #pragma unroll
                for (int c = 0; c < 3; ++c) {
                    ip[r][c] = PlaneIn<S>::value(lp[r][c]);
                    im[r][c] = PlaneIn<S>::value(lm[r][c]);
                }
            }
            float ib[R][3];
            if (DIR)
                #pragma unroll
                for (int r = 0; r < R; ++r)
                    #pragma unroll
                    for (int c = 0; c < 3; ++c) ib[r][c] = lb[r][c];
            load(zi + 1);
            #pragma unroll
            for (int i = 0; i < T; ++i) {
                const int zc = zi - i, zp = zc - 1, ex = (i + b * T) & 1;
                float rn[R][3], d[R];
                #pragma unroll
                for (int r = 0; r < R; ++r)
                    #pragma unroll
                    for (int c = 0; c < 3; ++c) rn[r][c] = ip[r][c] + a.par.mult[i] * (ip[r][c] - im[r][c]);
                if (DIR)
                    #pragma unroll
                    for (int r = 0; r < R; ++r) orthogonal(rn[r][0], rn[r][1], rn[r][2], ib[r]);
                rowR[ex][p.grp][p.lx] = rn[R - 1][1];
                __syncthreads();
                const float ab = rowR[ex][p.grp > 0 ? p.grp - 1 : 0][p.lx];
                const float above = p.grp > 0 ? ab : 0.0f;
                if (zc == 0) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) cr[i][r][2] = 0.0f;   // R3(-1) = 0
                }
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float b1 = deep_left(rn[r][0]), b2 = r > 0 ? rn[r > 0 ? r - 1 : 0][1] : above;
                    d[r] = fi[r] - lam * (rn[r][0] + rn[r][1] + rn[r][2] - b1 - b2 - cr[i][r][2]);
                }
                if (nonneg) {
                    #pragma unroll
                    for (int r = 0; r < R; ++r) d[r] = d[r] < 0.0f ? 0.0f : d[r];
                }
                rowD[i][b][p.grp][p.lx] = d[0];
                const bool inz = zc >= z0 && zc < z1;
                if (CHK && inz && ((a.check >> i) & 1u)) {
                    double sd = 0.0, su = 0.0;
                    #pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (p.out(r)) {
                            const float df = d[r] - dp[r];
                            sd += (double)df * (double)df;
                            su += (double)d[r] * (double)d[r];
                        }
                    acc[2 * i][tid] += sd;
                    acc[2 * i + 1][tid] += su;
                }
                if (i == T - 1) {
                    const PlaneOut<float> o(a.res + plane_offset(zc, p.sxy), inz && a.write_res, p.sxy);
                    #pragma unroll
                    for (int r = 0; r < R; ++r) o.st(so[r], d[r]);
                }
                // P_{i+1} at plane zc - 1
                const float dbl = rowD[i][b ^ 1][p.grp + 1 < G ? p.grp + 1 : p.grp][p.lx];
                float q1[R], q2[R], q3[R], g1[R], g2[R], g3[R];
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float dc = cd[i][r];
                    g1[r] = dc - deep_right(dc);
                    g2[r] = dc - (r + 1 < R ? cd[i][r + 1 < R ? r + 1 : r] : dbl);
                    g3[r] = dc - d[r];
                }
                if (p.xedge) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) g1[r] = xlast ? 0.0f : g1[r];
                }
                if (p.yedge) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) g2[r] = p.y + r == p.ny - 1 ? 0.0f : g2[r];
                }
                if (zp == nz - 1) {
                    deep_keep_branch();
                    #pragma unroll
                    for (int r = 0; r < R; ++r) g3[r] = 0.0f;
                }
                if (DIR)
                    #pragma unroll
                    for (int r = 0; r < R; ++r) orthogonal(g1[r], g2[r], g3[r], cb[DIR ? i : 0][r]);
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    q1[r] = cr[i][r][0] + step * g1[r];
                    q2[r] = cr[i][r][1] + step * g2[r];
                    q3[r] = cr[i][r][2] + step * g3[r];
                }
                project_unit_n<3, float, ISO>(q1, q2, q3);
                if (i == T - 1) {
                    const bool on = a.write_state && zp >= z0 && zp < z1;
                    const size_t zo = plane_offset(zp, p.sxy);
                    #pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const PlaneOut<S> pn((S*)a.out[c] + zo, on, p.sxy), pm((S*)a.out[3 + c] + zo, on, p.sxy);
                        #pragma unroll
                        for (int r = 0; r < R; ++r) {
                            pn.st(so[r], c == 0 ? q1[r] : c == 1 ? q2[r] : q3[r]);
                            pm.st_rounded(so[r], cp[i][r][c]);
                        }
                    }
                }
                // carry this plane; the next level takes P_{i+1}, P_i, f and D_i of plane zp
                #pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float o1 = cp[i][r][0], o2 = cp[i][r][1], o3 = cp[i][r][2], of = cf[i][r], od = cd[i][r];
                    #pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        cr[i][r][c] = rn[r][c];
                        cp[i][r][c] = ip[r][c];
                    }
                    cf[i][r] = fi[r];
                    cd[i][r] = d[r];
                    ip[r][0] = through_storage<float, S>(q1[r]);
                    ip[r][1] = through_storage<float, S>(q2[r]);
                    ip[r][2] = through_storage<float, S>(q3[r]);
                    im[r][0] = o1;
                    im[r][1] = o2;
                    im[r][2] = o3;
                    fi[r] = of;
                    dp[r] = od;
                    if (DIR)
                        #pragma unroll
                        for (int c = 0; c < 3; ++c) {
                            const float ob = cb[DIR ? i : 0][r][c];
                            cb[DIR ? i : 0][r][c] = ib[r][c];
                            ib[r][c] = ob;
                        }
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
constexpr Deep3Cost kFgp3Cost[kDeep3Shapes] = {
    {{1.9, 2.5, 3.15, 3.55}, {4.8, 4.8, 5.0, 4.9}},
    {{1.6, 2.15, 2.6, 3.1}, {4.4, 4.4, 4.5, 3.6}},
};
// with 16-bit P (conversions at every level)
constexpr Deep3Cost kFgp3Cost16[kDeep3Shapes] = {
    {{1.9, 2.5, 3.3, 4.1}, {3.5, 3.6, 4.0, 4.4}},
    {{1.7, 2.25, 2.85, 3.5}, {3.3, 3.3, 3.5, 3.6}},
};

// with B (no pass has four levels)
constexpr Deep3Cost kDtv3Cost[kDeep3Shapes] = {
    {{2.4, 3.2, 4.05}, {5.0, 5.0, 5.4}},
    {{2.1, 2.8, 3.25}, {4.6, 4.6, 4.8}},
};

template <typename S, bool DIR = false>
struct Fgp3 {
    using Args = Fgp3Args;
    static constexpr int NF = 6, rlo = 1, rhi = 1, max = DIR ? 3 : 4;
    static constexpr bool seeded = true;
    Fgp3Par par;
    bool iso;
    std::vector<float> mult;
    // dTV's three levels with checks spill (128^3 checked every iteration: 33 us, two
    // levels 26)
    int most(bool checked) const { return DIR && checked ? 2 : max; }
    size_t field_size(int) const { return sizeof(S); }
    const Deep3Cost (&cost() const)[kDeep3Shapes] {
        return DIR ? kDtv3Cost : sizeof(S) == 4 ? kFgp3Cost : kFgp3Cost16;
    }
    size_t bytes() const { return 12 * sizeof(S) + (DIR ? 16 : 4); }
    void prepare(Args& a, int k, int nk, bool) const {
        a.par = par;
        for (int i = 0; i < kDeep3Max; ++i) a.par.mult[i] = i < nk ? mult[k + i] : 0.0f;
    }
    template <int T>
    void go(int shape, const Args& a, hipStream_t s) const {
        deep3_dispatch(shape, [&](auto sh) {
            using Sh = decltype(sh);
            const dim3 grid(a.g.nblocks), block(64 * Sh::NW);
            if (a.check) {
                if (iso) hipLaunchKernelGGL((fgp_deep3_kernel<Sh, T, S, true, true, DIR>), grid, block, 0, s, a);
                else hipLaunchKernelGGL((fgp_deep3_kernel<Sh, T, S, false, true, DIR>), grid, block, 0, s, a);
            } else {
                if (iso) hipLaunchKernelGGL((fgp_deep3_kernel<Sh, T, S, true, false, DIR>), grid, block, 0, s, a);
                else hipLaunchKernelGGL((fgp_deep3_kernel<Sh, T, S, false, false, DIR>), grid, block, 0, s, a);
            }
        });
    }
    void launch(int T, int shape, const Args& a, hipStream_t s) const {
        switch (T) {
            case 1: go<1>(shape, a, s); break;
            case 2: go<2>(shape, a, s); break;
            case 3: go<3>(shape, a, s); break;
            default: go<max>(shape, a, s); break;
        }
    }
    // caller state channels: P1, P2, P3, then the previous P1, P2, P3
    void load(int i, void* dst, const WarmState& ws, size_t n, hipStream_t s) const {
        state_in<S>((S*)dst, ws.d_state + (size_t)i * n, n, s);
    }
    void store(int i, const void* src, const WarmState& ws, size_t n, hipStream_t s) const {
        state_out<S>(ws.d_state + (size_t)i * n, (const S*)src, n, s);
    }
};

}  // namespace

template <typename S>
int fgp_solve_3d(const float* d_f, float* d_out, float lambda, int iter, float epsil, int method, int nonneg, int nx,
                 int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws) {
    Fgp3<S> m;
    m.par.lambda = lambda;
    m.par.step = 1.0f / (12.0f * lambda);
    m.par.nonneg = nonneg != 0;
    for (const float*& b : m.par.B) b = nullptr;
    m.iso = method == 0;
    std::vector<float> tks;
    fgp_multipliers(iter, ws, m.mult, tks);
    int last = 0;
    if (deep3_solve(m, d_f, d_out, nx, ny, nz, iter, epsil, opts, s, iters_done, re, ws, &last) != 0) return -1;
    if (ws) {
        ws->tstate[0] = tks[last + 1];
        ws->tstate[1] = m.mult[last + 1];
    }
    return 0;
}

// FGP-dTV (arguments as dtv_solve_2d's).
int dtv_solve_3d(const float* d_f, const RefGrad& refgrad, float* d_out, float lambda, int iter, float epsil,
                 int method, int nonneg, int nx, int ny, int nz, const std::vector<float>& mult, const Opts& opts,
                 hipStream_t s, int* iters_done, float* re) {
    Fgp3<float, true> m;
    m.par.lambda = lambda;
    m.par.step = 1.0f / (26.0f * lambda);
    m.par.nonneg = nonneg != 0;
    m.iso = method == 0;
    m.mult = mult;
    const DeepExtra b{3, [&](float* const (&B)[3]) {
        for (int c = 0; c < 3; ++c) m.par.B[c] = B[c];
        refgrad(B);
    }};
    return deep3_solve(m, d_f, d_out, nx, ny, nz, iter, epsil, opts, s, iters_done, re, nullptr, nullptr, &b);
}

template int fgp_solve_3d<float>(const float*, float*, float, int, float, int, int, int, int, int, const Opts&,
                                 hipStream_t, int*, float*, const WarmState*);
template int fgp_solve_3d<bf16_t>(const float*, float*, float, int, float, int, int, int, int, int, const Opts&,
                                  hipStream_t, int*, float*, const WarmState*);
template int fgp_solve_3d<_Float16>(const float*, float*, float, int, float, int, int, int, int, int, const Opts&,
                                    hipStream_t, int*, float*, const WarmState*);

}  // namespace cilreg
