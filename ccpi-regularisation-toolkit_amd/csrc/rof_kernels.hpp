// rof_kernels.hpp -- device code of the ROF iteration: argument block,
// per-tile body and the single-volume kernel.  The body is shared by the
// single-volume kernel (rof.hip) and the grouped multi-volume kernel
// (batch.hip); the algorithm and its reference citations are described at the
// top of rof.hip.
#pragma once
#include "runtime.hpp"

namespace cilreg {

template <typename T>
struct RofArgs {
    const T* f;
    const T* U;
    T* Uout;
    T lambda, tau;
    int check;
    double* partials;
    const Ctrl* ctrl;
    Geom g;
};

__device__ inline int mirror_p(int i, int n) { return i + 1 >= n ? (i - 1 >= 0 ? i - 1 : 0) : i + 1; }
__device__ inline int mirror_m(int i, int n) { return i - 1 < 0 ? (i + 1 < n ? i + 1 : 0) : i - 1; }

// The flux D1 (along y) from the forward difference fj and the squared
// minmods across x (mi) and, in 3D, z (mk): ROF_TV_core.c:131-137 (3D, double
// sqrt), :157-161 (2D).  eps is the floor added in double under the square
// root: 1e-8 for ROF-TV, 1e-12 for the ROF part of LLT-ROF
// (LLT_ROF_core.c:22,198-363).
template <int DIM, typename T>
__device__ inline T rof_d1(T fj, T mi, T mk, double eps) {
    if (DIM == 3) return fj / Mixed<T>::rof_sqrt_d(fj * fj + mi + mk, eps);
    return fj / Mixed<T>::rof_sqrt_f(fj * fj + mi, eps);
}

// The flux D2 (along x): ROF_TV_core.c:194-200 (3D), :220-224 (2D).
template <int DIM, typename T>
__device__ inline T rof_d2(T fi, T mj, T mk, double eps) {
    if (DIM == 3) return fi / Mixed<T>::rof_sqrt_f(fi * fi + mj + mk, eps);
    return fi / Mixed<T>::rof_sqrt_f(fi * fi + mj, eps);
}

// The fluxes D1, D2 and, in 3D, D3 (along z, ROF_TV_core.c:257-263) at a
// point from u there (uc) and at its mirrored neighbours, as the reference
// writes them.
template <int DIM, typename T>
__device__ inline void rof_flux_ref(T uc, T uip, T uim, T ujp, T ujm, T ukp, T ukm, T& d1, T& d2, T& d3,
                                    double eps) {
    const T fi = uip - uc, bi = uc - uim, fj = ujp - uc, bj = uc - ujm;
    if (DIM == 3) {
        const T fk = ukp - uc, bk = uc - ukm;
        T m[3];
        Mixed<T>::minmod_sq_n({fi, fj, fk}, {bi, bj, bk}, m);
        const T mi = m[0], mj = m[1], mk = m[2];
        d1 = rof_d1<DIM, T>(fj, mi, mk, eps);
        d2 = rof_d2<DIM, T>(fi, mj, mk, eps);
        d3 = fk / Mixed<T>::rof_sqrt_f(fk * fk + mj + mi, eps);
    } else {
        T m[2];
        Mixed<T>::minmod_sq_n({fi, fj}, {bi, bj}, m);
        d1 = rof_d1<DIM, T>(fj, m[0], T(0), eps);
        d2 = rof_d2<DIM, T>(fi, m[1], T(0), eps);
        d3 = 0;
    }
}

// sq: a sum of squares; prod: a sum of products.  True when sq is not below 2^52
// or either is NaN or infinite (|prod| adds at most 2^48 otherwise).
__device__ inline bool rof_odd(float prod, float sq) {
    return !(__builtin_fmaf(fabsf(prod), 0x1p-80f, sq) < 0x1p+52f);
}

// The same values.  In-range points take sqrt_in and div_in; one test sends a
// wave with any other point to rof_flux_ref: sums of squares not below 2^52
// (with numerators from 2^-100 up every quotient is then a normal number), a
// product of a minmod's operands that is NaN or infinite, or a numerator in
// (0, 2^-100).  Each quotient issues in 26 cycles instead of 49, and the minmods
// need no test of their own (ROF 256^3 84 -> 80 us per iteration, 128^3 13.8 ->
// 12.7).
template <int DIM, typename T>
__device__ inline void rof_flux_math(T uc, T uip, T uim, T ujp, T ujm, T ukp, T ukm, T& d1, T& d2, T& d3,
                                     double eps = 1.0e-8) {
    if constexpr (std::is_same<T, float>::value) {
        const float fi = uip - uc, bi = uc - uim, fj = ujp - uc, bj = uc - ujm;
        const float ai = __builtin_amdgcn_fmed3f(fi, bi, 0.f), aj = __builtin_amdgcn_fmed3f(fj, bj, 0.f);
        const float mi = ai * ai, mj = aj * aj;
        float s1 = fj * fj + mi, s2 = fi * fi + mj, s3 = 0.f, fk = 0.f, prod = __builtin_fmaf(fi, bi, fj * bj);
        uint32_t key = min_key(tiny_key(fi), tiny_key(fj));
        if (DIM == 3) {
            fk = ukp - uc;
            const float bk = uc - ukm, ak = __builtin_amdgcn_fmed3f(fk, bk, 0.f), mk = ak * ak;
            s1 = s1 + mk;
            s2 = s2 + mk;
            s3 = fk * fk + mj + mi;
            prod = __builtin_fmaf(fk, bk, prod);
            key = min_key(key, tiny_key(fk));
        }
        const bool odd = rof_odd(prod, s1 + s2 + s3) || key < kTinyKey;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd) == 0, 1)) {
            const double x1 = (double)s1 + eps;
            const float b1 = DIM == 3 ? (float)sqrt_dn(x1) : sqrt_in((float)x1);
            const float b2 = sqrt_in((float)((double)s2 + eps));
            d1 = div_in(fj, b1, rcp_in(b1));
            d2 = div_in(fi, b2, rcp_in(b2));
            d3 = 0;
            if (DIM == 3) {
                const float b3 = sqrt_in((float)((double)s3 + eps));
                d3 = div_in(fk, b3, rcp_in(b3));
            }
            return;
        }
    }
    rof_flux_ref<DIM, T>(uc, uip, uim, ujp, ujm, ukp, ukm, d1, d2, d3, eps);
}

// A ring lane's D2 (side) or D1, from the forward difference f along its axis,
// those across it (fo, bo) and along z: in range as in rof_flux_math.
template <int DIM>
__device__ inline float rof_ring_flux(bool side, float f, float fo, float bo, float fk, float bk, double eps) {
    const float ao = __builtin_amdgcn_fmed3f(fo, bo, 0.f), ak = __builtin_amdgcn_fmed3f(fk, bk, 0.f);
    const float mo = ao * ao, mk = ak * ak, s = DIM == 3 ? f * f + mo + mk : f * f + mo;
    const bool odd = rof_odd(__builtin_fmaf(fo, bo, fk * bk), s) || tiny_key(f) < kTinyKey;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd) == 0, 1)) {
        const double x = (double)s + eps;
        float w = sqrt_in((float)x);
        if (DIM == 3) {
            const float w1 = (float)sqrt_dn(x);   // D1's root is rounded from double
            w = side ? w : w1;
        }
        return div_in(f, w, rcp_in(w));
    }
    const float no = Mixed<float>::minmod_sq(fo, bo), nk = DIM == 3 ? Mixed<float>::minmod_sq(fk, bk) : 0.f;
    return side ? rof_d2<DIM, float>(f, no, nk, eps) : rof_d1<DIM, float>(f, no, nk, eps);
}

// The fluxes D1 (along y), D2 (along x) and, in 3D, D3 (along z) at
// (px, py, z) from one load of the 7-point mirrored neighbourhood.
template <int DIM, typename I, typename T>
__device__ inline void rof_fluxes(const RofArgs<T>& a, int px, int py, int z, T& d1, T& d2, T& d3) {
    const Geom& g = a.g;
    const I sxy = (I)g.sxy, nx = (I)g.nx;
    const I zo = (I)z * sxy, c = zo + (I)py * nx + (I)px;
    const T uc = ldx<T>(a.U, c);
    const T uip = ldx<T>(a.U, zo + (I)py * nx + (I)mirror_p(px, g.nx));
    const T uim = ldx<T>(a.U, zo + (I)py * nx + (I)mirror_m(px, g.nx));
    const T ujp = ldx<T>(a.U, zo + (I)mirror_p(py, g.ny) * nx + (I)px);
    const T ujm = ldx<T>(a.U, zo + (I)mirror_m(py, g.ny) * nx + (I)px);
    T ukp = 0, ukm = 0;
    if (DIM == 3) {
        ukp = ldx<T>(a.U, (I)mirror_p(z, g.nz) * sxy + (I)py * nx + (I)px);
        ukm = ldx<T>(a.U, (I)mirror_m(z, g.nz) * sxy + (I)py * nx + (I)px);
    }
    rof_flux_math<DIM, T>(uc, uip, uim, ujp, ujm, ukp, ukm, d1, d2, d3);
}

template <int DIM, int TY, typename T, typename I>
__device__ inline void rof_body(const RofArgs<T>& a, const TileCoord& tc) {
    const Geom& g = a.g;
    constexpr int NT = TX * TY;
    // U plane ring: rows y0-1 and y0+TY on [x0-1, x0+64] (corners included),
    // columns x0-1 and x0+64 on the tile's rows
    constexpr int NR = 2 * (TX + 2) + 2 * TY;
    static_assert(NR <= NT, "ring lanes must fit the workgroup");
    const int lx = threadIdx.x, ly = threadIdx.y, tid = ly * TX + lx;
    const int x = tc.x0 + lx, y = tc.y0 + ly;
    const bool own = x < g.nx && y < g.ny;
    const int ox = own ? x : 0, oy = own ? y : 0;
    // ring lane: one point of the U ring, on the low or high waves by block index
    const int hbase = (tc.lin & 1) ? NT - NR : 0;
    const int h = tid - hbase;
    const bool rlane = h >= 0 && h < NR;
    int sx, sy;   // ring slot in the (TY+2) x (TX+2) plane with origin (x0-1, y0-1)
    if (h < TX + 2) { sx = h; sy = 0; }
    else if (h < 2 * (TX + 2)) { sx = h - (TX + 2); sy = TY + 1; }
    else if (h < 2 * (TX + 2) + TY) { sx = 0; sy = 1 + h - 2 * (TX + 2); }
    else { sx = TX + 1; sy = 1 + h - 2 * (TX + 2) - TY; }
    const int rx = tc.x0 + sx - 1, ry = tc.y0 + sy - 1;
    const bool rin = rlane && rx >= 0 && ry >= 0 && rx < g.nx && ry < g.ny;
    const int rcx = rin ? rx : 0, rcy = rin ? ry : 0;   // clamped stand-in
    // ring lanes that also evaluate a flux: D1 on row y0-1 over x0..x0+63 and
    // D2 on column x0-1 over the tile's rows
    const bool d1lane = rlane && sy == 0 && sx >= 1 && sx <= TX;
    const bool d2lane = rlane && sx == 0 && sy >= 1 && sy <= TY;

    __shared__ T Us[TY + 2][TX + 2];    // U of plane z: tile and ring
    __shared__ T D1l[TY + 1][TX];       // [ly + 1][lx]; row 0 = y0 - 1
    __shared__ T D2l[TY][TX + 1];       // [ly][lx + 1]; column 0 = x0 - 1
    __shared__ double red[kRedSlots];
    const I sxy = (I)g.sxy, nx = (I)g.nx;

    // mirrored neighbour slots (loop-invariant) of the own point; threads
    // outside the volume read their own slot (their results are not stored)
    const int oxp = own ? mirror_p(x, g.nx) - tc.x0 + 1 : lx + 1, oxm = own ? mirror_m(x, g.nx) - tc.x0 + 1 : lx + 1;
    const int oyp = own ? mirror_p(y, g.ny) - tc.y0 + 1 : ly + 1, oym = own ? mirror_m(y, g.ny) - tc.y0 + 1 : ly + 1;
    // flux lanes: the neighbours a D1 on row y0-1 / a D2 on column x0-1 reads
    const int rxp = mirror_p(rcx, g.nx) - tc.x0 + 1, rxm = mirror_m(rcx, g.nx) - tc.x0 + 1;
    const int ryp = mirror_p(rcy, g.ny) - tc.y0 + 1, rym = mirror_m(rcy, g.ny) - tc.y0 + 1;

    const I ocol = (I)oy * nx + (I)ox, rcol = (I)rcy * nx + (I)rcx;
    // z pipeline of the own column and of the ring point
    T uc = ldx<T>(a.U, (I)tc.z0 * sxy + ocol), um = 0;
    T hc = 0, hm = 0;
    if (rlane) hc = ldx<T>(a.U, (I)tc.z0 * sxy + rcol);
    // D3 at the mirrored z-predecessor of the chunk's first plane
    T d3m = 0;
    if (DIM == 3) {
        const int zm = mirror_m(tc.z0, g.nz);
        um = ldx<T>(a.U, (I)zm * sxy + ocol);
        if (rlane) hm = ldx<T>(a.U, (I)zm * sxy + rcol);
        if (g.nz > 1) {
            T t1, t2;
            rof_fluxes<DIM, I>(a, ox, oy, zm, t1, t2, d3m);
        }
    }
    double sdd = 0.0, suu = 0.0;
    for (int z = tc.z0; z < tc.z1; ++z) {
        T up = 0, hp = 0;
        if (DIM == 3) {
            const int zp = mirror_p(z, g.nz);
            up = (zp == z + 1) ? ldx<T>(a.U, (I)zp * sxy + ocol) : um;
            if (rlane) hp = (zp == z + 1) ? ldx<T>(a.U, (I)zp * sxy + rcol) : hm;
        }
        Us[ly + 1][lx + 1] = uc;
        if (rlane) Us[sy][sx] = hc;
        __syncthreads();
        // fluxes of the own point
        T d1, d2, d3;
        rof_flux_math<DIM, T>(uc, Us[ly + 1][oxp], Us[ly + 1][oxm], Us[oyp][lx + 1], Us[oym][lx + 1], up, um, d1, d2,
                              d3);
        D1l[ly + 1][lx] = d1;
        D2l[ly][lx + 1] = d2;
        if (d1lane || d2lane) {
            // the neighbour outside the ring (y0-2 for D1, x0-2 for D2) feeds
            // only the other fluxes; it is replaced by the point itself
            const T uxp = Us[sy][rxp >= 0 && rxp < TX + 2 ? rxp : sx];
            const T uxm = Us[sy][rxm >= 0 && rxm < TX + 2 ? rxm : sx];
            const T uyp = Us[ryp >= 0 && ryp < TY + 2 ? ryp : sy][sx];
            const T uym = Us[rym >= 0 && rym < TY + 2 ? rym : sy][sx];
            // only the flux the lane stores: D2 on the column, D1 on the row
            // (the across-difference pair: y for D2, x for D1)
            const T fa = d2lane ? uyp - hc : uxp - hc, ba = d2lane ? hc - uym : hc - uxm;
            const T q = rof_ring_flux<DIM>(d2lane, (d2lane ? uxp : uyp) - hc, fa, ba, DIM == 3 ? hp - hc : T(0),
                                           DIM == 3 ? hc - hm : T(0), 1.0e-8);
            if (rin) {
                if (d2lane) D2l[sy - 1][0] = q;
                else D1l[0][sx - 1] = q;
            }
        }
        __syncthreads();
        if (own) {
            const I i = (I)z * sxy + ocol;
            const T dv1 = d1 - D1l[oym][lx];
            const T dv2 = d2 - D2l[ly][oxm];
            T dv = dv1 + dv2;
            if (DIM == 3) {
                // at z = 0 the mirrored predecessor is plane 1 (d3m from the prologue)
                dv = dv + (d3 - d3m);
            }
            const T un = uc + a.tau * (a.lambda * dv - (uc - ldx<T>(a.f, i)));
            if (a.check) {
                const T df = un - uc;
                sdd += (double)df * (double)df;
                suu += (double)un * (double)un;
            }
            stnt<T>(a.Uout, i, un);
        }
        d3m = d3;
        um = uc;
        uc = up;
        hm = hc;
        hc = hp;
    }
    if (a.check) {
        block_sum2(sdd, suu, red);
        if (tid == 0) {
            a.partials[2 * tc.lin] = sdd;
            a.partials[2 * tc.lin + 1] = suu;
        }
    }
}

// One iteration on one volume: the workgroup's tile comes from its block index.
template <int DIM, int TY, typename T, typename I>
__global__ __launch_bounds__(TX * TY) void rof_iter_kernel(RofArgs<T> a) {
    if (solve_stopped(a.ctrl)) return;
    rof_body<DIM, TY, T, I>(a, tile_of_block(a.g, TY));
}

}  // namespace cilreg
