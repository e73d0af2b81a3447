// deep3d.hpp -- several iterations per pass over a volume: a workgroup owns a
// column of 64 x H points, marches it through a chunk of z planes and keeps
// every iteration's plane-to-plane state in registers.
//
// Each thread holds R vertically adjacent points of one column of the region
// (as in the 2D passes): values move along x by lane shifts, along y as
// registers and through one LDS row per row group, along z as registers
// carried from plane to plane.  Level i of the pass (iteration k + i) works one
// plane behind level i - 1, whose result it takes from registers, so a pass of
// T iterations reads the input state and writes the output state once; it
// loses `lo` / `hi` columns and rows per iteration at the region's inner edges
// and repeats T planes at either end of its chunk.
#pragma once
#include "deep2d.hpp"
#include <algorithm>

namespace cilreg {

struct Deep3D {
    Deep2D xy;     // regions of one plane (nblocks: of the plane)
    int nz, zc, nzc;
    int nblocks;   // regions x chunks
};

// T iterations per pass, chunks of zc planes
inline Deep3D make_deep3(int nx, int ny, int nz, int lx, int h, int lo, int hi, int zc) {
    Deep3D g;
    g.xy = make_deep(nx, ny, lx, h, lo, hi);
    g.nz = nz;
    g.zc = zc < 1 ? 1 : (zc > nz ? nz : zc);
    g.nzc = (nz + g.zc - 1) / g.zc;
    g.nblocks = g.xy.nblocks * g.nzc;
    return g;
}

// Distance added between the fields of a solve: fields of 2^k bytes that follow
// each other agree in the address bits that pick the memory channel, and a
// pass then meets the same channels in all of them (256^3 FGP, two iterations
// per pass: 154 -> 135 us per iteration).
constexpr size_t kFieldSkew = 17 * 256;

// State that stays in the last-level cache (256 MB) from pass to pass.
constexpr size_t kDeep3CacheBytes = 200000000;

// The shapes a pass is built in, and how many of its workgroups run at once.
struct Deep3Shape { int nw, r, slots; };
constexpr Deep3Shape kDeep3Shapes_[] = {{16, 2, 256}, {8, 2, 512}};   // 64 x 32 and 64 x 16 columns
constexpr int kDeep3Shapes = 2;
constexpr int kDeep3Max = 4;   // iterations per pass at most
struct Deep3Cost { double cached_us[kDeep3Max], stream_us[kDeep3Max]; };
struct Deep3Plan { int shape, T; Deep3D g; };
// rlo / rhi: columns lost per iteration; bytes: of state per voxel; most: the
// largest T allowed; zchunk: planes per chunk (0: planned).
Deep3Plan plan_deep3(int nx, int ny, int nz, int rlo, int rhi, const Deep3Cost (&cost)[kDeep3Shapes], size_t bytes,
                     int most, int zchunk);

// The element offset of a plane, opaque to the optimiser: a field's address is
// then formed as scalar base + 32-bit lane offset at every access instead of
// a 64-bit lane pointer per field and row carried through the plane loop
// (28 VGPRs for FGP).
__device__ inline size_t plane_offset(int z, size_t sxy) {
    size_t o = (size_t)z * sxy;
    asm volatile("" : "+s"(o));
    return o;
}

// A value that has been waited for.
template <typename V>
__device__ inline void landed(V& v) { asm volatile("" : "+v"(v)); }

// Loads of one plane through a buffer descriptor: a field that is not read has
// size 0 and reads as zero, so the loads of the next plane stay unconditional
// and nothing waits for them before that plane.  off4: byte offset of the
// element in a 4-byte field.
template <typename S>
struct PlaneIn {
    __amdgpu_buffer_rsrc_t r;
    __device__ inline PlaneIn(const S* base, bool on, size_t sxy)
        : r(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, on ? (uint32_t)(sxy * sizeof(S)) : 0u, 0x00027000)) {}
    // what a load returns, kept as it is until it is used: a conversion right
    // after the load would wait for it
    using Word = typename std::conditional<sizeof(S) == 4, float, uint16_t>::type;
    __device__ inline Word word(uint32_t off4) const {
        if constexpr (sizeof(S) == 4)
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off4, 0, 0));
        else
            return __builtin_amdgcn_raw_buffer_load_b16(r, off4 >> 1, 0, 0);
    }
    __device__ static inline float value(Word w) {
        if constexpr (sizeof(S) == 4) return w;
        else if constexpr (std::is_same<S, bf16_t>::value) return __uint_as_float((uint32_t)w << 16);
        else return (float)__builtin_bit_cast(_Float16, w);
    }
    __device__ inline float ld(uint32_t off4) const { return value(word(off4)); }
};

// Store of v at byte offset `bytes` of a plane through a buffer
// descriptor, which drops an offset past its size: lanes that store nothing
// carry kNoStore, a plane that is not stored has size 0.  The store itself is
// unconditional, so the compiler knows how many are in flight and a wait for
// the next plane's loads (issued before them) does not wait for them too.
constexpr uint32_t kNoStore = 0x80000000u;   // planes are below 2^31 bytes
template <typename S>
struct PlaneOut {
    __amdgpu_buffer_rsrc_t r;
    __device__ inline PlaneOut(S* base, bool on, size_t sxy)
        : r(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, on ? (uint32_t)(sxy * sizeof(S)) : 0u, 0x00027000)) {}
    // off4: byte offset of the element in a 4-byte field
    __device__ inline void st(uint32_t off4, float v) const {
        if constexpr (sizeof(S) == 4) {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, off4, 0, 0);
        } else if constexpr (std::is_same<S, bf16_t>::value) {
            __builtin_amdgcn_raw_buffer_store_b16(Store<bf16_t>::bits_of(v), r, off4 >> 1, 0, 0);
        } else {
            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (_Float16)v), r, off4 >> 1, 0, 0);
        }
    }
    // v has been through_storage already: its upper half is the bf16 (no conversion)
    __device__ inline void st_rounded(uint32_t off4, float v) const {
        if constexpr (std::is_same<S, bf16_t>::value)
            __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(__float_as_uint(v) >> 16), r, off4 >> 1, 0, 0);
        else
            st(off4, v);
    }
};

// One thread's place in its workgroup's column.
template <class Sh>
struct DeepPos3 : DeepPos<Sh> {
    int z0, z1, nz;
    size_t sxy;
    __device__ inline DeepPos3(const Deep3D& g, int logical)
        : DeepPos<Sh>(g.xy, logical % g.xy.nblocks) {
        const int zi = logical / g.xy.nblocks;
        nz = g.nz;
        z0 = zi * g.zc;
        z1 = z0 + g.zc < g.nz ? z0 + g.zc : g.nz;
        sxy = (size_t)g.xy.nx * (size_t)g.xy.ny;
        this->lin = logical;
    }
};

// ---------------------------------------------------------------------------
// the solve loop
// ---------------------------------------------------------------------------
// What a pass reads and writes (state fields as in DeepArgs).
template <int NF, class Par>
struct Deep3Args {
    const float* f;
    const void* in[NF];
    void* out[NF];
    float* res;
    int cold, write_state, write_res;
    unsigned check;     // bit i: the pass's iteration i is checked
    double* partials;
    const Ctrl* ctrl;
    Deep3D g;
    Par par;
};

// deep_solve for volumes: the same state sets, stops, warm starts and output
// rule.  M supplies Args, NF, rlo, rhi, max (iterations per pass), seeded,
// field_size, load, store and prepare as there, cost(), bytes() (state per
// voxel), most(checked) (iterations per pass of a checked or unchecked solve)
// and launch(T, shape, args, stream).
template <class M>
int deep3_solve(M& m, const float* d_f, float* d_out, int nx, int ny, int nz, int iter, float epsil, const Opts& opts,
                hipStream_t s, int* iters_done, float* re, const WarmState* ws, int* last_iter = nullptr,
                const DeepExtra* extra = nullptr) {
    const size_t n = (size_t)nx * ny * nz;
    const bool use_tol = epsil != 0.0f;
    const int most = std::min(iter, m.most(use_tol));
    // shorter passes (the last one, a rerun up to a stop) run on the same regions and chunks
    const Deep3Plan plan = plan_deep3(nx, ny, nz, M::rlo, M::rhi, m.cost(), m.bytes(), most, opts.zchunk);
    const int width = plan.T;
    Arena ar;
    size_t of[2][M::NF], oX[3] = {0, 0, 0}, oR = 0;
    for (int i = 0; extra && i < extra->fields; ++i) oX[i] = ar.reserve(n * sizeof(float) + kFieldSkew);
    for (int b = 0; b < 2; ++b)
        for (int i = 0; i < M::NF; ++i) of[b][i] = ar.reserve(n * m.field_size(i) + kFieldSkew);
    const bool apart = d_out + n <= d_f || d_f + n <= d_out;
    if (!apart) oR = ar.reserve(n * sizeof(float));
    const size_t oCtrl = ar.reserve(sizeof(Ctrl));
    const size_t oPart = ar.reserve((size_t)plan.g.nblocks * 2 * width * sizeof(double));
    if (ar.allocate() != 0) return -1;
    if (extra) extra->fill({(float*)ar.at(oX[0]), (float*)ar.at(oX[1]), (float*)ar.at(oX[2])});
    float* res = apart ? d_out : (float*)ar.at(oR);
    Ctrl* ctrl = (Ctrl*)ar.at(oCtrl);
    const bool warm = ws && ws->warm;
    if (warm)
        for (int i = 0; i < M::NF; ++i) m.load(i, ar.at(of[0][i]), *ws, n, s);
    if (M::seeded && use_tol && !apart) launch_copy(res, d_out, n * sizeof(float), s);
    auto launch_pass = [&](int in, int k, int nk, unsigned mask, bool write_state, bool write_res, bool stop,
                           const Ctrl* c) {
        typename M::Args a;
        a.f = d_f;
        for (int i = 0; i < M::NF; ++i) {
            a.in[i] = ar.at(of[in][i]);
            a.out[i] = ar.at(of[in ^ 1][i]);
        }
        a.res = res;
        a.cold = k == 0 && !warm;
        a.write_state = write_state;
        a.write_res = write_res;
        a.check = mask;
        a.partials = (double*)ar.at(oPart);
        a.ctrl = c;
        a.g = plan.g;
        m.prepare(a, k, nk, stop);
        m.launch(nk, plan.shape, a, s);
    };
    int passes = 0;
    auto step = [&](int k, int nk, unsigned mask) {
        const bool last = k + nk == iter;
        const bool seed = M::seeded && use_tol && (k + nk) % opts.check_every == 0;
        launch_pass(passes & 1, k, nk, mask, !last || ws, last || seed, false, ctrl);
        ++passes;
    };
    int done = 0;
    if (drive_deep(iter, width, epsil, opts, ctrl, (double*)ar.at(oPart), plan.g.nblocks, s, step, &done, re) != 0)
        return -1;
    *iters_done = done;
    const int last = done < iter ? done : iter - 1, q = last / width;
    if (done < iter) launch_pass(q & 1, q * width, last - q * width + 1, 0, ws != nullptr, true, true, nullptr);
    if (!apart) launch_copy(d_out, res, n * sizeof(float), s);
    if (ws)
        for (int i = 0; i < M::NF; ++i) m.store(i, ar.at(of[(q & 1) ^ 1][i]), *ws, n, s);
    if (last_iter) *last_iter = last;
    const hipError_t launched = hipGetLastError();
    CILREG_CK(hipStreamSynchronize(s));
    CILREG_CK(launched);
    return 0;
}

// Calls fn(DeepShape<...>{}) for shape index s of a volume pass.
template <class Fn>
void deep3_dispatch(int s, Fn&& fn) {
    if (s == 0) fn(DeepShape<64, 16, 2>{});
    else fn(DeepShape<64, 8, 2>{});
}

// What a method's register passes need to be ahead of its passes on 64 x 8
// tiles beside half a million voxels.
struct Deep3Least {
    int rows, planes;   // at least so many
    bool small;         // also where a small volume's regions cover twice the points of its tiles
};
// Volumes the register passes take: enough voxels to fill the chip with
// regions (FGP 64^3 6.7 us per iteration in registers and 5.7 on tiles, 96^3 9.4
// and 11.1), planes below 2^31 bytes, and, by method,
//   rows: a region is 16 or 32 rows high, a tile 8 (2 rows of 5380, 171 planes,
//     FGP 34 to 50 us and 33 to 40; 5 rows of 2497, 494 planes, 41 and 57),
//   planes: a chunk repeats T planes at its ends,
//   small: below 1.2 million voxels regions of 64 x 16 points that lose two
//     columns and rows a side and are as many as the 64 x 8 tiles (128 x 48 x 128:
//     12 and 12) step no faster than these (PD 10.6 us and 9.6, FGP 10.4 and 10.3;
//     of 140 such volumes measured these are the only ones that lose).
inline bool deep3_fits(int nx, int ny, int nz, const Deep3Least& least) {
    const size_t sxy = (size_t)nx * ny, n = sxy * nz;
    if (n < 500000 || sxy >= ((size_t)1 << 29) || ny < least.rows || nz < least.planes) return false;
    const int tiles = ((nx + 63) / 64) * ((ny + 7) / 8);
    return least.small || n >= 1200000 || make_deep(nx, ny, 64, 16, 2, 2).nblocks < tiles;
}

// Rows of whole 128-byte lines whose state (bytes per voxel) streams from HBM:
// the tiled passes' best case.
inline bool deep3_lines(int nx, int ny, int nz, size_t bytes) {
    return nx % 32 == 0 && bytes * nx * ny * nz > kDeep3CacheBytes;
}

}  // namespace cilreg
