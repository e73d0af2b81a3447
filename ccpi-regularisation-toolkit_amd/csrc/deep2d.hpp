// deep2d.hpp -- many iterations per launch on a 2D image: the pass geometry,
// the neighbour exchange, the choice of the pass shape and the solve loop
// shared by every 2D method (kernels: *2d.hip).
//
// A 2D image is small: one iteration is a few microseconds of arithmetic, a
// launch costs about as much, and the traffic of one iteration is what
// remains.  A pass therefore keeps a region of the image in registers and
// advances it by up to kDeepMax iterations before it stores.  A workgroup of
// NW waves owns a region of LX columns (LX = 64: a wave is one row group; 32:
// two) by H = (64 NW / LX) R rows; every thread holds R vertically adjacent
// points of one column.  Per iteration a value moves
//   along x by a DPP wave shift (5 issue cycles; a shuffle through LDS
//   measured 24),
//   along y within a thread as a register, and between row groups through one
//   LDS row per group, with one or two barriers.
// Each iteration invalidates `lo` columns and rows at the low and `hi` at the
// high edge of a region, unless that edge is the image's own: a pass of n
// iterations stores the region's interior, and neighbouring regions overlap
// by (lo + hi) n.  Values are computed by the one-iteration kernels'
// expressions in the same order, so the results are bit-identical to one
// iteration per launch.
#pragma once
#include "runtime.hpp"
#include "state.hpp"
#include <functional>

namespace cilreg {

constexpr int kDeepMax = 8;   // iterations per pass at most

// Regions of LX x H points that cover nx x ny when each loses lo / hi columns
// and rows at its inner edges.
struct Deep2D {
    int nx, ny;
    int tiles_x, tiles_y;
    int step_x, step_y;   // distance between region origins
    int lo, hi;           // columns (rows) lost at a low / high inner edge
    int nblocks;
};

inline Deep2D make_deep(int nx, int ny, int lx, int h, int lo, int hi) {
    Deep2D g;
    g.nx = nx;
    g.ny = ny;
    g.lo = lo;
    g.hi = hi;
    g.step_x = lx - lo - hi;
    g.step_y = h - lo - hi;
    g.tiles_x = nx <= lx ? 1 : (nx - lx + g.step_x - 1) / g.step_x + 1;
    g.tiles_y = ny <= h ? 1 : (ny - h + g.step_y - 1) / g.step_y + 1;
    g.nblocks = g.tiles_x * g.tiles_y;
    return g;
}

template <int LX_, int NW_, int R_>
struct DeepShape {
    static constexpr int LX = LX_, NW = NW_, R = R_;
    static constexpr int G = 64 * NW / LX;   // row groups
    static constexpr int H = G * R;
};

// What a pass reads and writes.  State fields have their own element types
// (the kernel knows them); a cold pass starts from the method's initial state
// instead of reading them.
template <typename T, int NF, class Par>
struct DeepArgs {
    const T* f;
    const void* in[NF];
    void* out[NF];
    T* res;             // the output of the pass's last iteration, written when write_res
    int nit, cold, write_state, write_res;
    unsigned check;     // bit i: the pass's iteration i is checked
    double* partials;
    const Ctrl* ctrl;
    Deep2D g;
    Par par;
};

// One thread's place in its workgroup's region.
template <class Sh>
struct DeepPos {
    int lx, grp;       // column and row group within the region
    int x, y;          // image coordinates of the thread's first point
    int nx, ny;
    bool xout;         // the column is stored by this region
    bool xedge, yedge; // wave-uniform: the wave holds the image's first or last column / row
    int ylo, yhi;      // image rows [ylo, yhi) are stored by this region
    int lin;

    __device__ inline DeepPos(const Deep2D& g) : DeepPos(g, xcd_logical_block((int)blockIdx.x, g.nblocks)) {}
    __device__ inline DeepPos(const Deep2D& g, int logical) {
        lin = logical;
        nx = g.nx;
        ny = g.ny;
        const int ty = lin / g.tiles_x, tx = lin - ty * g.tiles_x;
        const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
        lx = lane & (Sh::LX - 1);
        grp = Sh::LX == 64 ? wave : wave + Sh::NW * (lane >> 5);
        const int xs = tx * g.step_x, ys = ty * g.step_y;
        x = xs + lx;
        y = ys + grp * Sh::R;
        const int xlo = xs + (tx > 0 ? g.lo : 0), xhi = tx + 1 < g.tiles_x ? xs + Sh::LX - g.hi : nx;
        xout = x >= xlo && x < xhi;
        xedge = tx == 0 || tx + 1 == g.tiles_x;
        const bool ye = y == 0 || y + Sh::R >= ny;
        yedge = Sh::LX == 64 ? ye : __builtin_amdgcn_ballot_w64(ye) != 0;
        ylo = ys + (ty > 0 ? g.lo : 0);
        yhi = ty + 1 < g.tiles_y ? ys + Sh::H - g.hi : ny;
    }
    __device__ inline bool out(int r) const { return xout && y + r >= ylo && y + r < yhi; }
    // element of row r (a valid stand-in outside the image)
    __device__ inline size_t elem(int r) const {
        const int cx = x < nx ? x : nx - 1, cy = y + r < ny ? y + r : ny - 1;
        return (size_t)cy * (size_t)nx + (size_t)cx;
    }
};

// First in a wave-uniform branch that few waves take: keeps the compiler from
// turning the branch into selects that every wave issues.
__device__ inline void deep_keep_branch() { asm volatile(""); }

// The value one column to the left / right: lane -/+ 1 of the wave, zero past
// its ends.  All lanes must take part (call it outside divergent code).  With
// LX = 32 a wave's halves are different rows, so lane 32's left and lane 31's
// right neighbour belong to the other half; both are region edges.
__device__ inline float deep_left(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ inline float deep_right(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}
// The left neighbour with zero before the region's first column (which is the
// image's first column or an edge where no valid value is read).
template <class Sh>
__device__ inline float deep_left0(const DeepPos<Sh>& p, float v) {
    const float l = deep_left(v);
    return Sh::LX == 64 || p.lx > 0 ? l : 0.0f;
}

// One row per group of one value, double-buffered by iteration parity so one
// barrier separates its writes from its reads.
template <class Sh>
struct DeepRow {
    float v[2][Sh::G][Sh::LX];
    __device__ inline void put(const DeepPos<Sh>& p, int b, float x) { v[b][p.grp][p.lx] = x; }
    // the row of the group below (the last group's own row at the region's end)
    __device__ inline float below(const DeepPos<Sh>& p, int b) const {
        return v[b][p.grp + 1 < Sh::G ? p.grp + 1 : p.grp][p.lx];
    }
    // the row of the group above (the first group's own row at the region's start)
    __device__ inline float above(const DeepPos<Sh>& p, int b) const {
        return v[b][p.grp > 0 ? p.grp - 1 : 0][p.lx];
    }
};

// Residual sums of one check: per wave by shuffles into red, summed in wave
// order by deep_store_checks after the pass.
template <class Sh>
struct DeepRed { double v[2 * kDeepMax * Sh::NW]; };
template <class Sh>
__device__ inline void deep_check(DeepRed<Sh>& red, double sd, double su, int c) {
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        sd += __shfl_xor(sd, off, 64);
        su += __shfl_xor(su, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        const int w = (int)threadIdx.x >> 6;
        red.v[2 * (c * Sh::NW + w)] = sd;
        red.v[2 * (c * Sh::NW + w) + 1] = su;
    }
}
// partials: nblocks pairs per check, check after check.
template <class Sh>
__device__ inline void deep_store_checks(const DeepRed<Sh>& red, int nchk, double* partials, int nblocks, int lin) {
    if (nchk == 0) return;
    __syncthreads();
    const int t = (int)threadIdx.x;
    if (t < 2 * nchk) {
        const int c = t >> 1, h = t & 1;
        double s = 0;
        for (int w = 0; w < Sh::NW; ++w) s += red.v[2 * (c * Sh::NW + w) + h];
        partials[2 * ((size_t)c * nblocks + lin) + h] = s;
    }
}

// ---------------------------------------------------------------------------
// choice of the pass shape (host)
// ---------------------------------------------------------------------------
// The shapes a kernel is built in, and a launch's fixed time (launch, first
// loads, last stores) in microseconds.
struct DeepShapeCost { int lx, nw, r; double base_us; };
constexpr DeepShapeCost kDeepShapes[] = {
    {32, 16, 1, 3.1},   // 32 x 32: small images, every CU gets a region
    {64, 16, 2, 3.4},   // 64 x 32
    {64, 16, 4, 4.4},   // 64 x 64: least overlap
    {64, 8, 4, 3.7},    // 64 x 32 on half the waves: several regions per CU
    // 64 x 4 and 64 x 8: images of so few rows.  Long ones would leave 3/4 and
    // more of the others empty, which is slower than the one-iteration kernels'
    // 64 x 4 tiles (10^6 x 4, us per iteration by tiles, in 64 x 32 regions and
    // here: FGP 26.4, 35.7, 9.0; TGV 58, 109, 18; ROF 28, 56, 12; 10^6 x 8: FGP
    // 51, 37, 13.5; TGV with BF16 storage 92, 129, 33).
    {64, 4, 1, 3.1},
    {64, 4, 2, 3.1},
};
constexpr int kDeepShapeCount = (int)(sizeof(kDeepShapes) / sizeof(kDeepShapes[0]));

// A method's microseconds per iteration in each shape, measured on this
// device: of one workgroup alone on a CU, and per workgroup when a CU holds
// several.
struct DeepIterCost { double alone_us, shared_us; };

struct DeepPlan { int shape, width; Deep2D g; };
// rlo / rhi: columns lost per iteration at a low / high edge; words: read and
// written per point and pass; most: the largest width allowed; rows: the most
// rows per thread.
DeepPlan plan_deep(int nx, int ny, int rlo, int rhi, const DeepIterCost (&cost)[kDeepShapeCount], int words, int most,
                   int rows);

// Calls fn(DeepShape<...>{}) for shape index s.
template <class Fn>
void deep_dispatch(int s, Fn&& fn) {
    switch (s) {
        case 0: fn(DeepShape<32, 16, 1>{}); break;
        case 1: fn(DeepShape<64, 16, 2>{}); break;
        case 2: fn(DeepShape<64, 16, 4>{}); break;
        case 3: fn(DeepShape<64, 8, 4>{}); break;
        case 4: fn(DeepShape<64, 4, 1>{}); break;
        default: fn(DeepShape<64, 4, 2>{}); break;
    }
}

// Fields of a solve's own beside its state (FGP-dTV's B): they lie in the
// solve's allocation, so that no kernel is queued before the last allocation
// that can fail (a block given back while a kernel still writes it could reach
// another thread's solve).  fill queues the kernels that compute them.
struct DeepExtra {
    int fields;   // at most 3, float
    std::function<void(float* const (&)[3])> fill;
};

// ---------------------------------------------------------------------------
// the solve loop
// ---------------------------------------------------------------------------
// A method's shapes: the most rows per thread on an nx x ny image.
struct DeepMethod {
    static int most_rows(int, int) { return 4; }
};

// M, a DeepMethod, supplies
//   using Args                       its DeepArgs
//   static constexpr int NF          state fields per set
//   static constexpr int rlo, rhi    columns lost per iteration
//   static constexpr DeepIterCost cost[kDeepShapeCount]; int words
//   size_t field_size(i)             element size of state field i
//   void prepare(Args&, k, nk, stop) per-pass parameters; stop: this pass ends
//                                    with the iteration at which the rule fired
//   template <class Sh> void launch(const Args&, hipStream_t)
//   bool seeded                      res holds the iterate before the first
//                                    one (d_out's prior contents) and a pass
//                                    that ends before a check must write res
//   void load(i, dst, ws, n, s) / store(i, src, ws, n, s)  warm-start state
// The state lives in two sets, a pass reads one and writes the other; the
// first pass of a cold solve reads none.  A stop at iteration j reruns its
// pass from the input set up to j: the passes queued after the stop return at
// once and leave that set intact.  The result goes straight to d_out unless
// that overlaps the input, which later regions of the same pass still read.
template <class M, typename T>
int deep_solve(M& m, const T* d_f, T* d_out, int nx, int ny, int iter, T epsil, const Opts& opts, hipStream_t s,
               int* iters_done, float* re, const WarmState* ws, int* last_iter = nullptr,
               const DeepExtra* extra = nullptr) {
    const size_t n = (size_t)nx * ny;
    const bool use_tol = epsil != (T)0;
    int most = opts.depth >= 2 ? 2 : kDeepMax;
    if (most > iter) most = iter;
    const DeepPlan plan = plan_deep(nx, ny, M::rlo, M::rhi, M::cost, M::words, most, M::most_rows(nx, ny));
    const int width = plan.width;

    Arena ar;
    if (opts.scratch) ar.use_external(opts.scratch, opts.scratch_bytes);
    size_t of[2][M::NF], oX[3] = {0, 0, 0}, oR = 0;
    for (int b = 0; b < 2; ++b)
        for (int i = 0; i < M::NF; ++i) of[b][i] = ar.reserve(n * m.field_size(i));
    for (int i = 0; extra && i < extra->fields; ++i) oX[i] = ar.reserve(n * sizeof(float));
    const bool apart = d_out + n <= d_f || d_f + n <= d_out;
    if (!apart) oR = ar.reserve(n * sizeof(T));
    const size_t oCtrl = ar.reserve(sizeof(Ctrl));
    const size_t oPart = ar.reserve((size_t)plan.g.nblocks * 2 * width * sizeof(double));
    if (ar.allocate() != 0) return -1;
    if (extra) extra->fill({(float*)ar.at(oX[0]), (float*)ar.at(oX[1]), (float*)ar.at(oX[2])});
    T* res = apart ? d_out : (T*)ar.at(oR);
    Ctrl* ctrl = (Ctrl*)ar.at(oCtrl);
    const bool warm = ws && ws->warm;
    if (warm)
        for (int i = 0; i < M::NF; ++i) m.load(i, ar.at(of[0][i]), *ws, n, s);
    if (M::seeded && use_tol && !apart) launch_copy(res, d_out, n * sizeof(T), s);

    auto launch_pass = [&](int in, int k, int nk, unsigned mask, bool write_state, bool write_res, bool stop,
                           const Ctrl* c) {
        typename M::Args a;
        a.f = d_f;
        for (int i = 0; i < M::NF; ++i) {
            a.in[i] = ar.at(of[in][i]);
            a.out[i] = ar.at(of[in ^ 1][i]);
        }
        a.res = res;
        a.nit = nk;
        a.cold = k == 0 && !warm;
        a.write_state = write_state;
        a.write_res = write_res;
        a.check = mask;
        a.partials = (double*)ar.at(oPart);
        a.ctrl = c;
        a.g = plan.g;
        m.prepare(a, k, nk, stop);
        deep_dispatch(plan.shape, [&](auto sh) { m.template launch<decltype(sh)>(a, s); });
    };
    int passes = 0;
    auto step = [&](int k, int nk, unsigned mask) {
        const bool last = k + nk == iter;
        const bool seed = M::seeded && use_tol && (k + nk) % opts.check_every == 0;
        launch_pass(passes & 1, k, nk, mask, !last || ws, last || seed, false, ctrl);
        ++passes;
    };
    Opts o = opts;
    o.poll = 4 * width > o.poll ? 4 * width : o.poll;
    int done = 0;
    if (drive_deep(iter, width, (float)epsil, o, ctrl, (double*)ar.at(oPart), plan.g.nblocks, s, step, &done, re) != 0)
        return -1;
    *iters_done = done;
    const int last = done < iter ? done : iter - 1;
    const int q = last / width;   // the pass holding iteration `last`
    if (done < iter) launch_pass(q & 1, q * width, last - q * width + 1, 0, ws != nullptr, true, true, nullptr);
    if (!apart) launch_copy(d_out, res, n * sizeof(T), s);
    if (ws)
        for (int i = 0; i < M::NF; ++i) m.store(i, ar.at(of[(q & 1) ^ 1][i]), *ws, n, s);
    if (last_iter) *last_iter = last;
    const hipError_t launched = hipGetLastError();
    CILREG_CK(hipStreamSynchronize(s));
    CILREG_CK(launched);
    return 0;
}

}  // namespace cilreg
