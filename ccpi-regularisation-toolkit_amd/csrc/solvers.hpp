// solvers.hpp -- device-resident solver entry points shared by the C ABI, the
// extension API, the batch launcher and the serving loop.
//
// Every solver takes device pointers and a stream, runs `iter` iterations of
// its method with the reference's stopping rule, writes the reference's
// output into d_out and reports the iteration count and last residual.  FGP,
// PD and TGV (T = float) optionally start from and return their iterate state
// (WarmState): the state after the executed iterations -- all `iter`, or up
// to and including the iteration at which the stopping rule fired (one
// iteration per pass then).
#pragma once
#include "runtime.hpp"
#include "state.hpp"
#include <functional>

namespace cilreg {

template <typename T, typename S>
int rof_solve(const T* d_f, T* d_out, T lambda, int iter, T tau, T epsil, int nx, int ny, int nz, const Opts& opts,
              hipStream_t s, int* iters_done, float* re);
template <typename T, typename S>
int fgp_solve(const T* d_f, T* d_out, T lambda, int iter, T epsil, int method, int nonneg, int nx, int ny, int nz,
              const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws = nullptr);
template <typename T, typename S>
int pd_solve(const T* d_f, T* d_out, T lambda, int iter, T epsil, T lipschitz, int method, int nonneg, int nx, int ny,
             int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws = nullptr);
template <typename T, typename S>
int sb_solve(const T* d_f, T* d_out, T mu, int iter, T epsil, int method, int nx, int ny, int nz, const Opts& opts,
             hipStream_t s, int* iters_done, float* re, const WarmState* ws = nullptr);
template <typename T, typename S>
int tgv_solve(const T* d_f, T* d_out, T lambda, T alpha1, T alpha0, int iter, T L2, T epsil, int nx, int ny, int nz,
              const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws = nullptr);
int llt_solve(const float* d_f, float* d_out, float lambda_rof, float lambda_llt, int iter, float tau, float epsil,
              int nx, int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re);
int ndf_solve(const float* d_f, float* d_out, float lambda, float sigma, int iter, float tau, int penalty, float epsil,
              int nx, int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re);
int d4_solve(const float* d_f, float* d_out, float lambda, float sigma, int iter, float tau, float epsil, int nx,
             int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re);
template <typename T>
int dtv_solve(const T* d_f, const T* d_ref, T* d_out, T lambda, int iter, T epsil, T eta, int method, int nonneg,
              int nx, int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re);

// FGP's t_k sequence in float (FGP_TV_core.c:138,159), resumed from a warm
// state: mult[k] multiplies P_k - P_{k-1} in iteration k, tks[k] is t_k.
inline void fgp_multipliers(int iter, const WarmState* ws, std::vector<float>& mult, std::vector<float>& tks) {
    mult.resize(iter + 1);
    tks.resize(iter + 1);
    float tk = 1, m = 0;
    if (ws && ws->warm) {
        tk = ws->tstate[0];
        m = ws->tstate[1];
    }
    for (int k = 0; k <= iter; ++k) {
        mult[k] = m;
        tks[k] = tk;
        const float tkp1 = (1.0f + dsqrt_host(1.0f + 4.0f * tk * tk)) * 0.5f;
        m = (tk - 1.0f) / tkp1;
        tk = tkp1;
    }
}

// Whether fgp_solve / pd_solve take a volume to fgp_solve_3d / pd_solve_3d.
template <typename S>
bool fgp_in_registers(int nx, int ny, int nz, float epsil, const Opts& opts);
template <typename S>
bool pd_in_registers(int nx, int ny, int nz, float epsil, const Opts& opts);

// 2D solves with many iterations per launch (opts.depth: 0 = as many as pay,
// 2 = two; S: storage of the dual fields).
template <typename S>
int fgp_solve_2d(const float* d_f, float* d_out, float lambda, int iter, float epsil, int method, int nonneg, int nx,
                 int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws);
template <typename S>
int fgp_solve_3d(const float* d_f, float* d_out, float lambda, int iter, float epsil, int method, int nonneg, int nx,
                 int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re, const WarmState* ws);
int sb_solve_2d(const float* d_f, float* d_out, float lam, float mu, float nc, float thr, int iter, float epsil,
                int method, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                const WarmState* ws);
int ndf_solve_2d(const float* d_f, float* d_out, float lambda, float sigma, int iter, float tau, int penalty,
                 float epsil, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re);
// Queues the kernel that fills the components of FGP-dTV's B.
using RefGrad = std::function<void(float* const (&)[3])>;
int dtv_solve_2d(const float* d_f, const RefGrad& refgrad, float* d_out, float lambda, int iter, float epsil,
                 int method, int nonneg, int nx, int ny, const std::vector<float>& mult, const Opts& opts,
                 hipStream_t s, int* iters_done, float* re);
int dtv_solve_3d(const float* d_f, const RefGrad& refgrad, float* d_out, float lambda, int iter, float epsil,
                 int method, int nonneg, int nx, int ny, int nz, const std::vector<float>& mult, const Opts& opts,
                 hipStream_t s, int* iters_done, float* re);
template <typename S>
int pd_solve_3d(const float* d_f, float* d_out, float lambda, int iter, float epsil, float lipschitz, int method,
                int nonneg, int nx, int ny, int nz, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                const WarmState* ws);
template <typename S>
int pd_solve_2d(const float* d_f, float* d_out, float lambda, int iter, float epsil, float lipschitz, int method,
                int nonneg, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                const WarmState* ws);
template <typename S>
int tgv_solve_2d(const float* d_f, float* d_out, float lambda, float alpha1, float alpha0, int iter, float L2,
                 float epsil, int nx, int ny, const Opts& opts, hipStream_t s, int* iters_done, float* re,
                 const WarmState* ws);
int rof_solve_2d(const float* d_f, float* d_out, float lambda, int iter, float tau, float epsil, int nx, int ny,
                 const Opts& opts, hipStream_t s, int* iters_done, float* re);

}  // namespace cilreg
