// hd_lanczos.hip -- device-resident thick-restart Lanczos (FP64 recurrence).
//
// Reference: ArpackWrapper::DiagonalizeSymmetricMatrix (src/utilities/wrappers/arpack_wrapper.hpp:595-937)
// drives PARPACK p?naupd/p?neupd by reverse communication, WHICH = 'SR',
// NCV = min(N, 2*NEV+21), exact shifts, maxiter 2000 (arpack_wrapper.cpp:38-49),
// with every mat-vec a host round trip through MatrixVectorFunction::Simple.
// Here the Krylov basis, the operator and all vector work stay in HBM, and so do the
// coefficients and decisions inside a cycle; the host queues the cycle's launches and
// sees the small projected matrix at its end.  Method: thick-restart Lanczos (Wu and
// Simon, SIAM J. Matrix Anal. Appl. 22 (2000) 602) with full
// reorthogonalisation: each step first removes the three-term part locally
// (w -= beta v_{j-1}; alpha = v_j.w; w -= alpha v_j), then one classical
// Gram-Schmidt pass against the whole basis, with a second pass when the norm
// drops by more than 100x (the DGKS criterion); the first step after a restart
// (whose projection is the arrow, not tridiagonal) always takes two passes
// (Giraud et al., Numer. Math. 101 (2005) 87).  The projected
// tridiagonal-plus-arrow matrix is diagonalised on the host.
//
// Mixed precision (precision = HD_F32) chooses the operator per restart
// cycle.  An operator error F_j in the product of basis vector v_j enters the
// residual of a Ritz vector y = sum_j s_j v_j as sum_j s_j F_j, which the
// recurrence never sees (Simoncini, SIAM J. Numer. Anal. 43 (2005) 1155:
// products may be inexact where the Ritz coefficients are small).  The kept
// Ritz vectors carry O(1) coefficients on every vector of the cycles that made
// them, so the early cycles use the exact FP64 operator; once the wanted Ritz
// vectors' coefficients on a cycle's new vectors are small, the FP32-input
// operator (HD_TILED_X32, exact for x rounded to FP32, or the FP32-value CRS)
// takes the cycle.  The rounding such a cycle adds to the residual of wanted
// pair i is estimated by eps32 |T| |s_i,new| (eps32 the operator's relative
// rounding, |T| the largest projected row, s_i,new the pair's coefficients on
// the cycle's new vectors); a cycle runs in FP32 only while the sum of these
// estimates, with the next cycle's predicted coefficients, stays within
// f32_budget * tol * max(1, |theta_i|).  The prediction cannot see an
// eigenvalue that enters the wanted window during the cycle, so the estimate
// is checked again with the cycle's actual coefficients, and a cycle beyond
// the budget is discarded (its starting state is still there) and run in FP64.
// Convergence is the usual Ritz test;
// the eigenpairs are then checked with the FP64 operator, and hd_lanczos
// repeats the solve with the FP64 operator should a residual miss tol.  All
// reductions are FP64 and deterministic (per-block partials reduced in a fixed
// order).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <numeric>

#include "hd_internal.hpp"


namespace hd {

void lanczos_state_free(hd_lanczos_state* s)
{
    if (!s) return;
    dfree(s->d_vec);
    delete s;
}

// ------------------------------------------------------------ device side

template <bool C> struct E;
template <> struct E<false> { using T = double; using F = float; };
template <> struct E<true> { using T = double2; using F = float2; };

HD_DEV double conj_mul(double a, double b) { return a * b; }          // conj(a) b
HD_DEV double2 conj_mul(double2 a, double2 b)
{
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}
HD_DEV double mul(double a, double b) { return a * b; }
HD_DEV double2 mul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
HD_DEV double sub(double a, double b) { return a - b; }
HD_DEV double2 sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
HD_DEV double add2(double a, double b) { return a + b; }
HD_DEV double2 add2(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
HD_DEV double norm2(double a) { return a * a; }
HD_DEV double norm2(double2 a) { return a.x * a.x + a.y * a.y; }
HD_DEV double scale(double a, double s) { return a * s; }
HD_DEV double2 scale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
template <typename T> HD_DEV T zero();
template <> HD_DEV double zero<double>() { return 0.0; }
template <> HD_DEV double2 zero<double2>() { return make_double2(0.0, 0.0); }
HD_DEV float narrow(double a) { return (float)a; }
HD_DEV float2 narrow(double2 a) { return make_float2((float)a.x, (float)a.y); }
HD_DEV double widen(float a) { return (double)a; }
HD_DEV double2 widen(float2 a) { return make_double2((double)a.x, (double)a.y); }

constexpr int kVB = 256;  // block size of the vector kernels
constexpr int kNV = 16;   // vectors per dot-product pass
constexpr int kMaxBasis = 256;               // Krylov basis limit (ncv)

__global__ void __launch_bounds__(kVB) k_reduce_real(const double* __restrict__ partial, int nb, double* __restrict__ out)
{
    __shared__ double red[kVB];
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += kVB) s += partial[b];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = kVB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

template <bool C>
__global__ void k_scale(int64_t dim, const typename E<C>::T* __restrict__ src, double s,
                        typename E<C>::T* __restrict__ dst)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < dim; r += stride)
        dst[r] = scale(src[r], s);
}

// out_l = sum_i V_i Y[i][l] for l in [l0, l0+nl), nl <= NL, with the m x nl
// block of Y staged in LDS (m * nl doubles of dynamic LDS).
template <bool C, int NL>
__global__ void __launch_bounds__(kVB)
k_combine(int64_t dim, const typename E<C>::T* __restrict__ V, int64_t ld, int m,
          const double* __restrict__ Y, int ldy, int l0, int nl, typename E<C>::T* __restrict__ out)
{
    using T = typename E<C>::T;
    extern __shared__ double sy[];
    for (int i = threadIdx.x; i < m * nl; i += kVB) sy[i] = Y[(i / nl) * ldy + l0 + (i % nl)];
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * kVB;
    for (int64_t r = (int64_t)blockIdx.x * kVB + threadIdx.x; r < dim; r += stride) {
        T acc[NL];
#pragma unroll
        for (int l = 0; l < NL; ++l) acc[l] = zero<T>();
        // four basis vectors' loads in flight per thread; the sum over i keeps
        // its order
        for (int i0 = 0; i0 < m; i0 += 4) {
            T v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = i0 + u < m ? V[(int64_t)(i0 + u) * ld + r] : zero<T>();
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (i0 + u >= m) break;
#pragma unroll
                for (int l = 0; l < NL; ++l)
                    if (l < nl) acc[l] = add2(acc[l], scale(v[u], sy[(i0 + u) * nl + l]));
            }
        }
#pragma unroll
        for (int l = 0; l < NL; ++l)
            if (l < nl) out[(int64_t)l * ld + r] = acc[l];
    }
}

// ------------------------------------------------------- the Lanczos step
//
// A cycle's steps run without the host: the recurrence coefficients, the overlap
// estimates of the partial reorthogonalisation and the decision to make a full
// pass stay on the device, so the host enqueues whole cycles (or blocks of steps,
// where it tests convergence) and reads the coefficients once.  Step j works in
// place: the product writes H v_j to the slot of v_{j+1}, and every kernel below
// leaves at once when an earlier step stopped (`stop`), so that slot keeps its
// content for the host to deal with.  Each step used to wait for the host four
// times (product, <v,w>, |w|, pass coefficients).
constexpr int kStopSecond = 1;  // the pass cancelled too much: a second one is due
constexpr int kStopBreak = 2;   // beta_j vanished: invariant subspace

struct LzState {
    double alpha[kMaxBasis], beta[kMaxBasis];
    int stop, stop_step;
    int reorth;             // full passes made
    int full;               // this step makes a full pass
    int skip;               // its projection is skipped (overlaps at rounding level)
    int force[2];           // the next step must make one, by parity of the step
    double anorm[2];        // largest |alpha| + beta so far, by parity of the step
    double a, bj, wn2;      // <v_j, w>, |w| and |w|^2 of the running step
    double cdiag[2];        // Re <v_j, w> found by the passes
    double theta[kMaxBasis], arrow[kMaxBasis];  // the cycle's kept Ritz pairs
    double om[3][kMaxBasis + 2];                // overlap estimates of v_i in om[i % 3]
};

struct LzStep {
    int64_t n;
    int j, k;               // step, kept Ritz vectors at the head of the basis
    int first;              // j == k: the couplings to the kept vectors are the arrow
    int must;               // a full pass whatever the estimates say
    double eps_op, om_cycle;
    double skip_tol;        // see k_lz_project
};

template <int NT>
HD_DEV double block_sum(double v)
{
    __shared__ double red[NT / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();  // an earlier sum has been read
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) s += red[i];
    return s;
}

template <int NT>
HD_DEV double block_max(double v)
{
    __shared__ double red[NT / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) s = fmax(s, red[i]);
    return s;
}

// Sum of `nb` per-block partials in a fixed order, the same in every block.
template <int NT>
HD_DEV double sum_partials(const double* __restrict__ p, int nb)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < nb; i += NT) s += p[i];
    return block_sum<NT>(s);
}

HD_DEV double shfl_xor_t(double v, int o) { return __shfl_xor(v, o, 64); }
HD_DEV double2 shfl_xor_t(double2 v, int o) { return make_double2(__shfl_xor(v.x, o, 64), __shfl_xor(v.y, o, 64)); }
HD_DEV double real_of(double a) { return a; }
HD_DEV double real_of(double2 a) { return a.x; }

// Whether step j needs a full pass (H. D. Simon's estimates of <v_{j+1}, v_i>,
// i < j, from b_j v_{j+1} = A v_j - a_j v_j - b_{j-1} v_{j-1}).  Real: the signed
// recurrence.  Complex: the overlaps are complex, so their magnitudes are
// propagated by the triangle inequality (an upper bound).  Evaluated by every
// block alike; the one with `write` stores the new estimates, |w| and the flags,
// none of which a block of the same launch reads.
template <bool C, int NT>
HD_DEV bool needs_pass(LzState* st, const LzStep& p, double a, double wn2, bool write)
{
    const int j = p.j, k = p.k, par = j & 1;
    const double bj = sqrt(fmax(wn2, 0.0));
    const double anorm = fmax(st->anorm[par], fabs(a) + bj);
    bool full = p.must || st->force[par];
    bool force = false;
    if (!full) {
        if (!(bj > 1e-12 * fmax(anorm, 1e-300))) {
            full = true;  // breakdown: decided with the orthogonalised w
        } else {
            const double* cur = st->om[j % 3];
            const double* prev = st->om[(j + 2) % 3];
            double* next = st->om[(j + 1) % 3];
            const double noise = 2.0 * p.eps_op * anorm / bj;
            double worst = 0.0;
            for (int i = threadIdx.x; i < j; i += NT) {
                double tv, dii;  // (A v_i)^H v_j through the projected matrix, diagonal term apart
                auto f = [](double x) { return C ? fabs(x) : x; };
                if (i < k) {
                    dii = st->theta[i];
                    tv = f(st->arrow[i]) * cur[k];
                } else if (i == k) {
                    dii = st->alpha[k];
                    tv = f(st->beta[k]) * cur[k + 1];
                    for (int l = 0; l < k; ++l) tv += f(st->arrow[l]) * cur[l];
                } else {
                    dii = st->alpha[i];
                    tv = f(st->beta[i - 1]) * cur[i - 1] + f(st->beta[i]) * cur[i + 1];
                }
                const double v = (tv + f(dii - a) * cur[i] + (C ? 1.0 : -1.0) * st->beta[j - 1] * prev[i]) / bj;
                const double nx = v + (v >= 0 ? noise : -noise);
                if (write) next[i] = nx;
                worst = fmax(worst, fabs(nx));
            }
            if (write && threadIdx.x == 0) {
                next[j] = p.eps_op * anorm / bj;
                next[j + 1] = 1.0;
            }
            worst = block_max<NT>(worst);
            full = force = worst > p.om_cycle;
        }
    }
    if (write && threadIdx.x == 0) {
        st->wn2 = wn2;
        st->bj = bj;
        st->full = full;
        st->force[par ^ 1] = force;
    }
    return full;
}

// v_{j+1} = w / b and the step's coefficients.
struct LzBeta {
    double alpha, b, anorm;
    int stop;
};

// The step's alpha and beta; `full`: w has been through the pass(es).
HD_DEV LzBeta step_beta(const LzState* st, const LzStep& p, bool full, bool skip, double nrm2, bool second_done)
{
    LzBeta r{st->a, st->bj, 0.0, 0};
    if (full) {
        if (skip) {
            r.b = sqrt(fmax(st->wn2, 0.0));
        } else {
            if (!second_done && nrm2 * 1e4 < st->wn2) r.stop = kStopSecond;
            r.b = sqrt(fmax(nrm2, 0.0));
            r.alpha = st->a + (second_done ? st->cdiag[0] + st->cdiag[1] : st->cdiag[0]);
        }
    }
    r.anorm = fmax(st->anorm[p.j & 1], fabs(r.alpha) + r.b);
    if (!r.stop && r.b <= 1e-12 * fmax(r.anorm, 1e-300)) r.stop = kStopBreak;
    return r;
}

// Bookkeeping of a finished (or stopped) step, by one block of NT threads.
template <int NT>
HD_DEV void finish_step(LzState* st, const LzStep& p, const LzBeta& r, bool full)
{
    const int j = p.j;
    const double eps = 2.220446049250313e-16;
    if (threadIdx.x == 0) {
        if (full && r.stop != kStopSecond) ++st->reorth;
        if (r.stop) {
            st->stop_step = j;
            st->stop = r.stop;
        }
        if (r.stop != kStopSecond) {
            st->alpha[j] = r.alpha;
            st->anorm[(j & 1) ^ 1] = r.anorm;
        }
        if (!r.stop) st->beta[j] = r.b;
        if (p.first) st->force[(j & 1) ^ 1] = 0;
    }
    if (!full || r.stop) return;
    for (int i = threadIdx.x; i < kMaxBasis + 2; i += NT) {
        st->om[(j + 1) % 3][i] = i == j + 1 ? 1.0 : eps;
        if (p.first) st->om[j % 3][i] = i == j ? 1.0 : eps;
    }
}

// w -= beta_{j-1} v_{j-1};  partial[block] = Re sum conj(v_j) w.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_dot(LzStep p, const typename E<C>::T* __restrict__ vp, const typename E<C>::T* __restrict__ vc,
         typename E<C>::T* __restrict__ w, const LzState* __restrict__ st, double* __restrict__ partial)
{
    if (st->stop) return;
    const double b = st->beta[p.j - 1];
    double s = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kVB;
    for (int64_t r = (int64_t)blockIdx.x * kVB + threadIdx.x; r < p.n; r += stride) {
        const auto v = sub(w[r], scale(vp[r], b));
        w[r] = v;
        s += real_of(conj_mul(vc[r], v));
    }
    s = block_sum<kVB>(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// w -= a v_j with a from k_lz_dot's partials;  partial_n[block] = |w|^2.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_norm(LzStep p, const typename E<C>::T* __restrict__ vc, typename E<C>::T* __restrict__ w, LzState* __restrict__ st,
          const double* __restrict__ partial, double* __restrict__ partial_n)
{
    if (st->stop) return;
    const double a = sum_partials<kVB>(partial, gridDim.x);
    if (blockIdx.x == 0 && threadIdx.x == 0) st->a = a;
    double s = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kVB;
    for (int64_t r = (int64_t)blockIdx.x * kVB + threadIdx.x; r < p.n; r += stride) {
        const auto v = sub(w[r], scale(vc[r], a));
        w[r] = v;
        s += norm2(v);
    }
    s = block_sum<kVB>(s);
    if (threadIdx.x == 0) partial_n[blockIdx.x] = s;
}

// The decision of the step (pass 1 of a step other than the first) and, if it makes
// a full pass, the dot products of w with sixteen basis vectors per grid row:
// pd[(16 y + q) nb + block] = sum conj(V_{16y+q}) w.  First step, pass 1: also
// partial_n[block] = |w|^2.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_dots(LzStep p, int pass, const typename E<C>::T* __restrict__ V, const typename E<C>::T* __restrict__ w,
          LzState* __restrict__ st, double* __restrict__ partial_n, typename E<C>::T* __restrict__ pd)
{
    using T = typename E<C>::T;
    if (st->stop) return;
    const int nb = gridDim.x;
    const bool decide = pass == 1 && !p.first;
    if (decide) {
        const double wn2 = sum_partials<kVB>(partial_n, nb);
        if (!needs_pass<C, kVB>(st, p, st->a, wn2, blockIdx.x == 0 && blockIdx.y == 0)) return;
    } else if (p.first && pass == 1 && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        st->full = 1;
        st->a = 0.0;
    }
    const bool want_norm = p.first && pass == 1 && blockIdx.y == 0;
    const int q0 = blockIdx.y * kNV, nv = p.j + 1 - q0;
    T acc[kNV];
#pragma unroll
    for (int q = 0; q < kNV; ++q) acc[q] = zero<T>();
    double nrm = 0.0;
    const T* Vq = V + (int64_t)q0 * p.n;
    const int64_t stride = (int64_t)nb * kVB;
    for (int64_t r = (int64_t)blockIdx.x * kVB + threadIdx.x; r < p.n; r += stride) {
        const T wr = w[r];
        if (want_norm) nrm += norm2(wr);
#pragma unroll
        for (int q = 0; q < kNV; ++q)
            if (q < nv) acc[q] = add2(acc[q], conj_mul(Vq[(int64_t)q * p.n + r], wr));
    }
    // per-wave sums, then the four waves in order
    __shared__ T red[kVB / 64][kNV];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < kNV; ++q) {
        T v = acc[q];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v = add2(v, shfl_xor_t(v, o));
        if (lane == 0) red[wave][q] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < kNV && (int)threadIdx.x < nv) {
        const int q = threadIdx.x;
        pd[(int64_t)(q0 + q) * nb + blockIdx.x] = add2(add2(red[0][q], red[1][q]), add2(red[2][q], red[3][q]));
    }
    if (want_norm) {
        nrm = block_sum<kVB>(nrm);
        if (threadIdx.x == 0) partial_n[blockIdx.x] = nrm;
    }
}

// coef[q] = sum over blocks of pd[q], one block per vector (fixed order); the last
// block of the first step's pass 1 sums |w|^2 instead.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_coefs(LzStep p, int pass, int nb, LzState* __restrict__ st, const double* __restrict__ partial_n,
           const typename E<C>::T* __restrict__ pd, typename E<C>::T* __restrict__ coef)
{
    using T = typename E<C>::T;
    if (st->stop || !st->full) return;
    const int q = blockIdx.x;
    if (q > p.j) {
        const double s = sum_partials<kVB>(partial_n, nb);
        if (threadIdx.x == 0) st->wn2 = s;
        return;
    }
    T s = zero<T>();
    for (int i = threadIdx.x; i < nb; i += kVB) s = add2(s, pd[(int64_t)q * nb + i]);
    __shared__ T red[kVB / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s = add2(s, shfl_xor_t(s, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        s = add2(add2(red[0], red[1]), add2(red[2], red[3]));
        coef[q] = s;
        if (q == p.j) {
            st->cdiag[pass - 1] = real_of(s);
            if (pass == 1) st->cdiag[1] = 0.0;
        }
    }
}

// After the local step, w's components along the basis are at rounding level.
// When every one of them is below skip_tol |w| the projection is skipped and the
// coefficients count as zero (the recurrence then holds for the w actually kept):
// each new vector is measured against the whole basis, so the basis stays
// orthogonal to skip_tol throughout.  What a skipped projection leaves in w the
// recurrence misses, so skip_tol is 1e-12, and 0.02 tol where that is less (with
// 1e-12 at tol = 1e-12, N=7, 2S=18 missed tol and was solved again: 239 products
// instead of 118).
// w -= sum_{i<=j} V_i coef_i unless the step has no pass or skips it;
// partial_p[block] = |w|^2 of the result.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_project(LzStep p, int may_skip, const typename E<C>::T* __restrict__ V, const typename E<C>::T* __restrict__ coef,
             typename E<C>::T* __restrict__ w, LzState* __restrict__ st, double* __restrict__ partial_p)
{
    using T = typename E<C>::T;
    if (st->stop || !st->full) return;
    __shared__ T sc[kMaxBasis];
    const int nv = p.j + 1;
    double cm = 0.0;
    for (int i = threadIdx.x; i < nv; i += kVB) {
        sc[i] = coef[i];
        cm = fmax(cm, norm2(sc[i]));
    }
    __syncthreads();
    const bool skip = may_skip && block_max<kVB>(cm) <= p.skip_tol * p.skip_tol * st->wn2;
    if (blockIdx.x == 0 && threadIdx.x == 0) st->skip = skip;
    if (skip) return;
    double nrm = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kVB;
    for (int64_t r = (int64_t)blockIdx.x * kVB + threadIdx.x; r < p.n; r += stride) {
        T acc = w[r];
        // eight vectors' loads in flight; the subtractions keep their order
        int i = 0;
        for (; i + 8 <= nv; i += 8) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = V[(int64_t)(i + u) * p.n + r];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc = sub(acc, mul(v[u], sc[i + u]));
        }
        for (; i < nv; ++i) acc = sub(acc, mul(V[(int64_t)i * p.n + r], sc[i]));
        w[r] = acc;
        nrm += norm2(acc);
    }
    nrm = block_sum<kVB>(nrm);
    if (threadIdx.x == 0) partial_p[blockIdx.x] = nrm;
}

// alpha_j, beta_j, and v_{j+1} = w / beta_j in place.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_finish(LzStep p, int second_done, typename E<C>::T* __restrict__ w, LzState* __restrict__ st,
            const double* __restrict__ partial_p)
{
    if (st->stop) return;
    const bool full = st->full != 0, skip = st->skip != 0;
    const double nrm2 = full && !skip ? sum_partials<kVB>(partial_p, gridDim.x) : 0.0;
    const LzBeta r = step_beta(st, p, full, skip, nrm2, second_done != 0);
    if (!r.stop) {
        const double s = 1.0 / r.b;
        const int64_t stride = (int64_t)gridDim.x * kVB;
        for (int64_t i = (int64_t)blockIdx.x * kVB + threadIdx.x; i < p.n; i += stride) w[i] = scale(w[i], s);
    }
    if (blockIdx.x == 0) finish_step<kVB>(st, p, r, full);
}

// A whole step after the product in one launch of one block: for a short vector
// the six launches above cost more than their work (N=6, 2S=15, dim 338: 9.4 us
// per step against 20 us).  Beyond the limits below one CU's loads make a full
// pass slower than the launches.  Solve time per product, one launch against several, us:
//   real     dim 1,656: 30 / 38, 3,788: 36 / 39, 4,370: 38 / 40, 5,744: 45 / 44, 8,512: 60 / 41
//   complex  dim   490: 28 / 41, 1,932: 39 / 45, 2,130: 41 / 46, 3,876: 54 / 46, 4,751: 63 / 50
constexpr int kSmallThreads = 1024;
// one-launch steps up to this dimension (real, complex)
constexpr int64_t kSmallReal = 4096, kSmallComplex = 2048;
template <bool C>
__global__ void __launch_bounds__(kSmallThreads)
k_lz_small(LzStep p, const typename E<C>::T* __restrict__ V, typename E<C>::T* __restrict__ w, LzState* __restrict__ st)
{
    using T = typename E<C>::T;
    constexpr int NT = kSmallThreads;
    if (st->stop) return;
    __shared__ T sc[kMaxBasis];
    const int j = p.j, n = (int)p.n, nv = j + 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const T* vc = V + (int64_t)j * n;
    bool full = true;
    double a = 0.0, wn2;
    if (p.first) {
        double s = 0.0;
        for (int r = threadIdx.x; r < n; r += NT) s += norm2(w[r]);
        wn2 = block_sum<NT>(s);
        if (threadIdx.x == 0) st->wn2 = wn2;
    } else {
        const T* vp = vc - n;
        const double b = st->beta[j - 1];
        double s = 0.0;
        for (int r = threadIdx.x; r < n; r += NT) {
            const T v = sub(w[r], scale(vp[r], b));
            w[r] = v;
            s += real_of(conj_mul(vc[r], v));
        }
        a = block_sum<NT>(s);
        s = 0.0;
        for (int r = threadIdx.x; r < n; r += NT) {
            const T v = sub(w[r], scale(vc[r], a));
            w[r] = v;
            s += norm2(v);
        }
        wn2 = block_sum<NT>(s);
        full = needs_pass<C, NT>(st, p, a, wn2, true);
    }
    LzBeta r{a, sqrt(fmax(wn2, 0.0)), 0.0, 0};
    for (int pass = 1; full && pass <= 2; ++pass) {
        __syncthreads();  // w is written, sc has been read
        for (int q = wave; q < nv; q += NT / 64) {  // a wavefront per basis vector
            const T* v = V + (int64_t)q * n;
            T s = zero<T>();
            int i = lane;
            for (; i + 192 < n; i += 256) {  // four loads of each in flight
                T x[4], y[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) x[u] = v[i + 64 * u];
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] = w[i + 64 * u];
#pragma unroll
                for (int u = 0; u < 4; ++u) s = add2(s, conj_mul(x[u], y[u]));
            }
            for (; i < n; i += 64) s = add2(s, conj_mul(v[i], w[i]));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) s = add2(s, shfl_xor_t(s, o));
            if (lane == 0) sc[q] = s;
        }
        __syncthreads();
        if (pass == 1 && !p.first) {
            double cm = 0.0;
            for (int i = threadIdx.x; i < nv; i += NT) cm = fmax(cm, norm2(sc[i]));
            if (block_max<NT>(cm) <= p.skip_tol * p.skip_tol * wn2) break;
        }
        double nrm = 0.0;
        for (int i = threadIdx.x; i < n; i += NT) {
            T acc = w[i];
            int q = 0;
            for (; q + 8 <= nv; q += 8) {
                T v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = V[(int64_t)(q + u) * n + i];
#pragma unroll
                for (int u = 0; u < 8; ++u) acc = sub(acc, mul(v[u], sc[q + u]));
            }
            for (; q < nv; ++q) acc = sub(acc, mul(V[(int64_t)q * n + i], sc[q]));
            w[i] = acc;
            nrm += norm2(acc);
        }
        nrm = block_sum<NT>(nrm);
        r.alpha += real_of(sc[j]);
        r.b = sqrt(fmax(nrm, 0.0));
        if (!p.first && !(nrm * 1e4 < wn2)) break;  // a second pass only where the first cancelled too much
    }
    r.anorm = fmax(st->anorm[j & 1], fabs(r.alpha) + r.b);
    if (r.b <= 1e-12 * fmax(r.anorm, 1e-300)) r.stop = kStopBreak;
    if (!r.stop) {
        const double f = 1.0 / r.b;
        for (int i = threadIdx.x; i < n; i += NT) w[i] = scale(w[i], f);
    }
    __syncthreads();  // every read of the state is done
    finish_step<NT>(st, p, r, full);
}

// Clears a stop, so that the host's launches for the stopped step run.
__global__ void k_lz_clear(LzState* st) { st->stop = 0; }

// After a breakdown at step j: w, a random direction orthogonalised against the
// basis (|w|^2 in partial_p), becomes v_{j+1} with beta_j = 0.
template <bool C>
__global__ void __launch_bounds__(kVB)
k_lz_fresh(LzStep p, typename E<C>::T* __restrict__ w, LzState* __restrict__ st, const double* __restrict__ partial_p)
{
    const double s = 1.0 / sqrt(fmax(sum_partials<kVB>(partial_p, gridDim.x), 0.0));
    const int64_t stride = (int64_t)gridDim.x * kVB;
    for (int64_t i = (int64_t)blockIdx.x * kVB + threadIdx.x; i < p.n; i += stride) w[i] = scale(w[i], s);
    if (blockIdx.x) return;
    if (threadIdx.x == 0) {
        st->beta[p.j] = 0.0;
        st->force[(p.j & 1) ^ 1] = 1;
    }
    for (int i = threadIdx.x; i < kMaxBasis + 2; i += kVB)
        st->om[(p.j + 1) % 3][i] = i == p.j + 1 ? 1.0 : 2.220446049250313e-16;
}

template <bool C>
__global__ void k_to_f32(int64_t dim, const typename E<C>::T* __restrict__ src, typename E<C>::F* __restrict__ dst)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < dim; r += stride)
        dst[r] = narrow(src[r]);
}

template <bool C>
__global__ void k_to_f64(int64_t dim, const typename E<C>::F* __restrict__ src, typename E<C>::T* __restrict__ dst)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < dim; r += stride)
        dst[r] = widen(src[r]);
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) counter-based generator.
HD_DEV void philox(uint32_t c[4], uint32_t k0, uint32_t k1)
{
    for (int i = 0; i < 10; ++i) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
        c[1] = (uint32_t)p1;
        c[3] = (uint32_t)p0;
        c[0] = n0;
        c[2] = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// Standard normal entries (Box-Muller on Philox uniforms); element r uses
// counter (r, stream).
template <bool C>
__global__ void k_randn(int64_t dim, uint64_t seed, uint32_t stream, typename E<C>::T* __restrict__ out)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < dim; r += stride) {
        uint32_t c[4] = {(uint32_t)r, (uint32_t)((uint64_t)r >> 32), stream, 0x5EEDu};
        philox(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        const double u1 = ((double)c[0] + 1.0) * 2.3283064365386963e-10;  // (0,1]
        const double u2 = (double)c[1] * 2.3283064365386963e-10;
        const double rad = sqrt(-2.0 * log(u1));
        const double z0 = rad * cos(6.283185307179586 * u2);
        if constexpr (C) {
            const double z1 = rad * sin(6.283185307179586 * u2);
            out[r] = make_double2(z0, z1);
        } else {
            out[r] = z0;
        }
    }
}

// partial[b] = sum |y - theta x|^2
template <bool C>
__global__ void __launch_bounds__(kVB)
k_resid(int64_t dim, const typename E<C>::T* __restrict__ y, const typename E<C>::T* __restrict__ x,
        double theta, double* __restrict__ partial)
{
    __shared__ double red[kVB];
    double s = 0.0;
    const int64_t stride = (int64_t)gridDim.x * kVB;
    for (int64_t r = (int64_t)blockIdx.x * kVB + threadIdx.x; r < dim; r += stride)
        s += norm2(sub(y[r], scale(x[r], theta)));
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = kVB / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// -------------------------------------------------------- host: Jacobi

// Symmetric eigen-decomposition of the n x n row-major matrix A (destroyed)
// by cyclic Jacobi rotations; eigenvalues ascending in w, eigenvectors as the
// columns of Z (row-major n x n).
void jacobi_eigh(int n, std::vector<double>& A, std::vector<double>& w, std::vector<double>& Z)
{
    Z.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; ++i) Z[(size_t)i * n + i] = 1.0;
    auto a = [&](int i, int j) -> double& { return A[(size_t)i * n + j]; };
    for (int sweep = 0; sweep < 100; ++sweep) {
        double off = 0.0, tot = 0.0;
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < n; ++j) {
                tot += a(i, j) * a(i, j);
                if (i != j) off += a(i, j) * a(i, j);
            }
        if (off <= 1e-34 * tot || off == 0.0) break;
        for (int p = 0; p < n - 1; ++p)
            for (int q = p + 1; q < n; ++q) {
                const double apq = a(p, q);
                if (std::fabs(apq) < 1e-300) continue;
                const double theta = (a(q, q) - a(p, p)) / (2.0 * apq);
                const double t = (theta >= 0 ? 1.0 : -1.0) / (std::fabs(theta) + std::sqrt(theta * theta + 1.0));
                const double c = 1.0 / std::sqrt(t * t + 1.0), s = t * c;
                for (int k = 0; k < n; ++k) {
                    const double akp = a(k, p), akq = a(k, q);
                    a(k, p) = c * akp - s * akq;
                    a(k, q) = s * akp + c * akq;
                }
                for (int k = 0; k < n; ++k) {
                    const double apk = a(p, k), aqk = a(q, k);
                    a(p, k) = c * apk - s * aqk;
                    a(q, k) = s * apk + c * aqk;
                }
                for (int k = 0; k < n; ++k) {
                    const double zkp = Z[(size_t)k * n + p], zkq = Z[(size_t)k * n + q];
                    Z[(size_t)k * n + p] = c * zkp - s * zkq;
                    Z[(size_t)k * n + q] = s * zkp + c * zkq;
                }
            }
    }
    std::vector<int> idx(n);
    std::iota(idx.begin(), idx.end(), 0);
    std::sort(idx.begin(), idx.end(), [&](int x, int y) { return a(x, x) < a(y, y); });
    w.resize(n);
    std::vector<double> Zs((size_t)n * n);
    for (int c = 0; c < n; ++c) {
        w[c] = a(idx[c], idx[c]);
        for (int r = 0; r < n; ++r) Zs[(size_t)r * n + c] = Z[(size_t)r * n + idx[c]];
    }
    Z.swap(Zs);
}

// ------------------------------------------------------------ host driver

template <bool C>
struct Lanczos {
    using T = typename E<C>::T;
    using F = typename E<C>::F;
    hd_hamiltonian* h;
    hipStream_t st;
    int64_t n;
    int m;
    int nb;  // blocks of the vector kernels
    T* V = nullptr;     // (m+1) x n
    T* V2 = nullptr;    // the other basis buffer: a restart writes there, then they swap
    T* ritz = nullptr;  // nev Ritz vectors, handed to the handle at the end
    F* x32 = nullptr;
    F* y32 = nullptr;
    LzState* dst = nullptr;
    double *pa = nullptr, *pn = nullptr, *pp = nullptr;  // per-block partials
    T* pd = nullptr;    // per-block dot products
    T* coef = nullptr;
    double* dscal = nullptr;
    double* dY = nullptr;
    int mv32 = 0, mv64 = 0;
    int prec64 = HD_F64;  // the FP64 operator: FP64 values or the coded format
    // Event triples (before and after a product, after the step's pass) of timed
    // steps, read when the host waits anyway.  Long vectors: every step; short
    // ones, where an event costs as much as a kernel: one in sixteen.
    std::vector<hipEvent_t> ev;
    std::vector<int> ev_step;  // the step of each triple
    size_t ev_used = 0;
    double ms_spmv = 0, ms_ortho = 0;
    int timed = 0, steps = 0;
    hipError_t ev_err = hipSuccess;

    ~Lanczos()
    {
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        dfree(V); dfree(V2); dfree(ritz); dfree(x32); dfree(y32); dfree(dst); dfree(pa); dfree(pn); dfree(pp); dfree(pd);
        dfree(coef); dfree(dscal); dfree(dY);
    }

    int alloc(bool need_x32, bool need_y32)
    {
        HD_CHECK(dalloc_t(&V, (size_t)(m + 1) * n, "Lanczos basis"));
        HD_CHECK(dalloc_t(&V2, (size_t)(m + 1) * n, "restart buffer"));
        if (need_x32) HD_CHECK(dalloc_t(&x32, (size_t)n, "FP32 x"));
        if (need_y32) HD_CHECK(dalloc_t(&y32, (size_t)n, "FP32 y"));
        HD_CHECK(dalloc_t(&dst, 1, "Lanczos state"));
        HD_CHECK(dalloc_t(&pa, (size_t)nb, "dot partials"));
        HD_CHECK(dalloc_t(&pn, (size_t)nb, "norm partials"));
        HD_CHECK(dalloc_t(&pp, (size_t)nb, "norm partials"));
        HD_CHECK(dalloc_t(&pd, (size_t)(m + kNV) * nb, "basis dot partials"));
        HD_CHECK(dalloc_t(&coef, kMaxBasis, "coefficients"));
        HD_CHECK(dalloc_t(&dscal, 4, "scalars"));
        HD_CHECK(dalloc_t(&dY, (size_t)kMaxBasis * kMaxBasis, "Ritz coefficients"));
        return HD_OK;
    }

    T* vec(int j) { return V + (size_t)j * n; }

    void mark(bool on)
    {
        if (!on || ev_err != hipSuccess) return;
        if (ev_used == ev.size()) {
            hipEvent_t e = nullptr;
            ev_err = hipEventCreate(&e);
            if (ev_err != hipSuccess) return;
            ev.push_back(e);
        }
        ev_err = hipEventRecord(ev[ev_used++], st);
    }

    // Adds up the marked steps up to `last` (those queued behind a stop did nothing after
    // their product); the stream has been waited for.
    int read_marks(int last)
    {
        for (size_t i = 0; i + 2 < ev_used && ev_err == hipSuccess; i += 3) {
            if (ev_step[i / 3] > last) break;
            float a = 0.f, b = 0.f;
            ev_err = hipEventElapsedTime(&a, ev[i], ev[i + 1]);
            if (ev_err == hipSuccess) ev_err = hipEventElapsedTime(&b, ev[i + 1], ev[i + 2]);
            ms_spmv += a;
            ms_ortho += b;
            ++timed;
        }
        ev_used = 0;
        ev_step.clear();
        return ev_err == hipSuccess ? HD_OK
                                    : fail(HD_ERR_HIP, std::string("Lanczos timing: ") + hipGetErrorString(ev_err));
    }

    // y = H x in the requested precision (enqueued)
    int apply(const T* x, T* y, int prec)
    {
        if (prec != HD_F32 && prec != HD_TILED_X32) {
            ++mv64;
            return spmv_launch(h, prec, x, y, st);
        }
        ++mv32;
        hipLaunchKernelGGL(k_to_f32<C>, dim3(nb), dim3(kVB), 0, st, n, x, x32);
        if (prec == HD_TILED_X32) return spmv_launch(h, HD_TILED_X32, x32, y, st);
        HD_CHECK(spmv_launch(h, HD_F32, x32, y32, st));
        hipLaunchKernelGGL(k_to_f64<C>, dim3(nb), dim3(kVB), 0, st, n, y32, y);
        return HD_OK;
    }

    // The Ritz vectors; where there is no room beside those of the handle's last solve,
    // in their place.
    int alloc_ritz(int nev)
    {
        if (ritz) return HD_OK;
        int rc = dalloc_t(&ritz, (size_t)nev * n, "eigenvectors");
        if (rc == HD_ERR_NOMEM && h->lz && h->lz->d_vec) {
            dfree(h->lz->d_vec);
            h->lz->d_vec = nullptr;
            rc = dalloc_t(&ritz, (size_t)nev * n, "eigenvectors");
        }
        return rc;
    }

    // one Gram-Schmidt pass of w against V[0..j] (enqueued; the kernels decide)
    void pass(const LzStep& p, int number, bool may_skip, T* w)
    {
        const int groups = (p.j + 1 + kNV - 1) / kNV;
        hipLaunchKernelGGL(k_lz_dots<C>, dim3(nb, groups), dim3(kVB), 0, st, p, number, V, w, dst, pn, pd);
        hipLaunchKernelGGL(k_lz_coefs<C>, dim3(p.j + 1 + (p.first && number == 1)), dim3(kVB), 0, st, p, number, nb, dst,
                           pn, pd, coef);
        hipLaunchKernelGGL(k_lz_project<C>, dim3(nb), dim3(kVB), 0, st, p, may_skip ? 1 : 0, V, coef, w, dst, pp);
    }

    // Step j (enqueued): the product into vec(j + 1), the local three-term part
    // (before the pass, so that its large coefficients never multiply the basis'
    // own orthogonality error, which a single classical Gram-Schmidt pass would
    // amplify by alpha/beta per step), the full pass where one is due, the scaling.
    // A pass is one of classical Gram-Schmidt, and a second one only when the
    // first cancelled more than a factor 100 of the norm (the "twice is enough"
    // test of Daniel, Gragg, Kaufman and Stewart, Math. Comp. 30 (1976) 772),
    // or always in the first step of a cycle.
    int step(int j, int k, int prec, bool must, double eps_op, double om_cycle, double skip_tol)
    {
        const bool timing = n >= 65536 || steps % 16 == 0;
        ++steps;
        T* w = vec(j + 1);
        if (timing) ev_step.push_back(j);
        mark(timing);
        HD_CHECK(apply(vec(j), w, prec));
        mark(timing);
        const LzStep p{n, j, k, j == k, must, eps_op, om_cycle, skip_tol};
        if (n <= (C ? kSmallComplex : kSmallReal)) {
            hipLaunchKernelGGL(k_lz_small<C>, dim3(1), dim3(kSmallThreads), 0, st, p, V, w, dst);
        } else {
            if (!p.first) {
                hipLaunchKernelGGL(k_lz_dot<C>, dim3(nb), dim3(kVB), 0, st, p, vec(j - 1), vec(j), w, dst, pa);
                hipLaunchKernelGGL(k_lz_norm<C>, dim3(nb), dim3(kVB), 0, st, p, vec(j), w, dst, pa, pn);
            }
            pass(p, 1, !p.first, w);
            if (p.first) pass(p, 2, false, w);
            hipLaunchKernelGGL(k_lz_finish<C>, dim3(nb), dim3(kVB), 0, st, p, p.first, w, dst, pp);
        }
        mark(timing);
        HD_HIP(hipGetLastError());
        return HD_OK;
    }

    // The host part of a stopped step: the second pass, or a fresh direction after
    // a breakdown.
    int resume(int j, int why, uint64_t seed, uint32_t* rng_stream)
    {
        T* w = vec(j + 1);
        hipLaunchKernelGGL(k_lz_clear, dim3(1), dim3(1), 0, st, dst);
        if (why == kStopSecond) {
            const LzStep p{n, j, -1, 0, 1, 0.0, 0.0, 0.0};
            pass(p, 2, false, w);
            hipLaunchKernelGGL(k_lz_finish<C>, dim3(nb), dim3(kVB), 0, st, p, 1, w, dst, pp);
        } else {
            const LzStep p{n, j, -1, 1, 1, 0.0, 0.0, 0.0};
            HD_CHECK(random_start(seed, (*rng_stream)++, w));
            pass(p, 1, false, w);
            pass(p, 2, false, w);
            hipLaunchKernelGGL(k_lz_fresh<C>, dim3(nb), dim3(kVB), 0, st, p, w, dst, pp);
        }
        HD_HIP(hipGetLastError());
        return HD_OK;
    }

    // Waits for the enqueued steps and reads the part of the state before theta.
    int read_state(LzState* out)
    {
        HD_HIP(hipMemcpyAsync(out, dst, offsetof(LzState, theta), hipMemcpyDeviceToHost, st));
        HD_HIP(hipStreamSynchronize(st));
        return read_marks(out->stop ? out->stop_step : m);
    }

    int scale_into(const T* src, double s, T* dst_)
    {
        hipLaunchKernelGGL(k_scale<C>, dim3(nb), dim3(kVB), 0, st, n, src, s, dst_);
        HD_HIP(hipGetLastError());
        return HD_OK;
    }

    // out[0..kk) = V[0..mm) Y[:, 0..kk)  (Y row-major mm x ldy on the host)
    int combine(int mm, const std::vector<double>& Y, int ldy, int kk, T* out)
    {
        HD_HIP(hipMemcpyAsync(dY, Y.data(), sizeof(double) * mm * ldy, hipMemcpyHostToDevice, st));
        // real vectors: up to 32 outputs per pass over the basis; complex: 16
        constexpr int NL = C ? 16 : 32;
        for (int l0 = 0; l0 < kk; l0 += NL) {
            const int nl = std::min(NL, kk - l0);
            hipLaunchKernelGGL((k_combine<C, NL>), dim3(nb), dim3(kVB), sizeof(double) * mm * nl, st, n, V, n, mm, dY,
                               ldy, l0, nl, out + (size_t)l0 * n);
        }
        HD_HIP(hipGetLastError());
        HD_HIP(hipStreamSynchronize(st));  // Y may change from here on
        return HD_OK;
    }

    int random_start(uint64_t seed, uint32_t stream_id, T* out)
    {
        hipLaunchKernelGGL(k_randn<C>, dim3(nb), dim3(kVB), 0, st, n, seed, stream_id, out);
        HD_HIP(hipGetLastError());
        return HD_OK;
    }

    // |y - theta x|
    int residual_norm(const T* y, const T* x, double theta, double* out)
    {
        hipLaunchKernelGGL(k_resid<C>, dim3(nb), dim3(kVB), 0, st, n, y, x, theta, pp);
        hipLaunchKernelGGL(k_reduce_real, dim3(1), dim3(kVB), 0, st, pp, nb, dscal);
        HD_HIP(hipGetLastError());
        HD_HIP(hipMemcpyAsync(out, dscal, sizeof(double), hipMemcpyDeviceToHost, st));
        HD_HIP(hipStreamSynchronize(st));
        *out = std::sqrt(std::max(*out, 0.0));
        return HD_OK;
    }
};

template <bool C>
static int run_lanczos(hd_hamiltonian* h, const hd_lanczos_opts& o, double* evals, hd_lanczos_stats* stats)
{
    using T = typename E<C>::T;
    const auto t_start = std::chrono::steady_clock::now();
    Lanczos<C> L;
    L.h = h;
    L.st = h->stream;
    L.n = h->dim;
    const int nev = (int)std::min<int64_t>(o.nev, h->dim);
    int m = o.ncv > 0 ? o.ncv : 2 * nev + 21;
    m = (int)std::min<int64_t>(m, h->dim);
    m = std::min(m, kMaxBasis);
    if (m < nev + 2) return fail(HD_ERR_ARG, "ncv must be at least nev + 2 (and dim > nev + 1)");
    L.m = m;
    int n_cu = 256;
    HD_CHECK(device_props(&n_cu, nullptr));
    L.nb = (int)std::max<int64_t>(1, std::min<int64_t>((h->dim + kVB - 1) / kVB, (int64_t)n_cu * 4));
    const bool mixed = o.precision == HD_F32;
    // the FP32-input operator of the mixed solve: the tiled layout with FP32 x
    // (exact for FP32 inputs), else the FP32-value CRS (FP32 accumulation)
    const int prec32 = (h->d_tg_base && !h->is_complex) ? HD_TILED_X32 : HD_F32;
    if (mixed && prec32 == HD_F32 && !h->d_val32)
        return fail(HD_ERR_ARG, "FP32 Lanczos needs FP32 values (value_mask & 2) or a real tiled layout");
    const bool free_ = h->storage == HD_STORAGE_MATRIX_FREE;
    if (!free_ && !h->d_val64 && !h->d_code && !h->d_tg_base)
        return fail(HD_ERR_ARG, "Lanczos needs FP64, coded or tiled values for the FP64 operator");
    if (o.precision == HD_TILED && !h->d_tg_base) return fail(HD_ERR_ARG, "no tiled layout (hd_ham_tile)");
    if (o.precision < HD_F64 || o.precision > HD_TILED) return fail(HD_ERR_ARG, "unknown Lanczos precision");
    // the exact FP64 operator: the tiled layout when asked for (or, in a mixed
    // solve, when built: it is the fastest exact one), else FP64 values, else coded
    L.prec64 = free_ ? HD_F64
               : (o.precision == HD_TILED || (mixed && h->d_tg_base)) ? HD_TILED
               : (o.precision == HD_CODED || !h->d_val64) ? (h->d_code ? HD_CODED : HD_TILED)
                                                          : HD_F64;
    // a long solve times the schedules of the CRS formats that it uses
    int untuned = 0;
    for (int p : {L.prec64, mixed ? prec32 : L.prec64})
        if (p < HD_TILED) untuned |= 1 << p;
    untuned &= ~h->sched_chosen;
    if (!free_ && untuned && h->nnz >= kLongNnz) HD_CHECK(spmv_autotune(h, untuned));
    HD_CHECK(L.alloc(mixed, mixed && prec32 == HD_F32));
    const double tol = o.tol > 0 ? o.tol : 1e-10;
    const double budget = o.f32_budget > 0 ? std::min(o.f32_budget, 1.0) : 1.0;
    // relative rounding of one FP32-input product: x rounded to FP32, plus
    // FP32 values and accumulation over a row for the CRS form
    const double u32 = 5.9604644775390625e-8;  // 2^-24
    const double eps32 = prec32 == HD_TILED_X32 ? u32 : u32 * (1.0 + std::sqrt((double)std::max<int64_t>(h->max_row, 1)));
    const int max_restarts = o.max_restarts > 0 ? o.max_restarts : 2000;
    int prec = L.prec64;
    // HD_LANCZOS_TRACE=1: one line per restart cycle on stderr
    const char* trace_env = std::getenv("HD_LANCZOS_TRACE");
    const bool trace = trace_env && trace_env[0] == '1';
    int kk_keep = nev + (m - nev) / 2;
    kk_keep = std::min(std::max(kk_keep, nev + 1), m - 2 >= nev ? m - 2 : nev);
    kk_keep = std::max(kk_keep, nev);

    // start vector
    if (o.start == HD_START_USER) {
        if (!o.d_start) return fail(HD_ERR_ARG, "HD_START_USER needs d_start");
        HD_HIP(hipMemcpyAsync(L.vec(0), o.d_start, sizeof(T) * L.n, hipMemcpyDeviceToDevice, L.st));
    } else {
        HD_CHECK(L.random_start(o.seed, 0u, L.vec(0)));
    }
    uint32_t rng_stream = 1;
    double nrm;
    HD_CHECK(L.residual_norm(L.vec(0), L.vec(0), 0.0, &nrm));
    if (!(nrm > 0)) return fail(HD_ERR_ARG, "start vector is zero");
    HD_CHECK(L.scale_into(L.vec(0), 1.0 / nrm, L.vec(0)));

    auto hs = std::make_unique<LzState>();  // host copy of the device state
    std::memset(static_cast<void*>(hs.get()), 0, sizeof(LzState));
    const double *alpha = hs->alpha, *beta = hs->beta;
    std::vector<double> theta, arrow;
    std::vector<double> Tm, w, Y;
    int k = 0;  // kept Ritz vectors at the head of V
    int restarts = 0;
    bool converged = false;
    std::vector<double> res_est(m, 0.0);
    double anorm = 0.0;
    // Partial reorthogonalisation (H. D. Simon, Math. Comp. 42 (1984) 115): the
    // overlaps of the new vector are propagated by the recurrence the basis obeys,
    // A V = V T + rounding, with T the arrow of the kept Ritz pairs followed by the
    // tridiagonal of the cycle (needs_pass); a new vector is orthogonalised against
    // the whole basis only when an estimate exceeds the threshold, and then the next
    // one too (its recurrence still holds the old error).  The first vector of a
    // cycle (the arrow) and the last (which becomes the next cycle's first) are
    // always orthogonalised, so every cycle starts from an orthogonal pair.
    const bool pro = o.full_reorth == 0;
    const double eps = std::numeric_limits<double>::epsilon();
    // a pass removes coefficients of the size of the estimates, which the
    // recurrence (and so the Ritz vectors' residuals) then misses: keeping them
    // below a quarter of tol keeps that part of the residuals below tol
    // (semi-orthogonality, sqrt(eps), at most).  With tol itself as the threshold
    // some solves ended with such a part of 0.3 to 1 tol and were run again
    // (207 products became 414 on one parameter point of N=12, 2S=33).
    const double om_max = std::min(std::sqrt(eps), 0.25 * (o.tol > 0 ? o.tol : 1e-10));
    // mixed precision: bound of the rounding each wanted pair has taken from
    // FP32 cycles, and its coefficient norm on the previous cycle's new vectors
    std::vector<double> err32(nev, 0.0), nb_prev(nev, 1.0);
    // An FP32 cycle is speculative: when the cycle's own coefficients put a wanted
    // pair's rounding estimate beyond the budget (a pair that entered the wanted
    // window during the cycle carries O(1) coefficients on its vectors), the cycle
    // is discarded and run again with the FP64 operator.  The vectors it started
    // from are still there: a cycle only writes behind them.
    std::vector<double> err32_b, nb_prev_b;
    int rollbacks = 0;
    // Projected matrix of the first n basis vectors: diag(theta) + arrow at row
    // k, tridiagonal below.
    auto projected = [&](int n) {
        Tm.assign((size_t)n * n, 0.0);
        for (int i = 0; i < k; ++i) {
            Tm[(size_t)i * n + i] = theta[i];
            Tm[(size_t)i * n + k] = Tm[(size_t)k * n + i] = arrow[i];
        }
        for (int j = k; j < n; ++j) {
            Tm[(size_t)j * n + j] = alpha[j];
            if (j + 1 < n) Tm[(size_t)j * n + j + 1] = Tm[(size_t)(j + 1) * n + j] = beta[j];
        }
    };
    // Convergence inside a cycle: once the previous cycle ended with every
    // wanted Ritz estimate within 1e4 tol, the Ritz pairs of the basis built so
    // far are tested after each step (a (j+1)-square eigenproblem on the host, of
    // which the test needs the eigenvectors' last row only), and the cycle ends at
    // the first step where all wanted pairs meet tol.  An FP32 cycle ends there
    // only if its rounding estimate stays in the budget.  A short vector's steps
    // are enqueued four at a time: a step costs less than the wait for it.
    double r_prev = std::numeric_limits<double>::infinity();
    // The estimates miss what partial reorthogonalisation leaves in the residual (a
    // fraction of tol).  When an explicit residual misses tol although its estimate
    // met it, the estimates have to meet half as much from there on, and the cycle
    // goes on: a few more steps instead of the whole solve again.  (Not where the
    // missed part alone is at tol: more steps do not reduce that.)
    double tol_est = tol;
    int missed = 0;
    int mc = m;  // basis size at which the current cycle ends
    auto ends_at = [&](int n1, bool cyc32) {
        projected(n1);
        if (!sym_eig(n1, Tm, w, Y, n1 - 1)) return false;
        for (int i = 0; i < nev; ++i)
            if (!(std::fabs(beta[n1 - 1] * Y[i]) / std::max(1.0, std::fabs(w[i])) <= tol_est)) return false;
        if (!cyc32) return true;
        projected(n1);
        if (!sym_eig(n1, Tm, w, Y)) return false;
        for (int i = 0; i < nev; ++i) {
            double nb2 = 0.0;
            for (int jj = k; jj < n1; ++jj) nb2 += Y[(size_t)jj * n1 + i] * Y[(size_t)jj * n1 + i];
            if (err32[i] + eps32 * anorm * std::sqrt(nb2) > budget * tol * std::max(1.0, std::fabs(w[i]))) return false;
        }
        return true;
    };
    // Ritz vectors of the first mc basis vectors, and their FP64 residuals (V2 is
    // free between restarts)
    std::vector<double> resid(nev, 0.0);
    int nconv = 0;
    auto ritz_pairs = [&]() -> int {
        HD_CHECK(L.alloc_ritz(nev));
        HD_CHECK(L.combine(mc, Y, mc, nev, L.ritz));
        nconv = 0;
        for (int i = 0; i < nev; ++i) {
            T* xi = L.ritz + (size_t)i * L.n;
            HD_CHECK(L.apply(xi, L.V2, L.prec64));
            double r;
            HD_CHECK(L.residual_norm(L.V2, xi, w[i], &r));
            r /= std::max(1.0, std::fabs(w[i]));
            if (trace) std::fprintf(stderr, "[hd_lanczos] pair %d: theta %.15g FP64 residual %.3e (Ritz estimate %.3e)\n", i, w[i], r, res_est[i]);
            resid[i] = r;
            if (r <= tol) ++nconv;
        }
        return HD_OK;
    };
    // Steps enqueued before the host looks for a stop.  The products of the steps queued
    // behind a stop are lost, so after one the steps go singly and then twice as many each
    // time: a matrix of few distinct eigenvalues stops at every few steps (constant
    // pseudopotentials, N=10, 2S=27: 85 products with whole cycles, 30 needed).  Long
    // vectors begin that way, and from 2^20 entries on, where four steps take a hundred
    // times the wait, no more than four are queued.
    const int chunk_max = L.n >= (1 << 20) ? 4 : m;
    int chunk = L.n >= 65536 ? 2 : m;
    int done = 0;         // steps of the current cycle whose coefficients are here
    int tested = 0;       // basis sizes tested so far
    bool fresh = true;    // the next pass of the loop begins a cycle
    for (;;) {
        const bool cyc32 = prec == prec32 && mixed;
        const bool check_in_cycle = r_prev <= 1e4 * tol;
        if (fresh) {
            if (cyc32) {
                err32_b = err32;
                nb_prev_b = nb_prev;
            }
            hs->stop = hs->force[0] = hs->force[1] = 0;
            hs->anorm[0] = hs->anorm[1] = anorm;
            std::copy(theta.begin(), theta.end(), hs->theta);
            std::copy(arrow.begin(), arrow.end(), hs->arrow);
            HD_HIP(hipMemcpyAsync(L.dst, hs.get(), sizeof(LzState), hipMemcpyHostToDevice, L.st));
            done = k;
            tested = k;
            fresh = false;
        }
        // A rounding error of the FP32-input product is a vector A*delta with
        // delta ~ eps32 |x| spread over the sector: its overlap with a basis
        // vector is ~ eps32 |A| / sqrt(dim).  Such a cycle tolerates overlaps up
        // to eps32 (counted in err32 below).
        const double eps_op = cyc32 ? eps + eps32 / std::sqrt((double)std::max<int64_t>(L.n, 1)) : eps;
        const double om_cycle = cyc32 ? std::max(om_max, eps32) : om_max;
        mc = m;
        for (;;) {
            bool ended = false;
            if (check_in_cycle)
                for (int n1 = tested + 1; n1 <= done && !ended; ++n1) {
                    tested = n1;
                    if (n1 < m && n1 > k + 1 && n1 >= nev && beta[n1 - 1] > 0.0 && ends_at(n1, cyc32)) {
                        mc = n1;
                        ended = true;
                    }
                }
            if (ended || done >= m) break;
            const int upto = std::min(m, done + std::min(chunk, check_in_cycle ? (L.n >= 65536 ? 1 : 4) : m));
            for (int j = done; j < upto; ++j)
                HD_CHECK(L.step(j, k, prec, !pro || j == m - 1, eps_op, om_cycle, std::min(1e-12, 0.02 * tol)));
            HD_CHECK(L.read_state(hs.get()));
            chunk = hs->stop ? 1 : std::min(2 * chunk, chunk_max);
            if (hs->stop) {
                HD_CHECK(L.resume(hs->stop_step, hs->stop, o.seed, &rng_stream));
                done = hs->stop_step + 1;
                HD_CHECK(L.read_state(hs.get()));
                if (hs->stop) {  // the second pass cancelled the vector
                    HD_CHECK(L.resume(hs->stop_step, kStopBreak, o.seed, &rng_stream));
                    HD_CHECK(L.read_state(hs.get()));
                }
            } else {
                done = upto;
            }
            anorm = hs->anorm[done & 1];
        }
        projected(mc);
        if (!sym_eig(mc, Tm, w, Y)) return fail(HD_ERR_NOT_CONVERGED, "projected eigenproblem did not converge");
        const double bm = beta[mc - 1];
        bool all = true;
        bool allow32 = mixed;
        bool overshoot = false;
        for (int i = 0; i < nev; ++i) {
            const double scale_i = std::max(1.0, std::fabs(w[i]));
            res_est[i] = std::fabs(bm * Y[(size_t)(mc - 1) * mc + i]) / scale_i;
            if (mixed) {
                // the wanted Ritz vector's coefficients on this cycle's new vectors
                double nb2 = 0.0;
                for (int j = k; j < mc; ++j) nb2 += Y[(size_t)j * mc + i] * Y[(size_t)j * mc + i];
                const double nb = std::sqrt(nb2);
                if (cyc32) {
                    err32[i] += eps32 * anorm * nb;
                    if (err32[i] > budget * tol * scale_i) overshoot = true;
                }
                // the next cycle's coefficients, predicted from this cycle's decrease
                const double pred = nb * std::min(1.0, nb / std::max(nb_prev[i], 1e-300));
                nb_prev[i] = nb;
                if (err32[i] + eps32 * anorm * pred > budget * tol * scale_i) allow32 = false;
            }
            if (!(res_est[i] <= tol_est)) all = false;
        }
        r_prev = 0.0;
        for (int i = 0; i < nev; ++i) r_prev = std::max(r_prev, res_est[i]);
        ++restarts;
        if (trace) {
            double rmax = 0.0, emax = 0.0;
            for (int i = 0; i < nev; ++i) {
                rmax = std::max(rmax, res_est[i]);
                emax = std::max(emax, err32[i] / std::max(1.0, std::fabs(w[i])));
            }
            std::fprintf(stderr, "[hd_lanczos] cycle %d op %d k %d ritz-resid %.3e fp32-err %.3e next-fp32 %d anorm %.3e full-passes %d%s\n",
                         restarts, prec, k, rmax, emax, (int)(mixed && allow32 && !overshoot), anorm, hs->reorth,
                         overshoot ? " (discarded: run again in FP64)" : "");
        }
        if (overshoot) {
            err32 = err32_b;
            nb_prev = nb_prev_b;
            prec = L.prec64;
            ++rollbacks;
            if (restarts >= max_restarts) break;
            fresh = true;
            continue;
        }
        // A basis of the whole space has nothing to continue with (vec(mc) is rounding
        // noise): its pairs are the answer, whatever their residuals.
        const bool spans = mc >= L.n;
        if (all || spans) {
            HD_CHECK(ritz_pairs());
            bool hopeless = missed == 3 || spans;
            for (int i = 0; i < nev; ++i)
                if (missed && resid[i] * resid[i] - res_est[i] * res_est[i] > tol * tol) hopeless = true;
            if (nconv == nev || hopeless || restarts >= max_restarts) {
                converged = true;
                break;
            }
            ++missed;
            tol_est *= 0.5;
            if (mc < m) {  // the same cycle goes on
                if (cyc32) {
                    err32 = err32_b;
                    nb_prev = nb_prev_b;
                }
                --restarts;
                continue;
            }
        }
        if (restarts >= max_restarts) break;
        // thick restart: keep kk Ritz vectors, continue from the residual direction
        const int kk = kk_keep;
        HD_CHECK(L.combine(mc, Y, mc, kk, L.V2));
        HD_HIP(hipMemcpyAsync(L.V2 + (size_t)kk * L.n, L.vec(mc), sizeof(T) * L.n, hipMemcpyDeviceToDevice, L.st));
        std::swap(L.V, L.V2);
        theta.assign(w.begin(), w.begin() + kk);
        arrow.resize(kk);
        for (int i = 0; i < kk; ++i) arrow[i] = bm * Y[(size_t)(mc - 1) * mc + i];
        k = kk;
        if (mixed) prec = allow32 ? prec32 : L.prec64;
        fresh = true;
    }
    if (!converged) HD_CHECK(ritz_pairs());
    hd_lanczos_state* S = h->lz;
    if (!S) S = h->lz = new hd_lanczos_state();
    dfree(S->d_vec);
    S->d_vec = L.ritz;
    L.ritz = nullptr;
    S->dim = L.n;
    S->cplx = C;
    S->nev = nev;
    S->evals.assign(w.begin(), w.begin() + nev);
    for (int i = 0; i < nev; ++i) evals[i] = w[i];
    if (stats)
        for (int i = 0; i < 64; ++i) stats->residual[i] = i < nev ? resid[i] : 0.0;
    if (stats) {
        stats->converged = converged && nconv == nev;
        stats->nconv = nconv;
        stats->restarts = restarts;
        stats->matvecs = L.mv32 + L.mv64;
        stats->matvecs_f32 = L.mv32;
        stats->matvecs_f64 = L.mv64;
        // the timed steps' mean over all products and steps
        stats->time_spmv_ms = L.timed ? L.ms_spmv / L.timed * (L.mv32 + L.mv64) : 0.0;
        stats->time_ortho_ms = L.timed ? L.ms_ortho / L.timed * L.steps : 0.0;
        stats->reorth_steps = hs->reorth;
        stats->f32_cycles_discarded = rollbacks;
        stats->time_total_ms =
            std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
    }
    if (!converged) return fail(HD_ERR_NOT_CONVERGED, "Lanczos reached the restart limit before tol");
    return HD_OK;
}

}  // namespace hd

using namespace hd;

extern "C" {

int hd_lanczos(hd_hamiltonian* h, const hd_lanczos_opts* opts, double* h_evals, hd_lanczos_stats* stats)
{
    if (!h || !opts || !h_evals) return fail(HD_ERR_ARG, "hd_lanczos: null argument");
    if (opts->nev <= 0) return fail(HD_ERR_ARG, "nev must be positive");
    if (h->storage != HD_STORAGE_FULL && h->storage != HD_STORAGE_MATRIX_FREE)
        return fail(HD_ERR_ARG, "Lanczos needs full or matrix-free storage");
    if (h->storage == HD_STORAGE_MATRIX_FREE && (opts->precision != HD_F64 || opts->block > 1))
        return fail(HD_ERR_ARG, "matrix-free storage runs the single-vector Lanczos in FP64 (precision HD_F64)");
    if (opts->block > 1) {
        return run_block_lanczos(h, *opts, h_evals, stats);
    }
    auto run = [&](const hd_lanczos_opts& o, hd_lanczos_stats* s) {
        return h->is_complex ? run_lanczos<true>(h, o, h_evals, s) : run_lanczos<false>(h, o, h_evals, s);
    };
    hd_lanczos_stats s1{};
    const int rc = run(*opts, &s1);
    const bool mixed = opts->precision == HD_F32;
    if ((rc != HD_OK && rc != HD_ERR_NOT_CONVERGED) || s1.converged || (opts->full_reorth && !mixed)) {
        if (stats) *stats = s1;
        return rc;
    }
    // the Ritz estimates met tol but an explicit FP64 residual did not: solve
    // again with the FP64 operator (mixed precision) or with full
    // reorthogonalisation (partial reorthogonalisation)
    hd_lanczos_opts o2 = *opts;
    if (mixed) o2.precision = h->d_tg_base ? HD_TILED : (h->d_val64 ? HD_F64 : HD_CODED);
    else o2.full_reorth = 1;
    hd_lanczos_stats s2{};
    const int rc2 = run(o2, &s2);
    s2.matvecs += s1.matvecs;
    s2.matvecs_f32 += s1.matvecs_f32;
    s2.matvecs_f64 += s1.matvecs_f64;
    s2.restarts += s1.restarts;
    s2.reorth_steps += s1.reorth_steps;
    s2.f32_cycles_discarded += s1.f32_cycles_discarded;
    s2.time_total_ms += s1.time_total_ms;
    s2.time_spmv_ms += s1.time_spmv_ms;
    s2.time_ortho_ms += s1.time_ortho_ms;
    if (stats) *stats = s2;
    return rc2;
}

int hd_lanczos_vectors(const hd_hamiltonian* h, int32_t i, void* d_out, void* h_out)
{
    if (!h || !h->lz || !h->lz->d_vec) return fail(HD_ERR_ARG, "no Lanczos result on this handle");
    if (i < 0 || i >= h->lz->nev) return fail(HD_ERR_ARG, "eigenvector index out of range");
    const size_t es = 8 * (h->lz->cplx ? 2 : 1);
    const char* src = static_cast<const char*>(h->lz->d_vec) + (size_t)i * h->lz->dim * es;
    if (d_out) HD_HIP(hipMemcpy(d_out, src, h->lz->dim * es, hipMemcpyDeviceToDevice));
    else if (h_out) HD_HIP(hipMemcpy(h_out, src, h->lz->dim * es, hipMemcpyDeviceToHost));
    else return fail(HD_ERR_ARG, "no output buffer");
    return HD_OK;
}

int hd_full_diagonalize(hd_hamiltonian* h, int32_t nev, double* h_evals)
{
    if (!h || !h_evals || nev <= 0) return fail(HD_ERR_ARG, "hd_full_diagonalize: bad argument");
    if (h->is_complex) return fail(HD_ERR_UNSUPPORTED, "dense fallback handles real matrices; use hd_lanczos");
    if (h->dim > 4096) return fail(HD_ERR_ARG, "dense fallback limited to dim <= 4096");
    const int64_t n = h->dim;
    std::vector<int64_t> rp(n + 1);
    std::vector<int32_t> col((size_t)h->nnz);
    std::vector<double> val((size_t)h->nnz);
    HD_CHECK(hd_ham_copy_crs(h, 0, n, HD_F64, rp.data(), col.data(), val.data()));
    std::vector<double> A((size_t)n * n, 0.0), w, Z;
    for (int64_t i = 0; i < n; ++i)
        for (int64_t j = rp[i]; j < rp[i + 1]; ++j) {
            A[(size_t)i * n + col[j]] = val[j];
            if (h->storage == HD_STORAGE_UPPER_REF && col[j] != i) A[(size_t)col[j] * n + i] = val[j];
        }
    if (!sym_eig((int)n, A, w, Z)) return fail(HD_ERR_NOT_CONVERGED, "dense eigenproblem did not converge");
    for (int i = 0; i < std::min<int64_t>(nev, n); ++i) h_evals[i] = w[i];
    return HD_OK;
}

}  // extern "C"
