// libmfv batched sparse solves: (sigma_i I + tau_i A_i) x_i = b_i for many independent
// instances i stored as one block-diagonal ELL matrix in 64-row slices (one wavefront per
// slice). The solve is mixed precision: BiCGStab with Jacobi preconditioning in FP32 (FP64
// dot products) inside FP64 iterative refinement, r = b - op(x) in FP64 until
// ||r|| <= tol ||b||.
//
// Instances advance independently through a per-instance state machine kept in device memory
// (status + scalars); every kernel runs a fixed persistent grid over the live-slice or
// live-instance list and acts only on rows whose instance is in the state the kernel serves.
// A tick is therefore valid for any mix of instances at any stage and can be replayed from a captured
// graph while instances join and leave. mfv_krylov_fused_tick, two launches an iteration, is what the
// package's arenas run on; mfv_krylov_tick, eight launches, is the ABI's general form and the solver
// that the tests hold the other one against.
//
// Per-instance reductions of the latter are two-level and deterministic: each wave reduces its slice in a
// fixed shuffle pattern into partial[slice], then one block per instance adds the partials of
// its slices in a fixed order relative to its first slice. An instance's arithmetic therefore
// does not depend on where it sits in the batch or on what else is in it.
#include "mfv_common.hpp"

namespace mfv {

struct Ell {
    int S, W, I;
    const int32_t *__restrict__ slice_inst;
    const int32_t *__restrict__ slice_w;
    const int32_t *__restrict__ cols;
    const double *__restrict__ vals;
    const float *__restrict__ vals32;
    const double *__restrict__ diag;
    const int32_t *__restrict__ inst_slice0;
    const int32_t *__restrict__ inst_nslices;
    const int32_t *__restrict__ live_slices;
    const int32_t *__restrict__ n_live_slices;
    const int32_t *__restrict__ live_inst;
    const int32_t *__restrict__ n_live_inst;
    const int16_t *__restrict__ cols16;
    const uint8_t *__restrict__ narrow;
};

struct Work {
    double *__restrict__ x;
    double *__restrict__ b;
    float *__restrict__ d;
    float *__restrict__ r;
    float *__restrict__ rh;
    float *__restrict__ p;
    float *__restrict__ v;
    float *__restrict__ yz;
    float *__restrict__ t;
    float *__restrict__ dinv;
    double *__restrict__ partial;
    double *__restrict__ scal;
    int32_t *__restrict__ status;
};

static Ell to_kernel(const mfv_ell_batch *e)
{
    return Ell{e->nb_slices,    e->width,       e->nb_inst,       e->slice_inst, e->slice_w, e->cols,
               e->vals,         e->vals32,      e->diag,          e->inst_slice0, e->inst_nslices,
               e->live_slices,  e->n_live_slices, e->live_inst,   e->n_live_inst, e->cols16, e->slice_narrow};
}

static Work to_kernel(const mfv_krylov_work *w)
{
    return Work{w->x, w->b, w->d, w->r, w->rh, w->p, w->v, w->yz, w->t, w->dinv, w->partial, w->scal, w->status};
}

__device__ __forceinline__ double *S(const Work &w, int inst) { return w.scal + (size_t)inst * MFV_KS_NSCAL; }

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Iterates the live slices whose instance is in state `want`; body(slice, inst, row).
template <class Body>
__device__ __forceinline__ void for_slices(const Ell &e, const Work &w, int want0, int want1, Body body)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wpb = blockDim.x >> 6;
    const int n = *e.n_live_slices;
    for (int i = blockIdx.x * wpb + wave; i < n; i += gridDim.x * wpb) {
        const int s = e.live_slices[i];
        const int inst = e.slice_inst[s];
        if (inst < 0) continue;
        const int st = w.status[inst];
        if (st != want0 && st != want1) continue;
        body(s, inst, s * 64 + lane, lane);
    }
}

// sum_j A32[row][j] * x[col_j] in FP32 with explicit fused multiply-adds. A narrow slice reads
// its columns as 16-bit offsets from the row (the branch is uniform over the wave: one slice).
__device__ __forceinline__ bool slice_is_narrow(const Ell &e, int s) { return e.narrow && e.narrow[s]; }

// Sum over the row's slots j < wdt of val[j] * x[col[j]], accumulated in j order. The slots are
// taken in groups (8, then 4, then 1) whose column, value and x loads are all issued before the
// group's multiply-adds, so a slot no longer waits two memory latencies of its own; the
// accumulation order, hence the bits, are those of the slot-by-slot loop.
template <int G, class Val, class Col, class X, class Acc>
__device__ __forceinline__ int ell_group(int j, int wdt, size_t base, const Val *__restrict__ vals, Col col,
                                         const X *__restrict__ x, Acc &acc)
{
    for (; j + G <= wdt; j += G) {
        Val v[G];
        int c[G];
#pragma unroll
        for (int u = 0; u < G; u++) {
            const size_t q = base + (size_t)(j + u) * 64;
            v[u] = vals[q];
            c[u] = col(q);
        }
        X xv[G];
#pragma unroll
        for (int u = 0; u < G; u++) xv[u] = x[c[u]];
#pragma unroll
        for (int u = 0; u < G; u++) acc = fma(v[u], xv[u], acc);
    }
    return j;
}

template <class Val, class X, class Acc>
__device__ __forceinline__ Acc ell_row(const Ell &e, int s, int lane, const Val *__restrict__ vals,
                                       const X *__restrict__ x)
{
    const int wdt = e.slice_w[s];
    const size_t base = (size_t)s * e.W * 64 + lane;
    Acc acc = 0;
    if (slice_is_narrow(e, s)) {
        const int row = s * 64 + lane;
        auto col = [&](size_t q) { return row + e.cols16[q]; };
        int j = ell_group<8>(0, wdt, base, vals, col, x, acc);
        j = ell_group<4>(j, wdt, base, vals, col, x, acc);
        ell_group<1>(j, wdt, base, vals, col, x, acc);
    } else {
        auto col = [&](size_t q) { return e.cols[q]; };
        int j = ell_group<8>(0, wdt, base, vals, col, x, acc);
        j = ell_group<4>(j, wdt, base, vals, col, x, acc);
        ell_group<1>(j, wdt, base, vals, col, x, acc);
    }
    return acc;
}

__device__ __forceinline__ float ell_row32(const Ell &e, int s, int lane, const float *__restrict__ x)
{
    return ell_row<float, float, float>(e, s, lane, e.vals32, x);
}

__device__ __forceinline__ double ell_row64(const Ell &e, int s, int lane, const double *__restrict__ x)
{
    return ell_row<double, double, double>(e, s, lane, e.vals, x);
}

// One wave per slice: the slice is narrow when every used slot's column is within +-32767 of its
// row; then its 16-bit offsets are written. Slots past the slice width are never read.
__global__ void __launch_bounds__(256) k_ell_narrow(Ell e, int slice0, int nslices, int16_t *__restrict__ cols16,
                                                     uint8_t *__restrict__ narrow)
{
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= nslices) return;
    const int s = slice0 + i;
    const int wdt = e.slice_w[s];
    const int row = s * 64 + lane;
    const size_t base = (size_t)s * e.W * 64 + lane;
    int wide = 0;
    for (int j = 0; j < wdt; j++) {
        const int d = e.cols[base + (size_t)j * 64] - row;
        wide |= (d < -32767 || d > 32767) ? 1 : 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) wide |= __shfl_xor(wide, off, 64);
    if (!wide)
        for (int j = 0; j < wdt; j++) {
            const size_t q = base + (size_t)j * 64;
            cols16[q] = (int16_t)(e.cols[q] - row);
        }
    if (lane == 0) narrow[s] = wide ? 0 : 1;
}

// ---------------------------------------------------------------------------------------------
// refinement: x += d (state CORRECT), then r = b - op(x) (states START and CORRECT)

__global__ void __launch_bounds__(256) k_ir_correct(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_CORRECT, MFV_KS_CORRECT,
               [&](int, int, int row, int) { w.x[row] += (double)w.d[row]; });
}

__global__ void __launch_bounds__(256) k_ir_residual(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_START, MFV_KS_CORRECT, [&](int s, int inst, int row, int lane) {
        const double *sc = S(w, inst);
        const double sigma = sc[MFV_KS_SIGMA], tau = sc[MFV_KS_TAU];
        if (w.status[inst] == MFV_KS_START) {
            const double dg = sigma + tau * e.diag[row];
            w.dinv[row] = (dg != 0.) ? (float)(1. / dg) : 0.f;
        }
        const double ax = ell_row64(e, s, lane, w.x);
        const double bb = w.b[row];
        const double res = bb - (sigma * w.x[row] + tau * ax);
        const float r32 = (float)res;
        w.r[row] = r32;
        w.rh[row] = r32;
        w.d[row] = 0.f;
        w.p[row] = 0.f;
        w.v[row] = 0.f;
        const double s0 = wave_sum(res * res);
        const double s1 = wave_sum(bb * bb);
        const double s2 = wave_sum((double)r32 * (double)r32);
        if (lane == 0) {
            w.partial[4 * s + 0] = s0;
            w.partial[4 * s + 1] = s1;
            w.partial[4 * s + 2] = s2;
        }
    });
}

// Threads of a per-instance block: an instance's reduction runs in one block, so a wide block
// shortens the serial part of the largest instance's sum (1M rows = 15 625 slice partials).
constexpr int kInstBlock = 1024;

// Sums partial[slice][0..n) over the instance's slices into out[0..n) (thread 0 holds them).
// Each thread keeps four running sums over its slices (i, i + B, i + 2B, i + 3B, then the next
// 4B), added in that fixed order, then a tree over the block: the order depends only on the
// instance's own slice count.
template <int NSUM>
__device__ __forceinline__ void inst_reduce(const Ell &e, const Work &w, int inst, double *out)
{
    __shared__ double red[NSUM][kInstBlock];
    const int s0 = e.inst_slice0[inst], ns = e.inst_nslices[inst];
    double acc[4][NSUM];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int k = 0; k < NSUM; k++) acc[q][k] = 0.;
    for (int i = threadIdx.x; i < ns; i += 4 * kInstBlock) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int j = i + q * kInstBlock;
            if (j < ns) {
#pragma unroll
                for (int k = 0; k < NSUM; k++) acc[q][k] += w.partial[4 * (size_t)(s0 + j) + k];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NSUM; k++) red[k][threadIdx.x] = (acc[0][k] + acc[1][k]) + (acc[2][k] + acc[3][k]);
    __syncthreads();
    for (int h = kInstBlock / 2; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
#pragma unroll
            for (int k = 0; k < NSUM; k++) red[k][threadIdx.x] += red[k][threadIdx.x + h];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < NSUM; k++) out[k] = red[k][0];
}

// Per-instance kernels: one block per live instance (grid-stride over the live list).
template <class Body>
__device__ __forceinline__ void for_insts(const Ell &e, const Work &w, int want0, int want1, Body body)
{
    const int n = *e.n_live_inst;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const int inst = e.live_inst[i];
        const int st = w.status[inst];
        __syncthreads();
        if (st != want0 && st != want1) continue;
        body(inst);
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kInstBlock) k_ir_check(Ell e, Work w)
{
    for_insts(e, w, MFV_KS_START, MFV_KS_CORRECT, [&](int inst) {
        double sum[3];
        inst_reduce<3>(e, w, inst, sum);
        if (threadIdx.x == 0) {
            double *sc = S(w, inst);
            const double resn2 = sum[0], bn2 = sum[1];
            sc[MFV_KS_RESN2] = resn2;
            sc[MFV_KS_BN2] = bn2;
            if (w.status[inst] == MFV_KS_START) sc[MFV_KS_OUTER] = 0.;
            sc[MFV_KS_OUTER] += 1.;
            const double tol = sc[MFV_KS_TOL_OUT];
            int st;
            if (!isfinite(resn2) || !isfinite(bn2)) st = MFV_KS_FAILED;  // NaN/inf data: refinement cannot help
            else if (resn2 <= tol * tol * bn2) st = MFV_KS_DONE;
            else if (sc[MFV_KS_OUTER] > sc[MFV_KS_MAXIT_OUT]) st = MFV_KS_FAILED;
            else {
                sc[MFV_KS_RHO] = sum[2];
                sc[MFV_KS_R0N2] = sum[2];
                sc[MFV_KS_RN2] = sum[2];
                sc[MFV_KS_ALPHA] = 1.;
                sc[MFV_KS_OMEGA] = 1.;
                sc[MFV_KS_BETA] = 0.;
                sc[MFV_KS_IT] = 0.;
                st = MFV_KS_INNER;
            }
            w.status[inst] = st;
        }
    });
}

// ---------------------------------------------------------------------------------------------
// BiCGStab iteration (right Jacobi preconditioning, y = M^-1 p, z = M^-1 s), FP32 vectors

__global__ void __launch_bounds__(256) k_bicg_p(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int, int inst, int row, int) {
        const double *sc = S(w, inst);
        float p;
        if (sc[MFV_KS_IT] == 0.) {
            p = w.r[row];
        } else {
            const float beta = (float)sc[MFV_KS_BETA], omega = (float)sc[MFV_KS_OMEGA];
            p = fmaf(beta, fmaf(-omega, w.v[row], w.p[row]), w.r[row]);
        }
        w.p[row] = p;
        w.yz[row] = w.dinv[row] * p;
    });
}

// v = op(y); partial = rh . v
__global__ void __launch_bounds__(256) k_bicg_spmv_v(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int s, int inst, int row, int lane) {
        const double *sc = S(w, inst);
        const float sigma = (float)sc[MFV_KS_SIGMA], tau = (float)sc[MFV_KS_TAU];
        const float v = fmaf(sigma, w.yz[row], tau * ell_row32(e, s, lane, w.yz));
        w.v[row] = v;
        const double s0 = wave_sum((double)w.rh[row] * (double)v);
        if (lane == 0) w.partial[4 * s] = s0;
    });
}

__global__ void __launch_bounds__(kInstBlock) k_bicg_alpha(Ell e, Work w)
{
    for_insts(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int inst) {
        double sum[1];
        inst_reduce<1>(e, w, inst, sum);
        if (threadIdx.x == 0) {
            double *sc = S(w, inst);
            const double rv = sum[0];
            const double a = sc[MFV_KS_RHO] / rv;
            if (rv == 0. || !isfinite(a)) {
                w.status[inst] = MFV_KS_CORRECT;  // breakdown: refine with what d holds
            } else {
                sc[MFV_KS_ALPHA] = a;
            }
        }
    });
}

// s = r - alpha v (in place of r); d += alpha y; z = M^-1 s (in place of y)
__global__ void __launch_bounds__(256) k_bicg_s(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int, int inst, int row, int) {
        const float alpha = (float)S(w, inst)[MFV_KS_ALPHA];
        const float s = fmaf(-alpha, w.v[row], w.r[row]);
        w.r[row] = s;
        w.d[row] = fmaf(alpha, w.yz[row], w.d[row]);
        w.yz[row] = w.dinv[row] * s;
    });
}

// t = op(z); partial = (t . s, t . t)
__global__ void __launch_bounds__(256) k_bicg_spmv_t(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int s, int inst, int row, int lane) {
        const double *sc = S(w, inst);
        const float sigma = (float)sc[MFV_KS_SIGMA], tau = (float)sc[MFV_KS_TAU];
        const float t = fmaf(sigma, w.yz[row], tau * ell_row32(e, s, lane, w.yz));
        w.t[row] = t;
        const double s0 = wave_sum((double)t * (double)w.r[row]);
        const double s1 = wave_sum((double)t * (double)t);
        if (lane == 0) {
            w.partial[4 * s + 0] = s0;
            w.partial[4 * s + 1] = s1;
        }
    });
}

__global__ void __launch_bounds__(kInstBlock) k_bicg_omega(Ell e, Work w)
{
    for_insts(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int inst) {
        double sum[2];
        inst_reduce<2>(e, w, inst, sum);
        if (threadIdx.x == 0) {
            double *sc = S(w, inst);
            const double om = (sum[1] != 0.) ? sum[0] / sum[1] : 0.;
            sc[MFV_KS_OMEGA] = isfinite(om) ? om : 0.;
        }
    });
}

// d += omega z; r = s - omega t; partial = (r . r, rh . r)
__global__ void __launch_bounds__(256) k_bicg_x(Ell e, Work w)
{
    for_slices(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int s, int inst, int row, int lane) {
        const float omega = (float)S(w, inst)[MFV_KS_OMEGA];
        w.d[row] = fmaf(omega, w.yz[row], w.d[row]);
        const float r = fmaf(-omega, w.t[row], w.r[row]);
        w.r[row] = r;
        const double s0 = wave_sum((double)r * (double)r);
        const double s1 = wave_sum((double)w.rh[row] * (double)r);
        if (lane == 0) {
            w.partial[4 * s + 0] = s0;
            w.partial[4 * s + 1] = s1;
        }
    });
}

__global__ void __launch_bounds__(kInstBlock) k_bicg_rho(Ell e, Work w)
{
    for_insts(e, w, MFV_KS_INNER, MFV_KS_INNER, [&](int inst) {
        double sum[2];
        inst_reduce<2>(e, w, inst, sum);
        if (threadIdx.x == 0) {
            double *sc = S(w, inst);
            const double rn2 = sum[0], rho_new = sum[1];
            const double omega = sc[MFV_KS_OMEGA];
            sc[MFV_KS_RN2] = rn2;
            sc[MFV_KS_IT] += 1.;
            sc[MFV_KS_ITTOT] += 1.;
            const double tol = sc[MFV_KS_TOL_IN];
            const bool done = rn2 <= tol * tol * sc[MFV_KS_R0N2] || sc[MFV_KS_IT] >= sc[MFV_KS_MAXIT_IN] ||
                              rho_new == 0. || omega == 0.;
            if (done) {
                w.status[inst] = MFV_KS_CORRECT;
            } else {
                sc[MFV_KS_BETA] = (rho_new / sc[MFV_KS_RHO]) * (sc[MFV_KS_ALPHA] / omega);
                sc[MFV_KS_RHO] = rho_new;
            }
        }
    });
}

// y = A x (FP64) on the live slices, whatever their state
__global__ void __launch_bounds__(256) k_ell_spmv(Ell e, const double *__restrict__ x, double *__restrict__ y)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int n = *e.n_live_slices;
    for (int i = blockIdx.x * 4 + wave; i < n; i += gridDim.x * 4) {
        const int s = e.live_slices[i];
        y[s * 64 + lane] = ell_row64(e, s, lane, x);
    }
}

// ---------------------------------------------------------------------------------------------
// The same solve with two launches per iteration (mfv_krylov_fused_tick).
//
// The eight-launch iteration above is bound by launches and memory latency, not by bytes: at
// 13k rows each of its kernels takes 3 to 4.6 us for under 1 us of traffic (32.8 us an
// iteration). Here an iteration is two matrix products with everything else folded into them:
//
//   v:  omega, rho, beta from the sums of t;  d += alpha p + omega s;  r = s - omega t;
//       p = r + beta (p - omega v);  v = M op(p);                            sum rh.v
//   t:  alpha from the sum of v;  s = r - alpha v;  t = M op(s);
//                                           sums t.s, t.t, s.s, rh.s, rh.t
//
// * M = 1 / diag scales the rows of the product (the system M op(d) = M r), and the inner stop is on M r;
//   so a slot needs
//   nothing of its column but p (s), which is computed again from the column's record for each
//   slot: three multiply-adds (one) and one gather of 16 bytes (8) instead of a launch and a
//   trip of the vector through memory. The v product reads u = (s, t, p, v) and writes
//   w = (r, v) and p; the t product reads those and writes u, so no row writes what another one
//   reads. With M on the right the v product gathered 20 bytes and held 195 registers, two waves
//   a SIMD: 12.0 us at 193k rows in eight systems, 8.5 us so.
// * Measured, v and t product with all changes of state in them: 7.0 + 6.1 us at 12 800 rows and 8.3 +
//   8.4 us at 193k rows in eight systems (6.4 + 5.2 and 7.4 + 6.2 us without, and four launches more
//   a tick), against 28 us and 29 us for the eight kernels. What is left is the chain chunk -> columns -> records
//   with a trip to memory each, and the fixed cost of adding up.
// * |r|^2 and rh.r of the new residual follow from the t product's sums (r = s - omega t), so
//   omega, rho and beta need no third pass; the refinement's own residual stays FP64 and is
//   formed from x itself.
// * The sums have no launch of their own: every block of the next product adds up its
//   instance's chunk sums, in the same fixed order, so all blocks hold the same bits. A chunk is
//   four slices (one a wave) and an instance has at most 512, so that this costs two loads a
//   thread; larger instances take more slices a chunk.
// * The refinement has no launches of its own either. The product that finds the inner solve ended
//   adds d to x at once, the t product after it forms the FP64 residual instead of a product, and
//   the v product after that comes to the verdict on it and takes the first step of the next inner
//   solve. With a launch each for them (four, and a round of the host's, every n_iter iterations) a
//   change of state waited for the next tick: 20 implicit steps of eight systems took 154 ticks of
//   six iterations, 120 so; a system of 12.8k rows 13.0 -> 11.3 ms.
// * An instance that has time steps left (steps_left) takes the next one where it would be done: the
//   v product writes b = x + dt advection(x), the t product takes x = b and forms its residual.
//   Nothing of it waits for the host (serving, eight requests of 20 steps: 33.5 -> 26.5 ms).
// * A scalar is never read in the launch that writes it: the v product reads ALPHA, RHO_OLD, IT,
//   OUTER, steps_left and status and writes OMEGA, BETA, RHO, RN2, the scalars that an inner solve
//   starts from (in state CHECK, which reads none of them) and status_t; the t product reads RHO and
//   status_t and writes ALPHA, RHO_OLD, IT, ITTOT, OUTER, steps_left and status. Between pairs of
//   launches status is the instance's whole state. Only the instance's first block writes them.
struct Fused {
    double *__restrict__ x;
    double *__restrict__ b;
    float *__restrict__ d;
    float *__restrict__ rh;
    float *__restrict__ dinv;
    float4 *__restrict__ u;
    float2 *__restrict__ w;
    float *__restrict__ p;
    double *__restrict__ pa;
    double *__restrict__ pb;
    double *__restrict__ scal;
    int32_t *__restrict__ status;
    int32_t *__restrict__ status_t;
    const int4 *__restrict__ chunks;
    const int32_t *__restrict__ n_chunks;
    int32_t *__restrict__ steps_left;
    const int32_t *__restrict__ adv_up;
    const double *__restrict__ adv_coef;
    const double *__restrict__ adv_vol;
    int adv_slots;
};

// What a t product does with an instance besides its part of an iteration (status_t; the other
// values are those of status).
enum { kResidualStart = 16, kResidual, kResidualOfB };

static Fused to_kernel(const mfv_krylov_fused *w)
{
    return Fused{w->x,  w->b,  w->d,  w->rh,   w->dinv,   reinterpret_cast<float4 *>(w->u),
                 reinterpret_cast<float2 *>(w->w), w->p, w->pa, w->pb, w->scal, w->status,
                 w->status_t, reinterpret_cast<const int4 *>(w->chunks), w->n_chunks, w->steps_left, w->adv_up,
                 w->adv_coef, w->adv_vol, w->adv_slots};
}

constexpr int kChunkBlock = 256;
constexpr int kChunkWaves = kChunkBlock / 64;
static_assert(MFV_KRYLOV_SPAN(1) == kChunkWaves, "a chunk's first slices are one a wave");

// The wave's number in its block, known to be the same for all lanes (scalar slice tables).
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

struct Chunk {
    int inst, s0, c, nch, ns, begin, end;
};
__device__ __forceinline__ Chunk chunk_at(const Fused &w, int k)
{
    const int4 q = w.chunks[k];
    Chunk h;
    h.inst = q.x;
    h.s0 = q.y;
    h.c = q.z & 0xffff;
    h.nch = q.z >> 16;
    h.ns = q.w;
    const int span = MFV_KRYLOV_SPAN(q.w);
    h.begin = h.s0 + h.c * span;
    h.end = min(h.begin + span, h.s0 + h.ns);
    return h;
}

// Sum over the wave, in every lane: moves inside the register file (row shifts, then the two row
// broadcasts) instead of wave_sum's twelve trips through the LDS crossbar, which cost more than
// the loads of a small instance's sums (v product of a stopped instance: 4.8 us against 3.0 us
// for the t product, which adds one sum instead of five).
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_total(double v)
{
    v += dpp_move<0x111>(v);  // row_shr:1
    v += dpp_move<0x112>(v);  // row_shr:2
    v += dpp_move<0x114>(v);  // row_shr:4
    v += dpp_move<0x118>(v);  // row_shr:8: lane 15 of each row of 16 holds the row's sum
    const long long b = __double_as_longlong(v);
    double t = 0.;
#pragma unroll
    for (int r = 15; r < 64; r += 16) {
        const int lo = __builtin_amdgcn_readlane((int)b, r), hi = __builtin_amdgcn_readlane((int)(b >> 32), r);
        t += __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
    }
    return t;
}

// The chunk sums part[k][s0 .. s0 + nch) of an instance, in an order that depends on nch alone;
// every thread gets the totals. Up to 128 chunks (32 768 rows) each wave adds them up for itself,
// two loads a lane and no barrier; above, the block shares them. Block-uniform calls only.
template <int N>
__device__ __forceinline__ void chunk_totals(const double *__restrict__ part, size_t S, int s0, int nch,
                                             double (&out)[N])
{
    __shared__ double red[N][kChunkWaves];
    double acc[N];
    if (nch <= 128) {
        const int i = threadIdx.x & 63;
#pragma unroll
        for (int k = 0; k < N; k++) {
            const double a = part[k * S + s0 + min(i, nch - 1)], b = part[k * S + s0 + min(i + 64, nch - 1)];
            acc[k] = (i < nch ? a : 0.) + (i + 64 < nch ? b : 0.);
        }
#pragma unroll
        for (int k = 0; k < N; k++) out[k] = wave_total(acc[k]);
        return;
    }
#pragma unroll
    for (int k = 0; k < N; k++) acc[k] = 0.;
    for (int i = threadIdx.x; i < nch; i += kChunkBlock) {
#pragma unroll
        for (int k = 0; k < N; k++) acc[k] += part[k * S + s0 + i];
    }
    __syncthreads();  // the totals of the block's previous chunk have been read
#pragma unroll
    for (int k = 0; k < N; k++) {
        const double a = wave_total(acc[k]);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = a;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) {
        double a = red[k][0];
#pragma unroll
        for (int q = 1; q < kChunkWaves; q++) a += red[k][q];
        out[k] = a;
    }
}

// The block's sums of one chunk, from each lane's: stored at part[k][at] by one thread.
template <int N>
__device__ __forceinline__ void chunk_store(double *__restrict__ part, size_t S, int at, const double (&lane)[N])
{
    __shared__ double red[N][kChunkWaves];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) {
        const double a = wave_total(lane[k]);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = a;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        double a = red[threadIdx.x][0];
#pragma unroll
        for (int q = 1; q < kChunkWaves; q++) a += red[threadIdx.x][q];
        part[threadIdx.x * S + at] = a;
    }
}

// Slots of a row: values, and the records that load(column) returns, all requested before any is
// used; add() then sums the slots below the slice's width in slot order. first() takes the slots
// from 0 on without waiting for the width: the 16-bit columns, the values and the slice's width
// are requested together (the arrays hold e.W slots whatever the width), and a slot past the
// width takes the row itself. A triangle's row has at most 16 slots, so one first() is the row.
template <class Rec, int N>
struct SlotGroup {
    float v[N];
    Rec r[N];
    template <class Load>
    __device__ __forceinline__ int first(const Ell &e, int s, int lane, Load load)
    {
        const int row = s * 64 + lane;
        const size_t base = (size_t)s * e.W * 64 + lane;
        int c[N];
        if (e.cols16) {
#pragma unroll
            for (int k = 0; k < N; k++) c[k] = e.cols16[base + (size_t)min(k, e.W - 1) * 64];
        }
#pragma unroll
        for (int k = 0; k < N; k++) v[k] = e.vals32[base + (size_t)min(k, e.W - 1) * 64];
        const int wdt = e.slice_w[s];
        if (!slice_is_narrow(e, s)) {  // the same branch for the whole wave
#pragma unroll
            for (int k = 0; k < N; k++) c[k] = e.cols[base + (size_t)min(k, e.W - 1) * 64] - row;
        }
#pragma unroll
        for (int k = 0; k < N; k++) r[k] = load(row + (k < wdt ? c[k] : 0));
        return wdt;
    }
    template <class Load>
    __device__ __forceinline__ void next(const Ell &e, int s, int lane, int j, int wdt, Load load)
    {
        const int row = s * 64 + lane;
        const size_t base = (size_t)s * e.W * 64 + lane;
        int c[N];
        if (slice_is_narrow(e, s)) {
#pragma unroll
            for (int k = 0; k < N; k++) c[k] = row + e.cols16[base + (size_t)min(j + k, wdt - 1) * 64];
        } else {
#pragma unroll
            for (int k = 0; k < N; k++) c[k] = e.cols[base + (size_t)min(j + k, wdt - 1) * 64];
        }
#pragma unroll
        for (int k = 0; k < N; k++) v[k] = e.vals32[base + (size_t)min(j + k, wdt - 1) * 64];
#pragma unroll
        for (int k = 0; k < N; k++) r[k] = load(c[k]);
    }
    template <class Eval>
    __device__ __forceinline__ float add(float acc, int j, int wdt, Eval eval) const
    {
#pragma unroll
        for (int k = 0; k < N; k++)
            if (j + k < wdt) acc = fmaf(v[k], eval(r[k]), acc);
        return acc;
    }
};
constexpr int kFirst = 16, kNext = 8;

// x += d, with the last iteration's alpha p + omega s where they are still to come.
__device__ __forceinline__ void chunk_correct(const Fused &w, const Chunk &h, bool pending, float alpha, float omega)
{
    for (int row = h.begin * 64 + threadIdx.x; row < h.end * 64; row += kChunkBlock) {
        float d = w.d[row];
        if (pending) {
            const float4 u = w.u[row];
            d = fmaf(omega, u.x, fmaf(alpha, u.z, d));
        }
        w.x[row] += (double)d;
    }
}

// b = x + dt advection(x): the upwind values, their outward face velocities and the order of the
// sum are laid out per row (mfv_advection_rows).
__device__ __forceinline__ void chunk_advance(const Ell &e, const Fused &w, const Chunk &h, double dt)
{
    const size_t R = (size_t)e.S * 64;
    for (int row = h.begin * 64 + threadIdx.x; row < h.end * 64; row += kChunkBlock) {
        double rez = 0.;
        for (int j = 0; j < w.adv_slots; j += 4) {
            int up[4];
            double c[4], v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                up[k] = w.adv_up[(j + k) * R + row];
                c[k] = w.adv_coef[(j + k) * R + row];
            }
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = w.x[up[k] < 0 ? row : up[k]] + 0.;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (up[k] >= 0) rez -= c[k] * v[k];
        }
        w.b[row] = w.x[row] + dt * ((rez + 0.) / w.adv_vol[row] + 0.);
    }
}

// ell_row64 as the products of the iteration take their slots: the first sixteen (a triangle's row)
// at once, the columns asked for without waiting for the width, the rest in groups of four. Whatever
// state the others are in, a launch takes as long as the one system that forms its residual (t product
// of eight systems 10.8 us on average, 9.9 us so, and 8.4 us behind the loop, see k_fused_t).
__device__ __forceinline__ double row_product64(const Ell &e, int s, int lane, const double *__restrict__ x)
{
    const int row = s * 64 + lane;
    const size_t base = (size_t)s * e.W * 64 + lane;
    const int wdt = e.slice_w[s];
    const bool narrow = slice_is_narrow(e, s);
    double v[kFirst], xv[kFirst], acc = 0.;
    int c[kFirst];
    if (e.cols16) {
#pragma unroll
        for (int k = 0; k < kFirst; k++) c[k] = e.cols16[base + (size_t)min(k, e.W - 1) * 64];
    }
#pragma unroll
    for (int k = 0; k < kFirst; k++) v[k] = e.vals[base + (size_t)min(k, e.W - 1) * 64];
    if (!narrow) {
#pragma unroll
        for (int k = 0; k < kFirst; k++) c[k] = e.cols[base + (size_t)min(k, e.W - 1) * 64] - row;
    }
#pragma unroll
    for (int k = 0; k < kFirst; k++) xv[k] = x[row + (k < wdt ? c[k] : 0)];
#pragma unroll
    for (int k = 0; k < kFirst; k++)
        if (k < wdt) acc = fma(v[k], xv[k], acc);
    for (int j = kFirst; j < wdt; j += 4) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const size_t q = base + (size_t)min(j + k, wdt - 1) * 64;
            v[k] = e.vals[q];
            c[k] = narrow ? row + e.cols16[q] : e.cols[q];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) xv[k] = x[c[k]];
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (j + k < wdt) acc = fma(v[k], xv[k], acc);
    }
    return acc;
}

// r = b - op(x) in FP64 and the start of the inner solve.
__device__ __forceinline__ void chunk_residual(const Ell &e, const Fused &w, const Chunk &h, int how, double sigma,
                                               double tau)
{
    const int lane = threadIdx.x & 63;
    const double *x = how == kResidualOfB ? w.b : w.x;  // x = b then, and no row is read and written
    double sum[3] = {0., 0., 0.};
    for (int s = h.begin + wave_index(); s < h.end; s += kChunkWaves) {
        const int row = s * 64 + lane;
        const double bb = w.b[row], xx = x[row], diag = e.diag[row];
        float di = w.dinv[row];
        const double ax = row_product64(e, s, lane, x);
        if (how != kResidual) {
            const double dg = sigma + tau * diag;
            w.dinv[row] = di = (dg != 0.) ? (float)(1. / dg) : 0.f;
        }
        if (how == kResidualOfB) w.x[row] = xx;
        const double res = bb - (sigma * xx + tau * ax);
        const float r32 = (float)((double)di * res);
        w.rh[row] = r32;
        w.d[row] = 0.f;
        w.u[row] = make_float4(r32, 0.f, 0.f, 0.f);
        sum[0] += res * res;
        sum[1] += bb * bb;
        sum[2] += (double)r32 * (double)r32;
    }
    chunk_store<3>(w.pb, e.S, h.s0 + h.c, sum);  // pb's iteration has been closed
}

// omega, the new residual's norm and rho, and whether the inner solve ends, from the t product's
// sums (t.s, t.t, s.s, rh.s, rh.t).
struct Step {
    double omega, rn2, rho;
    bool done;
};
struct Stop {
    double tol, r0n2, it, maxit;
};
__device__ __forceinline__ Stop stop_of(const double *sc)
{
    return Stop{sc[MFV_KS_TOL_IN], sc[MFV_KS_R0N2], sc[MFV_KS_IT], sc[MFV_KS_MAXIT_IN]};
}
__device__ __forceinline__ Step close_step(const double (&q)[5], const Stop &s)
{
    Step r;
    const double om = (q[1] != 0.) ? q[0] / q[1] : 0.;
    r.omega = isfinite(om) ? om : 0.;
    r.rn2 = q[2] - 2. * r.omega * q[0] + r.omega * r.omega * q[1];
    r.rho = q[3] - r.omega * q[4];
    r.done = r.rn2 <= s.tol * s.tol * s.r0n2 || s.it >= s.maxit || r.rho == 0. || r.omega == 0.;
    return r;
}

__global__ void __launch_bounds__(kChunkBlock, 3) k_fused_v(Ell e, Fused w)
{
    const int lane = threadIdx.x & 63;
    Chunk h = chunk_at(w, min((int)blockIdx.x, e.S - 1));  // with the count, not after it
    const int n = *w.n_chunks;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        if (k != (int)blockIdx.x) h = chunk_at(w, k);
        double *sc = w.scal + (size_t)h.inst * MFV_KS_NSCAL;
        const bool first = h.c == 0 && threadIdx.x == 0;
        const int status = w.status[h.inst];  // the scalars too, before anything is waited for
        const double rho_old = sc[MFV_KS_RHO_OLD], alpha_old = sc[MFV_KS_ALPHA];
        const float sigma = (float)sc[MFV_KS_SIGMA], tau = (float)sc[MFV_KS_TAU];
        const Stop lim = stop_of(sc);
        auto load = [&](int c) { return w.u[c]; };
        // the first slots' records are on their way while the sums are added up, also for an
        // instance that turns out to be idle
        int s = h.begin + wave_index();
        SlotGroup<float4, kFirst> g;
        float4 own;
        float rh = 0.f, d = 0.f, di = 0.f;
        int wdt = 0;
        auto take = [&]() {
            const int row = s * 64 + lane;
            own = load(row);
            rh = w.rh[row];
            d = w.d[row];
            di = w.dinv[row];
            wdt = g.first(e, s, lane, load);
        };
        if (s < h.end) take();
        double q[5];
        chunk_totals<5>(w.pb, e.S, h.s0, h.nch, q);
        float alpha = 0.f, om = 0.f, be = 0.f;
        int next = status;  // status_t
        if (status == MFV_KS_INNER) {
            const Step st = close_step(q, lim);
            const double beta = (st.rho / rho_old) * (alpha_old / st.omega);
            if (first) {
                sc[MFV_KS_OMEGA] = st.omega;
                sc[MFV_KS_RN2] = st.rn2;
                if (!st.done) {
                    sc[MFV_KS_BETA] = beta;
                    sc[MFV_KS_RHO] = st.rho;
                }
            }
            alpha = (float)alpha_old;
            om = (float)st.omega;
            be = (float)beta;
            if (st.done) {
                chunk_correct(w, h, true, alpha, om);
                next = kResidual;
            }
        } else if (status == MFV_KS_CORRECT) {  // a breakdown in the t product: d holds all there is
            chunk_correct(w, h, false, 0.f, 0.f);
            next = kResidual;
        } else if (status == MFV_KS_START) {
            next = kResidualStart;
        } else if (status == MFV_KS_ADVANCE) {
            chunk_advance(e, w, h, sc[MFV_KS_DT]);
            next = kResidualOfB;
        } else if (status == MFV_KS_CHECK) {
            const double tol = sc[MFV_KS_TOL_OUT];
            if (!isfinite(q[0]) || !isfinite(q[1])) next = MFV_KS_FAILED;  // NaN/inf data: refinement cannot help
            else if (q[0] <= tol * tol * q[1]) next = MFV_KS_DONE;
            else if (sc[MFV_KS_OUTER] > sc[MFV_KS_MAXIT_OUT]) next = MFV_KS_FAILED;
            else next = MFV_KS_INNER;
            if (next == MFV_KS_DONE && w.steps_left && w.steps_left[h.inst] > 0) {
                chunk_advance(e, w, h, sc[MFV_KS_DT]);
                next = kResidualOfB;
            }
            if (first) {
                sc[MFV_KS_RESN2] = q[0];
                sc[MFV_KS_BN2] = q[1];
                if (next == MFV_KS_INNER) {
                    sc[MFV_KS_RHO] = q[2];
                    sc[MFV_KS_RHO_OLD] = q[2];
                    sc[MFV_KS_R0N2] = q[2];
                    sc[MFV_KS_RN2] = q[2];
                    sc[MFV_KS_ALPHA] = 0.;
                    sc[MFV_KS_OMEGA] = 0.;
                    sc[MFV_KS_BETA] = 0.;
                    sc[MFV_KS_IT] = 0.;
                }
            }
        }
        if (first) w.status_t[h.inst] = next;
        if (next != MFV_KS_INNER) continue;
        auto p_of = [&](const float4 &u) { return fmaf(be, fmaf(-om, u.w, u.z), fmaf(-om, u.y, u.x)); };
        double sum[1] = {0.};
        while (s < h.end) {
            const int row = s * 64 + lane;
            float acc = g.add(0.f, 0, wdt, p_of);
            for (int j = kFirst; j < wdt; j += kNext) {
                SlotGroup<float4, kNext> m;
                m.next(e, s, lane, j, wdt, load);
                acc = m.add(acc, j, wdt, p_of);
            }
            const float p = p_of(own);
            const float v = di * fmaf(sigma, p, tau * acc);
            w.d[row] = fmaf(om, own.x, fmaf(alpha, own.z, d));
            w.w[row] = make_float2(fmaf(-om, own.y, own.x), v);
            w.p[row] = p;
            sum[0] += (double)rh * (double)v;
            s += kChunkWaves;
            if (s < h.end) take();
        }
        chunk_store<1>(w.pa, e.S, h.s0 + h.c, sum);
    }
}

__global__ void __launch_bounds__(kChunkBlock, 3) k_fused_t(Ell e, Fused w)
{
    const int lane = threadIdx.x & 63;
    Chunk h = chunk_at(w, min((int)blockIdx.x, e.S - 1));
    const int n = *w.n_chunks;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        if (k != (int)blockIdx.x) h = chunk_at(w, k);
        double *sc = w.scal + (size_t)h.inst * MFV_KS_NSCAL;
        const bool first = h.c == 0 && threadIdx.x == 0;
        const int status = w.status_t[h.inst];
        const double rho = sc[MFV_KS_RHO];
        const float sigma = (float)sc[MFV_KS_SIGMA], tau = (float)sc[MFV_KS_TAU];
        auto load = [&](int c) { return w.w[c]; };
        int s = h.begin + wave_index();
        SlotGroup<float2, kFirst> g;
        float2 own;
        float rh = 0.f, di = 0.f, p = 0.f;
        int wdt = 0;
        auto take = [&]() {
            const int row = s * 64 + lane;
            own = load(row);
            rh = w.rh[row];
            di = w.dinv[row];
            p = w.p[row];
            wdt = g.first(e, s, lane, load);
        };
        if (s < h.end) take();
        double rv[1];
        chunk_totals<1>(w.pa, e.S, h.s0, h.nch, rv);
        if (status != MFV_KS_INNER) continue;
        const double a = rho / rv[0];
        const bool broken = rv[0] == 0. || !isfinite(a);  // breakdown: refine with what d holds
        if (first) {
            if (!broken) {
                sc[MFV_KS_ALPHA] = a;
                sc[MFV_KS_RHO_OLD] = rho;
                sc[MFV_KS_IT] += 1.;
                sc[MFV_KS_ITTOT] += 1.;
            }
            w.status[h.inst] = broken ? MFV_KS_CORRECT : MFV_KS_INNER;
        }
        if (broken) continue;
        const float al = (float)a;
        auto s_of = [&](const float2 &r) { return fmaf(-al, r.y, r.x); };
        double sum[5] = {0., 0., 0., 0., 0.};
        while (s < h.end) {
            const int row = s * 64 + lane;
            float acc = g.add(0.f, 0, wdt, s_of);
            for (int j = kFirst; j < wdt; j += kNext) {
                SlotGroup<float2, kNext> m;
                m.next(e, s, lane, j, wdt, load);
                acc = m.add(acc, j, wdt, s_of);
            }
            const float ss = s_of(own);
            const float t = di * fmaf(sigma, ss, tau * acc);
            w.u[row] = make_float4(ss, t, p, own.y);
            sum[0] += (double)t * (double)ss;
            sum[1] += (double)t * (double)t;
            sum[2] += (double)ss * (double)ss;
            sum[3] += (double)rh * (double)ss;
            sum[4] += (double)rh * (double)t;
            s += kChunkWaves;
            if (s < h.end) take();
        }
        chunk_store<5>(w.pb, e.S, h.s0 + h.c, sum);
    }
    // The block's chunks in another state, behind the loop: with the residual in it the kernel needs 197
    // registers or spills, 126 so; solves of 12.8k rows took 7.1 us a launch, 6.1 us now.
#pragma unroll 1
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const Chunk c = chunk_at(w, k);
        const int status = w.status_t[c.inst];
        if (status == MFV_KS_INNER) continue;
        double *sc = w.scal + (size_t)c.inst * MFV_KS_NSCAL;
        const bool first = c.c == 0 && threadIdx.x == 0;
        if (status < kResidualStart) {
            if (first) w.status[c.inst] = status;
            continue;
        }
        if (first) {
            sc[MFV_KS_OUTER] = (status == kResidual ? sc[MFV_KS_OUTER] : 0.) + 1.;
            if (status == kResidualOfB) w.steps_left[c.inst] -= 1;
            w.status[c.inst] = MFV_KS_CHECK;
        }
        chunk_residual(e, w, c, status, sc[MFV_KS_SIGMA], sc[MFV_KS_TAU]);
    }
}

static int validate_ell(const mfv_ell_batch *e)
{
    MFV_REQUIRE(e != nullptr, "ELL batch descriptor is NULL");
    MFV_REQUIRE(e->nb_slices >= 1 && e->width >= 1 && e->nb_inst >= 1, "ELL batch sizes must be positive");
    MFV_REQUIRE((e->cols16 == nullptr) == (e->slice_narrow == nullptr), "cols16 and slice_narrow go together");
    MFV_REQUIRE((long long)e->nb_slices * 64 < (1LL << 31), "ELL batch rows exceed int32");
    MFV_REQUIRE(e->slice_inst && e->slice_w && e->cols && e->vals && e->vals32 && e->diag && e->inst_slice0 &&
                    e->inst_nslices && e->live_slices && e->n_live_slices && e->live_inst && e->n_live_inst,
                "ELL batch descriptor has NULL pointers");
    return MFV_OK;
}

static int validate_work(const mfv_krylov_work *w)
{
    MFV_REQUIRE(w != nullptr, "Krylov work descriptor is NULL");
    MFV_REQUIRE(w->x && w->b && w->d && w->r && w->rh && w->p && w->v && w->yz && w->t && w->dinv && w->partial &&
                    w->scal && w->status,
                "Krylov work descriptor has NULL pointers");
    return MFV_OK;
}

}  // namespace mfv

using namespace mfv;

static int check_tick(const mfv_ell_batch *e, const mfv_krylov_work *w, int n_iter, int grid_slices, int grid_inst)
{
    if (int rc = validate_ell(e)) return rc;
    if (int rc = validate_work(w)) return rc;
    MFV_REQUIRE(n_iter >= 0 && n_iter <= 4096, "n_iter %d out of [0, 4096]", n_iter);
    MFV_REQUIRE(grid_slices >= 1 && grid_slices <= 65536, "grid_slices %d out of [1, 65536]", grid_slices);
    MFV_REQUIRE(grid_inst >= 1 && grid_inst <= 65536, "grid_inst %d out of [1, 65536]", grid_inst);
    return MFV_OK;
}

static int tick_launches(const mfv_ell_batch *e, const mfv_krylov_work *w, int n_iter, int grid_slices,
                         int grid_inst, hipStream_t st)
{
    const Ell ek = to_kernel(e);
    const Work wk = to_kernel(w);
    const dim3 gs(grid_slices), gi(grid_inst), b(256), bi(kInstBlock);
    hipLaunchKernelGGL(k_ir_correct, gs, b, 0, st, ek, wk);
    hipLaunchKernelGGL(k_ir_residual, gs, b, 0, st, ek, wk);
    hipLaunchKernelGGL(k_ir_check, gi, bi, 0, st, ek, wk);
    for (int it = 0; it < n_iter; it++) {
        hipLaunchKernelGGL(k_bicg_p, gs, b, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_spmv_v, gs, b, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_alpha, gi, bi, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_s, gs, b, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_spmv_t, gs, b, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_omega, gi, bi, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_x, gs, b, 0, st, ek, wk);
        hipLaunchKernelGGL(k_bicg_rho, gi, bi, 0, st, ek, wk);
    }
    return check_launch("krylov tick");
}

extern "C" int mfv_krylov_tick(const mfv_ell_batch *e, const mfv_krylov_work *w, int n_iter, int grid_slices,
                               int grid_inst, void *stream)
{
    if (int rc = check_tick(e, w, n_iter, grid_slices, grid_inst)) return rc;
    return tick_launches(e, w, n_iter, grid_slices, grid_inst, as_stream(stream));
}

extern "C" int mfv_krylov_graph(const mfv_ell_batch *e, const mfv_krylov_work *w, int n_iter, int grid_slices,
                                int grid_inst, void **graph_out)
{
    if (int rc = check_tick(e, w, n_iter, grid_slices, grid_inst)) return rc;
    MFV_REQUIRE(graph_out, "graph_out is NULL");
    *graph_out = nullptr;
    MfvGraph *g = new MfvGraph();
    int rc = graph_begin(g);
    if (rc == MFV_OK) rc = graph_finish(g, tick_launches(e, w, n_iter, grid_slices, grid_inst, g->stream));
    if (rc != MFV_OK) {
        graph_free(g);
        return rc;
    }
    *graph_out = g;
    return MFV_OK;
}

static int check_fused(const mfv_ell_batch *e, const mfv_krylov_fused *w, int n_iter, int grid_chunks)
{
    if (int rc = validate_ell(e)) return rc;
    MFV_REQUIRE(w != nullptr, "Krylov work descriptor is NULL");
    MFV_REQUIRE(w->x && w->b && w->d && w->rh && w->dinv && w->u && w->w && w->p && w->pa && w->pb && w->scal &&
                    w->status && w->status_t && w->chunks && w->n_chunks,
                "Krylov work descriptor has NULL pointers");
    MFV_REQUIRE(!w->steps_left || (w->adv_up && w->adv_coef && w->adv_vol && w->adv_slots >= 4 && w->adv_slots % 4 == 0),
                "steps_left needs the advection tables, in groups of four slots");
    MFV_REQUIRE(((reinterpret_cast<uintptr_t>(w->u) | reinterpret_cast<uintptr_t>(w->w) |
                  reinterpret_cast<uintptr_t>(w->chunks)) &
                 15) == 0,
                "u, w and chunks must be 16-byte aligned");
    MFV_REQUIRE(n_iter >= 1 && n_iter <= 4096, "n_iter %d out of [1, 4096]", n_iter);
    MFV_REQUIRE(grid_chunks >= 1 && grid_chunks <= 65536, "grid_chunks %d out of [1, 65536]", grid_chunks);
    return MFV_OK;
}

static int fused_launches(const mfv_ell_batch *e, const mfv_krylov_fused *w, int n_iter, int grid_chunks,
                          hipStream_t st)
{
    const Ell ek = to_kernel(e);
    const Fused wk = to_kernel(w);
    const dim3 gc(grid_chunks), b(kChunkBlock);
    for (int it = 0; it < n_iter; it++) {
        hipLaunchKernelGGL(k_fused_v, gc, b, 0, st, ek, wk);
        hipLaunchKernelGGL(k_fused_t, gc, b, 0, st, ek, wk);
    }
    return check_launch("krylov tick");
}

extern "C" int mfv_krylov_fused_tick(const mfv_ell_batch *e, const mfv_krylov_fused *w, int n_iter, int grid_chunks,
                                     void *stream)
{
    if (int rc = check_fused(e, w, n_iter, grid_chunks)) return rc;
    return fused_launches(e, w, n_iter, grid_chunks, as_stream(stream));
}

extern "C" int mfv_krylov_fused_graph(const mfv_ell_batch *e, const mfv_krylov_fused *w, int n_iter, int grid_chunks,
                                      void **graph_out)
{
    if (int rc = check_fused(e, w, n_iter, grid_chunks)) return rc;
    MFV_REQUIRE(graph_out, "graph_out is NULL");
    *graph_out = nullptr;
    MfvGraph *g = new MfvGraph();
    int rc = graph_begin(g);
    if (rc == MFV_OK) rc = graph_finish(g, fused_launches(e, w, n_iter, grid_chunks, g->stream));
    if (rc != MFV_OK) {
        graph_free(g);
        return rc;
    }
    *graph_out = g;
    return MFV_OK;
}

// ---------------------------------------------------------------------------------------------
// The rows of an instance in the advection tables of the fused solve.

__global__ void __launch_bounds__(256) k_advection_rows(Mesh m, const double *__restrict__ uf,
                                                        const double *__restrict__ vf, const double *__restrict__ wf,
                                                        int row0, int rows, size_t R, int slots,
                                                        int32_t *__restrict__ up, double *__restrict__ coef,
                                                        double *__restrict__ vol)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows) return;
    const size_t row = (size_t)row0 + i;
    const int nf = i < m.C ? m.cell_nfaces[i] : 0;
    vol[row] = i < m.C ? m.cell_volume[i] : 1.;
    for (int r = 0; r < slots; r++) {
        int u = -1;
        double c = 0.;
        if (r < nf) {
            const int f = m.cell_faces[(size_t)m.order_split[(size_t)r * m.C + i] * m.C + i];
            const int a = m.face_cells[2 * (size_t)f], b = m.face_cells[2 * (size_t)f + 1];
            const double *n = m.face_normal + 3 * (size_t)f;
            const double sign = uf[f] * n[0] + vf[f] * n[1] + wf[f] * n[2];
            u = row0 + ((sign >= 0 || b < 0) ? a : b);
            c = (a == i) ? sign : -sign;
        }
        up[r * R + row] = u;
        coef[r * R + row] = c;
    }
}

extern "C" int mfv_advection_rows(const mfv_mesh *m, const double *u_face, const double *v_face, const double *w_face,
                                  int row0, int rows, int nb_rows, int slots, int32_t *adv_up, double *adv_coef,
                                  double *adv_vol, void *stream)
{
    if (int rc = validate_mesh(m, 0, 1, 0)) return rc;
    MFV_REQUIRE(u_face && v_face && w_face && adv_up && adv_coef && adv_vol, "NULL array");
    MFV_REQUIRE(m->max_cell_faces <= slots, "%d faces a cell, %d slots", m->max_cell_faces, slots);
    MFV_REQUIRE(row0 >= 0 && rows >= m->nb_cells && (long long)row0 + rows <= nb_rows, "rows [%d, %lld) of %d", row0,
                (long long)row0 + rows, nb_rows);
    if (rows == 0) return MFV_OK;
    hipLaunchKernelGGL(k_advection_rows, dim3(grid_for(rows)), dim3(256), 0, as_stream(stream), to_kernel(m), u_face,
                       v_face, w_face, row0, rows, (size_t)nb_rows, slots, adv_up, adv_coef, adv_vol);
    return check_launch("k_advection_rows");
}

extern "C" int mfv_ell_narrow_columns(const mfv_ell_batch *e, int slice0, int nslices, int16_t *cols16,
                                      uint8_t *slice_narrow, void *stream)
{
    if (int rc = validate_ell(e)) return rc;
    MFV_REQUIRE(cols16 && slice_narrow, "NULL array");
    MFV_REQUIRE(slice0 >= 0 && nslices >= 0 && (long long)slice0 + nslices <= e->nb_slices,
                "slices [%d, %d) outside the batch's %d", slice0, slice0 + nslices, e->nb_slices);
    if (nslices == 0) return MFV_OK;
    hipLaunchKernelGGL(k_ell_narrow, dim3((nslices + 3) / 4), dim3(256), 0, as_stream(stream), to_kernel(e), slice0,
                       nslices, cols16, slice_narrow);
    return check_launch("k_ell_narrow");
}

extern "C" int mfv_ell_spmv(const mfv_ell_batch *e, const double *x, double *y, int grid_slices, void *stream)
{
    if (int rc = validate_ell(e)) return rc;
    MFV_REQUIRE(x && y, "NULL array");
    MFV_REQUIRE(grid_slices >= 1 && grid_slices <= 65536, "grid_slices %d out of [1, 65536]", grid_slices);
    hipLaunchKernelGGL(k_ell_spmv, dim3(grid_slices), dim3(256), 0, as_stream(stream), to_kernel(e), x, y);
    return check_launch("k_ell_spmv");
}
