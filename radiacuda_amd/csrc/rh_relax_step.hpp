// rh_relax_step.hpp -- device code of one relaxation step: the element update
// with its Anderson bookkeeping, the Anderson step itself and the update
// coefficients, shared by the forward and the adjoint iteration.
//
// Latency bound: a step is one wave per 64 elements and a last block of one
// wave, so what counts is the length of the dependent chain.
#pragma once

#include <hip/hip_runtime.h>

#include "rh_kernels.hpp"

namespace rh {

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// The sums over the wave of 2 kHistMax = 32 values per lane: at each step a
// lane hands half of its values to its partner and adds the partner's to the
// rest, so that 32 exchanges do instead of 192.  Lane l ends up with the total
// of value l / 2.
static_assert(kHistMax == 16, "wave_sum32 and the Anderson step are written for 16 differences");
template <int M>
__device__ __forceinline__ void wave_halve(double (&v)[2 * kHistMax], int lane)
{
    const bool up = lane & (2 * M);
#pragma unroll
    for (int k = 0; k < M; k++) {
        const double keep = up ? v[k + M] : v[k], give = up ? v[k] : v[k + M];
        v[k] = keep + __shfl_xor(give, 2 * M, 64);
    }
    if constexpr (M > 1) wave_halve<M / 2>(v, lane);
}
__device__ __forceinline__ double wave_sum32(double (&v)[2 * kHistMax], int lane)
{
    wave_halve<kHistMax>(v, lane);
    return v[0] + __shfl_xor(v[0], 1, 64);
}

// One relaxation step with its Anderson bookkeeping (one wave per block):
// lane i updates element i by `law` (proposal and |H|); dF[k] (k < nh, oldest
// first) are the stored differences, the newest of which (dF[nh - 1]) is the
// one written here when dFw is set.
static_assert(kRelaxLanes == 64, "a step reduces over one wave per block");
template <class Law>
__device__ __forceinline__ void relax_step_block(int64_t n, const Law& law, const double* __restrict__ M,
                                                 double* __restrict__ F, double* __restrict__ partials,
                                                 double* Fp, double* xp, double* dFw, double* dXw,
                                                 const double* const* dF, int nh)
{
    const int64_t i = int64_t(blockIdx.x) * kRelaxLanes + threadIdx.x;
    double f2 = 0.0, mm = 0.0, hh = 0.0;
    double dd[2 * kHistMax];
#pragma unroll
    for (int k = 0; k < 2 * kHistMax; k++) dd[k] = 0.0;
    if (i < n) {
        double mp[3];
        law(i, mp, hh);
        double fi[3], dfn[3] = {0.0, 0.0, 0.0};
        for (int k = 0; k < 3; k++) {
            const int64_t j = 3 * i + k;
            const double xk = M[j];
            const double d = mp[k] - xk;
            fi[k] = d;
            F[j] = d;
            f2 += d * d;
            if (dFw) {
                dfn[k] = d - Fp[j];
                dFw[j] = dfn[k];
                dXw[j] = xk - xp[j];
            }
            Fp[j] = d;
            xp[j] = xk;
        }
        mm = sqrt(mp[0] * mp[0] + mp[1] * mp[1] + mp[2] * mp[2]);
#pragma unroll
        for (int h = 0; h < kHistMax; h++) {
            if (h < nh) {
                double a = 0.0, b = 0.0;
                for (int k = 0; k < 3; k++) {
                    const double v = (h == nh - 1) ? dfn[k] : dF[h][3 * i + k];
                    a += dfn[k] * v;
                    b += v * fi[k];
                }
                dd[h] = a;
                dd[kHistMax + h] = b;
            }
        }
    }
    f2 = wave_sum(f2);
    mm = wave_max(mm);
    hh = wave_max(hh);
    const int lane = threadIdx.x;
    double* o = partials + int64_t(kRelaxPart) * blockIdx.x;
    if (lane == 0) {
        o[0] = f2;
        o[1] = mm;
        o[2] = hh;
    }
    const double t = wave_sum32(dd, lane);
    if ((lane & 1) == 0) o[3 + (lane >> 1)] = t;
}

// lane k's value, k a constant
__device__ __forceinline__ double lane_value(double v, int k)
{
    union {
        double d;
        int i[2];
    } u{v};
    u.i[0] = __builtin_amdgcn_readlane(u.i[0], k);
    u.i[1] = __builtin_amdgcn_readlane(u.i[1], k);
    return u.d;
}

// The Anderson step of the device-driven loop on one wave: the step partials
// reduced across the wave in a fixed order, then the residual and convergence
// test, the restart safeguard, the Gram matrix of the differences in use
// (kept oldest first, the newest row from this step), the regularized
// Cholesky solve of the least-squares problem and the update coefficients,
// and the history extension for the next iteration.
//
// The solve is one chain of 16 pivots.  Lane i holds row i of the matrix in
// registers, pivot rows and multipliers reach the other lanes as lane reads
// (scalar registers), and the row of a pivot, which is l_kk times column k of
// the factor, serves the back substitution where it lies; one reciprocal
// square root per pivot takes the place of a root and two divisions.  The step
// of 500 linear elements took 23 us with the matrix in LDS and takes 12.6, the
// transposed one, formerly 60 us over six launches and a wait, 11.3.
__device__ inline void anderson_wave(int64_t nb, const double* __restrict__ partials, RelaxDevState* __restrict__ st)
{
    constexpr int H = kHistMax;
    __shared__ double sv[2 * H];
    const int lane = threadIdx.x & 63, row = lane & (H - 1);
    const int hist = st->hist;
    const int head = st->head;
    // live part of the Gram matrix (rows and columns but the newest)
    double g[H];
#pragma unroll
    for (int c = 0; c < H; c++) g[c] = (row < hist - 1 && c < hist - 1) ? st->G[row * H + c] : 0.0;
    double v0 = 0.0, v1 = 0.0, v2 = 0.0, v[2 * H];
#pragma unroll
    for (int k = 0; k < 2 * H; k++) v[k] = 0.0;
    for (int64_t b = lane; b < nb; b += 64) {
        const double* o = partials + int64_t(kRelaxPart) * b;
        v0 += o[0];
        v1 = fmax(v1, o[1]);
        v2 = fmax(v2, o[2]);
#pragma unroll
        for (int k = 0; k < 2 * H; k++) v[k] += o[3 + k];
    }
    v0 = wave_sum(v0);
    v1 = wave_max(v1);
    v2 = wave_max(v2);
    const double dots = wave_sum32(v, lane);
    if ((lane & 1) == 0) sv[lane >> 1] = dots;
    __syncthreads();
    // wave-uniform decisions (every lane reads the same state)
    const int it = st->it + 1;
    const double misfit = sqrt(v0 / st->n);
    const bool finite = isfinite(misfit);
    const bool finish = !finite || misfit <= st->prec || it >= st->max_iter;
    const bool restart = !finish && misfit > 1e4 * st->best;
    const double best = fmin(st->best, misfit);
    const double beta = restart ? fmax(0.05, 0.5 * st->beta) : st->beta;
    bool ok = !finish && !restart && hist > 0;
    double gam = 0.0;  // of difference `row`
    if (ok) {
        const double newest = (row < hist) ? sv[row] : 0.0;
        double z = (row < hist) ? sv[H + row] : 0.0;
        double tr = 0.0;
#pragma unroll
        for (int c = 0; c < H; c++) {
            if (c == hist - 1) g[c] = newest;
            else if (row == hist - 1 && c < hist) g[c] = sv[c];
            tr += lane_value(g[c], c);
        }
        const double lam = 1e-10 * (tr > 0 ? tr / hist : 1.0);
        double a[H];
#pragma unroll
        for (int c = 0; c < H; c++) a[c] = g[c] + ((row == c && c < hist) ? lam : 0.0);
        double own = 0.0;  // 1 / l of this lane's row
#pragma unroll
        for (int k = 0; k < H; k++) {
            if (k >= hist || !ok) continue;
            const double d = lane_value(a[k], k);
            if (!(d > 0.0)) {
                ok = false;
                continue;
            }
            // 1/sqrt(d) from the seed y: e = 1 - d y^2, y (1 + e/2 + 3 e^2/8)
            const double y = __builtin_amdgcn_rsq(d);
            const double e = fma(-(d * y), y, 1.0);
            const double inv = fma(y * e, fma(e, 0.375, 0.5), y);
            const double l = (row > k) ? a[k] * inv : 0.0;  // L_row,k below the pivot
#pragma unroll
            for (int c = k + 1; c < H; c++) a[c] = fma(-l, lane_value(l, c), a[c]);
            const double zk = lane_value(z, k) * inv;  // L z = r on the way
            z = (row == k) ? zk : fma(-l, zk, z);
            if (row == k) own = inv;
        }
        // L^T gam = z: row k still holds l_kk L_ck in a[c], c > k
#pragma unroll
        for (int c = H - 1; c >= 0; c--) {
            if (c >= hist || !ok) continue;
            const double gc = lane_value(z * own, c);
            if (row < c) z = fma(-(a[c] * own), gc, z);
        }
        gam = z * own;
    }
    // state of the next iteration
    if (lane == 0) {
        st->arrive = 0;  // every block of this step has arrived
        st->it = it;
        st->misfit = misfit;
        st->maxM = fmax(1e-17, v1);
        st->maxH = fmax(1e-17, v2);
        if (!finite) {
            st->fail = 1;
            st->done = 2;
        } else if (misfit <= st->prec && it == 1 && st->keep_if_converged) {
            st->done = 2;
        } else if (finish) {
            st->done = 1;
        } else {
            const int nh = ok ? hist : 0, hd = ok ? head : 0;
            st->best = best;
            st->beta = beta;
            st->cF = beta;
            // the next iteration writes a new difference into slot hd
            st->ext = 1;
            st->head = (hd + 1) % H;
            st->hist = nh + 1 < H ? nh + 1 : H;
        }
    }
    if (!finish && lane < H) {
        // coefficients by buffer slot; the oldest difference lies in slot head - hist
        const int p = (head - hist + row + 2 * H) % H;
        const bool use = ok && row < hist;
        st->cdX[p] = use ? -gam : 0.0;
        st->cdF[p] = use ? -beta * gam : 0.0;
    }
    // the Gram matrix of the next iteration: the oldest difference drops out
    // when the history is full
    if (ok) {
        const int sh = (hist == H) ? 1 : 0;
#pragma unroll
        for (int c = 0; c < H; c++)
            if (lane < H && row >= sh && c >= sh) st->G[(row - sh) * H + c - sh] = g[c];
    }
}

// A step of the device-driven loop (history slots from the state); the last
// block to finish runs the Anderson step on the partials of all blocks.
template <class Law>
__device__ __forceinline__ void relax_step_dev(int64_t n, const Law& law, const double* __restrict__ M,
                                               double* __restrict__ F, double* __restrict__ partials,
                                               const HistBufs& hb, RelaxDevState* __restrict__ st)
{
    if (st->done) return;
    const int nh = st->hist, head = st->head;
    const double* dF[kHistMax];
#pragma unroll
    for (int k = 0; k < kHistMax; k++) dF[k] = hb.dF + ((head - nh + k + 2 * kHistMax) % kHistMax) * hb.stride;
    const int w = (head - 1 + kHistMax) % kHistMax;
    relax_step_block(n, law, M, F, partials, hb.Fp, hb.xp, st->ext ? hb.dF + w * hb.stride : nullptr,
                     st->ext ? hb.dX + w * hb.stride : nullptr, dF, nh);
    // release this block's partials, then count it in
    __threadfence();
    int arrived = 0;
    if (threadIdx.x == 0) arrived = atomicAdd(&st->arrive, 1);
    arrived = __shfl(arrived, 0, 64);
    if (arrived != int(gridDim.x) - 1) return;
    __threadfence();  // the other blocks' partials are visible to the last one
    anderson_wave(int64_t(gridDim.x), partials, st);
}

// x + cF F + sum_b (cdX[b] dX[b] + cdF[b] dF[b]) of one component.  All slots
// are loaded at once, also the unused ones, whose values are dropped: a branch
// per slot would make the loads a chain of 16 (5.4 us a launch; 4.3 now).
struct UpdateCoef {
    double cF, cX[kHistMax], cD[kHistMax];
    __device__ __forceinline__ explicit UpdateCoef(const RelaxDevState* st) : cF(st->cF)
    {
#pragma unroll
        for (int b = 0; b < kHistMax; b++) {
            cX[b] = st->cdX[b];
            cD[b] = st->cdF[b];
        }
    }
    __device__ __forceinline__ double apply(double xi, const double* F, const HistBufs& hb, int64_t i) const
    {
        double dx[kHistMax], df[kHistMax];
#pragma unroll
        for (int b = 0; b < kHistMax; b++) {
            dx[b] = hb.dX[b * hb.stride + i];
            df[b] = hb.dF[b * hb.stride + i];
        }
        double acc = xi + cF * F[i];
#pragma unroll
        for (int b = 0; b < kHistMax; b++)
            acc = (cX[b] != 0.0 || cD[b] != 0.0) ? acc + (cX[b] * dx[b] + cD[b] * df[b]) : acc;
        return acc;
    }
};

}  // namespace rh
