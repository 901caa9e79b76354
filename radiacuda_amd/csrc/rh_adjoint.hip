// rh_adjoint.hip -- gfx950 adjoint kernels: dL/dM and dL/d(vertex) of the
// field at observation points for given weights g = dL/dB, the transposed
// matrix pass and the per-element update of the linear-material adjoint
// relaxation.
//
// Mapping of dL/dM: as in the forward field sweep, each lane owns one
// observation point and every lane of the workgroup visits the same source
// elements (wave-uniform records); a lane's contribution to an element is
// summed over the wavefront with cross-lane shuffles and accumulated per wave
// in LDS.  dL/d(vertex) has it the other way round: a lane owns a triangle and
// visits the block's points.  In both, each workgroup writes one partial per
// element or vertex and a second kernel sums the partials in a fixed order, so
// gradients are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "rh_adjoint.hpp"
#include "rh_eval.hpp"
#include "rh_kernels.hpp"
#include "rh_relax_step.hpp"

namespace rh {

namespace {

constexpr int kAdjSliceE = 64;   // elements per workgroup slice (dL/dM), at most
constexpr int kAdjHex = 8;       // hexahedron records staged at a time (dL/dM)
constexpr int kAdjSliceV = 128;  // vertices per workgroup slice (dL/dvertex)

// dL/dM partials: part[bx][j][3] for the elements of slice blockIdx.y.
// FP64-issue bound where the blocks fill the chip: 1,000 hexahedra at 2,048
// points, 8 tiles, 279 us in 1,000 blocks of 8 elements and 816 us in 128
// blocks of 64; 165 us with hexahedron records from LDS (gen_block).
template <bool SYM>
__global__ __launch_bounds__(256, 2) void k_adj_m(DevModel m, const double* __restrict__ pts,
                                               int64_t np, const double* __restrict__ g,
                                               int addin, int slice, double* __restrict__ part)
{
    __shared__ double acc[4][kAdjSliceE * 3];
    __shared__ double hexes[kAdjHex * kHex];  // hexahedron records
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * kAdjSliceE * 3; i += 256) (&acc[0][0])[i] = 0.0;
    const int64_t j0 = int64_t(blockIdx.y) * slice;
    const int64_t j1 = (j0 + slice < m.n) ? (j0 + slice) : m.n;
    const int64_t tiles = (np + 255) / 256;
    for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int64_t p = tile * 256 + threadIdx.x;
        const bool live = p < np;
        const double x[3] = {live ? pts[3 * p] : 0.0, live ? pts[3 * p + 1] : 0.0,
                             live ? pts[3 * p + 2] : 0.0};
        const double gp[3] = {live ? g[3 * p] : 0.0, live ? g[3 * p + 1] : 0.0,
                              live ? g[3 * p + 2] : 0.0};
        for (int64_t j = j0; j < j1; j++) {
            const int r = int(j - j0) % kAdjHex;
            if (r == 0) {
                __syncthreads();  // the previous records have been consumed
                const int cnt = int((j1 - j < kAdjHex) ? (j1 - j) : kAdjHex);
                for (int i = threadIdx.x; i < cnt * kHex; i += 256) {
                    const int q = i / kHex, at = m.hex_at[j + q];
                    if (at >= 0) hexes[i] = m.hex[int64_t(kHex) * at + i - kHex * q];
                }
                __syncthreads();
            }
            const int kind = m.kind[j];
            const double* rec = m.data + m.off[j];
            const double* hex = (m.hex_at[j] >= 0) ? hexes + kHex * r : nullptr;
            double v[3] = {0.0, 0.0, 0.0};
            if (live) {
                for (int64_t c = m.copy_off[j]; c < m.copy_off[j + 1]; c++) {
                    const double* cp = m.copies + 24 * c;
                    double xl[3], q6[6], gl[3];
                    if (SYM) {
                        apply_inv(cp, x, xl);
                        // F^T g
                        for (int k = 0; k < 3; k++)
                            gl[k] = cp[12 + k] * gp[0] + cp[15 + k] * gp[1] + cp[18 + k] * gp[2];
                    } else {
                        for (int k = 0; k < 3; k++) {
                            xl[k] = x[k];
                            gl[k] = gp[k];
                        }
                    }
                    const bool in = hex ? gen_block(hex, rec, xl, q6) : eval_k<double, -1>(kind, rec, xl, q6);
                    const double e = (in && addin) ? 1.0 : 0.0;
                    v[0] += (q6[0] + e) * gl[0] + q6[3] * gl[1] + q6[4] * gl[2];
                    v[1] += q6[3] * gl[0] + (q6[1] + e) * gl[1] + q6[5] * gl[2];
                    v[2] += q6[4] * gl[0] + q6[5] * gl[1] + (q6[2] + e) * gl[2];
                }
            }
            for (int k = 0; k < 3; k++) {
                const double s = wave_sum(v[k]);
                if (lane == 0) acc[wave][3 * (j - j0) + k] += s;
            }
        }
    }
    __syncthreads();
    const int64_t cnt = 3 * (j1 - j0);
    for (int64_t i = threadIdx.x; i < cnt; i += 256)
        part[int64_t(blockIdx.x) * 3 * m.n + 3 * j0 + i] = acc[0][i] + acc[1][i] + acc[2][i] + acc[3][i];
}

// dL/dvertex partials: partv[bx][vertex slot][3] for the vertices of element
// slice [sl[y], sl[y+1]); optional per-point dL/dx partials partx[y][p][3].
//
// FP64-issue bound.  A lane holds one triangle (of one transform copy) of the
// slice in registers and walks the block's points, which lie in LDS and are the
// same for all lanes; the four waves take every fourth point.  A triangle's
// nine sums then cross lanes once per block instead of once per point, and
// what depends on the triangle alone is computed once per block; dL/dx, three
// sums, is the one that crosses lanes per point.  About 330 FP64 operations
// for all nine derivatives (forward-mode duals seeded per corner took some
// 2,700 and nine wave sums): 1,000 hexahedra at 2,048 points 0.35 ms instead
// of 5.4 ms, of which 0.3 ms is the operations' issue.
constexpr int kAdjTile = 128;  // points staged at a time
template <bool SYM, bool GX>
__global__ __launch_bounds__(256, 2) void k_adj_geom(DevModel m, const double* __restrict__ adj,
                                                  const int64_t* __restrict__ adj_off,
                                                  const int64_t* __restrict__ vert_off,
                                                  const int64_t* __restrict__ sl, int64_t nvert,
                                                  const double* __restrict__ M,
                                                  const double* __restrict__ pts, int64_t np, int64_t per_block,
                                                  const double* __restrict__ g,
                                                  double* __restrict__ partv,
                                                  double* __restrict__ partx)
{
    __shared__ double acc[3 * kAdjSliceV];
    __shared__ double xs[kAdjTile][6];
    __shared__ double lanes[4][9][64];
    __shared__ int corner[3][64];
    __shared__ double copy[SYM ? 21 : 1][64];  // every lane's transform copy
    __shared__ int first[kAdjSliceV + 1];  // first triangle of each element
    __shared__ int owner[kAdjSliceV];      // element of each vertex
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t j0 = sl[blockIdx.y], j1 = sl[blockIdx.y + 1];
    const int64_t v0 = vert_off[j0];
    const int nel = int(j1 - j0);  // at most kAdjSliceV
    for (int i = threadIdx.x; i < 3 * kAdjSliceV; i += 256) acc[i] = 0.0;
    for (int e = threadIdx.x; e < nel; e += 256) {
        first[e + 1] = adj_ntri(adj + adj_off[j0 + e]) * int(m.copy_off[j0 + e + 1] - m.copy_off[j0 + e]);
        for (int64_t v = vert_off[j0 + e]; v < vert_off[j0 + e + 1]; v++) owner[v - v0] = e;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        first[0] = 0;
        for (int e = 0; e < nel; e++) first[e + 1] += first[e];
    }
    __syncthreads();
    const int total = first[nel];
    const int64_t p0 = int64_t(blockIdx.x) * per_block;
    const int64_t p1 = (p0 + per_block < np) ? (p0 + per_block) : np;
    if (GX && total == 0)
        for (int64_t i = 3 * p0 + threadIdx.x; i < 3 * p1; i += 256) partx[int64_t(blockIdx.y) * 3 * np + i] = 0.0;
    for (int base = 0; base < total; base += 64) {
        // lanes past the end repeat the last triangle with M = 0
        const bool live = base + lane < total;
        const int item = live ? base + lane : total - 1;
        int el = 0;
        while (first[el + 1] <= item) el++;
        const int64_t j = j0 + el;
        const double* rec = adj + adj_off[j];
        const int nt = adj_ntri(rec);
        const double* tri = rec + 2 + 3 * adj_nv(rec) + 3 * ((item - first[el]) % nt);
        const double* cp = m.copies + 24 * (m.copy_off[j] + (item - first[el]) / nt);
        const int slot = int(vert_off[j] - v0);
        if (SYM && wave == 0)
            for (int k = 0; k < 21; k++) copy[k][lane] = cp[k];
        TriLane T;
        for (int k = 0; k < 3; k++) {
            const int id = int(tri[k]);
            if (wave == 0) corner[k][lane] = slot + id;
            T.v[k] = V3<double>{rec[2 + 3 * id], rec[3 + 3 * id], rec[4 + 3 * id]};
        }
        tri_open(T, live ? V3<double>{M[3 * j], M[3 * j + 1], M[3 * j + 2]} : V3<double>{0.0, 0.0, 0.0});
        for (int64_t q0 = p0; q0 < p1; q0 += kAdjTile) {
            const int cnt = int((p1 - q0 < kAdjTile) ? (p1 - q0) : kAdjTile);
            __syncthreads();
            for (int i = threadIdx.x; i < 3 * cnt; i += 256) {
                xs[i / 3][i % 3] = pts[3 * q0 + i];
                xs[i / 3][3 + i % 3] = kInv4Pi * g[3 * q0 + i];
            }
            __syncthreads();
            for (int i = wave; i < cnt; i += 4) {
                const double* z = xs[i];
                double x[3] = {z[0], z[1], z[2]};
                V3<double> gl{z[3], z[4], z[5]}, gx{0.0, 0.0, 0.0};
                if (SYM) {
                    double cm[21];
                    for (int k = 0; k < 21; k++) cm[k] = copy[k][lane];
                    apply_inv(cm, z, x);
                    gl.x = cm[12] * z[3] + cm[15] * z[4] + cm[18] * z[5];
                    gl.y = cm[13] * z[3] + cm[16] * z[4] + cm[19] * z[5];
                    gl.z = cm[14] * z[3] + cm[17] * z[4] + cm[20] * z[5];
                }
                tri_point(T, x, gl, gx);
                if (GX) {
                    double d[3] = {gx.x, gx.y, gx.z};
                    if (SYM)
                        for (int a = 0; a < 3; a++)
                            d[a] = copy[a][lane] * gx.x + copy[3 + a][lane] * gx.y + copy[6 + a][lane] * gx.z;
                    for (int a = 0; a < 3; a++) d[a] = wave_sum(d[a]);
                    if (lane < 3) {
                        // the wave's own point: earlier triangles' sum, then these
                        double* o = partx + (int64_t(blockIdx.y) * np + q0 + i) * 3 + lane;
                        const double s = (lane == 0) ? d[0] : (lane == 1 ? d[1] : d[2]);
                        *o = (base == 0) ? s : *o + s;
                    }
                }
            }
        }
        V3<double> G[3];
        tri_close(T, G);
        for (int k = 0; k < 3; k++) {
            lanes[wave][3 * k][lane] = G[k].x;
            lanes[wave][3 * k + 1][lane] = G[k].y;
            lanes[wave][3 * k + 2][lane] = G[k].z;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 9 * 64; i += 256)
            (&lanes[0][0][0])[i] += (&lanes[1][0][0])[i] + (&lanes[2][0][0])[i] + (&lanes[3][0][0])[i];
        __syncthreads();
        // each vertex coordinate sums its corners in order
        for (int i = threadIdx.x; i < 3 * int(vert_off[j1] - v0); i += 256) {
            const int v = i / 3, a = i % 3;
            const int l0 = max(0, first[owner[v]] - base), l1 = min(64, first[owner[v] + 1] - base);
            double s = acc[i];
            for (int l = l0; l < l1; l++)
                for (int k = 0; k < 3; k++)
                    if (corner[k][l] == v) s += lanes[0][3 * k + a][l];
            acc[i] = s;
        }
        __syncthreads();
    }
    const int64_t cnt = 3 * (vert_off[j1] - v0);
    for (int64_t i = threadIdx.x; i < cnt; i += 256)
        partv[int64_t(blockIdx.x) * 3 * nvert + 3 * v0 + i] = acc[i];
}

// out[i] = sum_k part[k * stride + i], i < len: 256 / G columns to a block, G
// threads to a column, each summing every G-th row, then in order over the
// threads.  93 rows of 1,500 columns: 21 us with a thread per column (a chain
// of 93 loads in 6 blocks), 3.6 us with 16.
template <int G>
__global__ __launch_bounds__(256) void k_sum_parts(int64_t len, int64_t ns, int64_t stride,
                                                   const double* __restrict__ part,
                                                   double* __restrict__ out, const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    constexpr int C = 256 / G;
    __shared__ double red[G][C];
    const int c = threadIdx.x % C, r = threadIdx.x / C;
    const int64_t i = int64_t(blockIdx.x) * C + c;
    double s = 0.0;
    if (i < len) {
#pragma unroll 8
        for (int64_t k = r; k < ns; k += G) s += part[k * stride + i];
    }
    if (G > 1) {
        red[r][c] = s;
        __syncthreads();
        if (r > 0) return;
#pragma unroll
        for (int k = 1; k < G; k++) s += red[k][c];
    }
    if (i < len) out[i] = s;
}

void sum_parts(int64_t len, int64_t ns, int64_t stride, const double* part, double* out, hipStream_t s,
               const int32_t* skip = nullptr)
{
    auto go = [&](auto g) {
        constexpr int G = decltype(g)::value;
        const int64_t cols = 256 / G;
        hipLaunchKernelGGL(k_sum_parts<G>, dim3(unsigned((len + cols - 1) / cols)), dim3(256), 0, s, len, ns, stride,
                           part, out, skip);
    };
    // up to 16 rows a thread's chain is one round of loads
    if (ns <= 16) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, 16>{});
}

// Transposed matrix pass: part[rc][col] = sum over rows of chunk rc of
// Q[r][col] x[r]; each lane owns 4 consecutive columns (16-byte FP32 or 2x16
// byte FP64 loads along the row), rows of a chunk are streamed in order.
template <class T>
__global__ __launch_bounds__(256) void k_matvec_t(const T* __restrict__ Q, int64_t nrows, int64_t ld,
                                                  int64_t rows_per_chunk, const double* __restrict__ x,
                                                  double* __restrict__ part, const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const int64_t c0 = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
    const int64_t r0 = int64_t(blockIdx.y) * rows_per_chunk;
    const int64_t r1 = (r0 + rows_per_chunk < nrows) ? (r0 + rows_per_chunk) : nrows;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (c0 < ld) {
        for (int64_t r = r0; r < r1; r++) {
            const T* row = Q + r * ld + c0;
            const double xr = x[r];
#pragma unroll
            for (int k = 0; k < 4; k++) acc[k] += double(row[k]) * xr;
        }
        double* o = part + int64_t(blockIdx.y) * ld + c0;
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = acc[k];
    }
}

// Transposed pass over the symmetric-block layout: every stored block is
// symmetric, so (Q^T x)_j = sum_i Q_ij x_i; part[rc][3j + a] sums the element
// rows of chunk rc.  Each lane owns two consecutive column elements.
template <class T, int P>
__global__ __launch_bounds__(256) void k_matvec_t_sym(const T* __restrict__ Q, int64_t nel, int64_t ldp,
                                                      int64_t el_per_chunk, const double* __restrict__ x,
                                                      double* __restrict__ part, int64_t ld,
                                                      const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const int64_t j0 = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 2;
    const int64_t i0 = int64_t(blockIdx.y) * el_per_chunk;
    const int64_t i1 = (i0 + el_per_chunk < nel) ? (i0 + el_per_chunk) : nel;
    if (j0 >= ldp) return;
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int64_t i = i0; i < i1; i++) {
        const T* b = Q + i * P * ldp + j0;
        const double x0 = x[3 * i], x1 = x[3 * i + 1], x2 = x[3 * i + 2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const double xx = double(b[e]), xy = double(b[ldp + e]), xz = double(b[2 * ldp + e]);
            const double yy = double(b[3 * ldp + e]), yz = double(b[4 * ldp + e]);
            const double zz = (P == 6) ? double(b[5 * ldp + e]) : -(xx + yy);
            acc[3 * e] += xx * x0 + xy * x1 + xz * x2;
            acc[3 * e + 1] += xy * x0 + yy * x1 + yz * x2;
            acc[3 * e + 2] += xz * x0 + yz * x1 + zz * x2;
        }
    }
    double* o = part + int64_t(blockIdx.y) * ld + 3 * j0;
#pragma unroll
    for (int k = 0; k < 6; k++) o[k] = acc[k];
}

// Linear susceptibility tensor of an element (element frame).
__device__ __forceinline__ void lin_tensor(const double* mat, double K[9])
{
    if (int(mat[0]) == 0) {
        for (int k = 0; k < 9; k++) K[k] = 0.0;
        K[0] = K[4] = K[8] = mat[1];
    } else {
        for (int k = 0; k < 9; k++) K[k] = mat[4 + k];
    }
}

// mu = K^T lam
__device__ __forceinline__ void adj_scale(const double* mat, const double l[3], double* mu)
{
    double K[9];
    lin_tensor(mat, K);
    for (int a = 0; a < 3; a++) mu[a] = K[a] * l[0] + K[3 + a] * l[1] + K[6 + a] * l[2];
}

__global__ __launch_bounds__(256) void k_adj_scale(int64_t n, const double* __restrict__ mats,
                                                   const double* __restrict__ lam,
                                                   double* __restrict__ mu)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const double l[3] = {lam[3 * i], lam[3 * i + 1], lam[3 * i + 2]};
    adj_scale(mats + 16 * i, l, mu + 3 * i);
}

// Block-Jacobi update of the transposed system (I - Q^T K^T) lam = rhs:
// lam_new_i = (I - Qii^T K_i^T)^{-1} (rhs_i + y_i), y = offdiag(Q)^T K^T lam.
struct TransposedLaw {
    const double *mats, *rhs, *qdiag, *y;
    __device__ __forceinline__ void operator()(int64_t i, double* nl, double&) const
    {
        double K[9];
        lin_tensor(mats + 16 * i, K);
        const double* D = qdiag + 9 * i;
        // A = I - D^T K^T = I - (K D)^T
        double KD[9], A[9], Ai[9];
        for (int a = 0; a < 3; a++)
            for (int b = 0; b < 3; b++)
                KD[3 * a + b] = K[3 * a] * D[b] + K[3 * a + 1] * D[3 + b] + K[3 * a + 2] * D[6 + b];
        for (int a = 0; a < 3; a++)
            for (int b = 0; b < 3; b++) A[3 * a + b] = (a == b ? 1.0 : 0.0) - KD[3 * b + a];
        const double det = A[0] * (A[4] * A[8] - A[5] * A[7]) - A[1] * (A[3] * A[8] - A[5] * A[6]) +
                           A[2] * (A[3] * A[7] - A[4] * A[6]);
        const double id = 1.0 / det;
        Ai[0] = (A[4] * A[8] - A[5] * A[7]) * id;
        Ai[1] = (A[2] * A[7] - A[1] * A[8]) * id;
        Ai[2] = (A[1] * A[5] - A[2] * A[4]) * id;
        Ai[3] = (A[5] * A[6] - A[3] * A[8]) * id;
        Ai[4] = (A[0] * A[8] - A[2] * A[6]) * id;
        Ai[5] = (A[2] * A[3] - A[0] * A[5]) * id;
        Ai[6] = (A[3] * A[7] - A[4] * A[6]) * id;
        Ai[7] = (A[1] * A[6] - A[0] * A[7]) * id;
        Ai[8] = (A[0] * A[4] - A[1] * A[3]) * id;
        const double r[3] = {rhs[3 * i] + y[3 * i], rhs[3 * i + 1] + y[3 * i + 1],
                             rhs[3 * i + 2] + y[3 * i + 2]};
        for (int a = 0; a < 3; a++) nl[a] = Ai[3 * a] * r[0] + Ai[3 * a + 1] * r[1] + Ai[3 * a + 2] * r[2];
    }
};

__global__ __launch_bounds__(kRelaxLanes) void k_adj_step_dev(int64_t n, TransposedLaw law,
                                                              const double* __restrict__ lam,
                                                              double* __restrict__ F,
                                                              double* __restrict__ partials, HistBufs hb,
                                                              RelaxDevState* __restrict__ st)
{
    relax_step_dev(n, law, lam, F, partials, hb, st);
}

// The update of lam and the next matrix pass's input mu = K^T lam.
__global__ __launch_bounds__(kRelaxLanes) void k_adj_update_dev(int64_t n, const double* __restrict__ mats,
                                                                double* __restrict__ lam, double* __restrict__ mu,
                                                                const double* __restrict__ F, HistBufs hb,
                                                                double* __restrict__ lam_out,
                                                                const RelaxDevState* __restrict__ st)
{
    const int done = st->done;
    if (done == 2) return;
    const int64_t i = int64_t(blockIdx.x) * kRelaxLanes + threadIdx.x;
    if (i >= n) return;
    if (done == 1) {
        for (int k = 0; k < 3; k++) lam_out[3 * i + k] = lam[3 * i + k] + F[3 * i + k];
        return;
    }
    const UpdateCoef c(st);
    double l[3];
    for (int k = 0; k < 3; k++) {
        l[k] = c.apply(lam[3 * i + k], F, hb, 3 * i + k);
        lam[3 * i + k] = l[k];
    }
    adj_scale(mats + 16 * i, l, mu + 3 * i);
}

}  // namespace

int64_t adj_point_groups(int64_t np, int64_t slices)
{
    const int64_t tiles = (np + 255) / 256;
    int64_t pg = std::max<int64_t>(1, (2048 + slices - 1) / std::max<int64_t>(1, slices));
    return std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(pg, tiles), 64));
}

// Groups of points of the geometry pass: blocks for four a compute unit, each
// with at least 16 points (four a wave) to spread the triangles' set-up over.
int64_t adj_geom_groups(int64_t np, int64_t slices)
{
    const int64_t g = std::min<int64_t>((np + 15) / 16, 1024 / std::max<int64_t>(1, slices));
    return std::max<int64_t>(1, std::min<int64_t>(g, 64));
}

// Elements per slice of the dL/dM sweep: 64, fewer where the tiles of 256 points
// do not fill the chip (down to 4, below which the blocks' own reductions show).
static int adj_m_slice(int64_t n, int64_t np)
{
    const int64_t tiles = (np + 255) / 256;
    int e = kAdjSliceE;
    while (e > 4 && tiles * ((n + e - 1) / e) < 1000) e /= 2;
    return e;
}

int64_t adj_m_slices(int64_t n, int64_t np)
{
    const int e = adj_m_slice(n, np);
    return (n + e - 1) / e;
}

std::vector<int64_t> adj_geom_slices(const std::vector<int64_t>& vert_off, std::string* err)
{
    std::vector<int64_t> sl{0};
    const int64_t n = int64_t(vert_off.size()) - 1;
    for (int64_t j = 0; j < n; j++) {
        const int64_t nv = vert_off[j + 1] - vert_off[j];
        if (nv > kAdjSliceV) {
            if (err) *err = "element with more than 128 vertices";
            return {};
        }
        if (vert_off[j + 1] - vert_off[sl.back()] > kAdjSliceV || j - sl.back() >= kAdjSliceV) sl.push_back(j);
    }
    sl.push_back(n);
    return sl;
}

hipError_t launch_adj_m(const DevModel& m, const double* pts, int64_t np, const double* g, bool addin,
                        double* part, int64_t groups, double* gM, hipStream_t s)
{
    const int64_t ns = adj_m_slices(m.n, np);
    const int slice = adj_m_slice(m.n, np);
    const dim3 grid{unsigned(groups), unsigned(ns), 1u};
    if (m.sym)
        hipLaunchKernelGGL(k_adj_m<true>, grid, dim3(256), 0, s, m, pts, np, g, addin ? 1 : 0, slice, part);
    else
        hipLaunchKernelGGL(k_adj_m<false>, grid, dim3(256), 0, s, m, pts, np, g, addin ? 1 : 0, slice, part);
    const int64_t len = 3 * m.n;
    sum_parts(len, groups, len, part, gM, s);
    return hipGetLastError();
}

hipError_t launch_adj_geom(const DevModel& m, const double* adj, const int64_t* adj_off,
                           const int64_t* vert_off, const int64_t* sl, int64_t nslices,
                           int64_t nvert, const double* M, const double* pts, int64_t np,
                           const double* g, double* partv, double* partx, int64_t groups,
                           double* gV, double* gX, hipStream_t s)
{
    const dim3 grid{unsigned(groups), unsigned(nslices), 1u};
    const int64_t per = (np + groups - 1) / groups;
    auto k = m.sym ? (gX ? k_adj_geom<true, true> : k_adj_geom<true, false>)
                   : (gX ? k_adj_geom<false, true> : k_adj_geom<false, false>);
    hipLaunchKernelGGL(k, grid, dim3(256), 0, s, m, adj, adj_off, vert_off, sl, nvert, M, pts, np, per, g, partv,
                       partx);
    if (gV) {
        const int64_t len = 3 * nvert;
        sum_parts(len, groups, len, partv, gV, s);
    }
    if (gX) {
        const int64_t len = 3 * np;
        sum_parts(len, nslices, len, partx, gX, s);
    }
    return hipGetLastError();
}

int64_t matvec_t_chunks(int64_t nrows, int64_t ld)
{
    const int64_t ctiles = (ld + 1023) / 1024;
    int64_t ch = std::max<int64_t>(1, (4096 + ctiles - 1) / ctiles);
    ch = std::min<int64_t>(ch, std::max<int64_t>(1, nrows / 16));
    return std::min<int64_t>(ch, 256);
}

hipError_t launch_matvec_t(const void* Q, int elem_bytes, int64_t nrows, int64_t ld, const double* x,
                           double* part, int64_t chunks, double* y, hipStream_t s, const int32_t* skip)
{
    const int64_t rpc = (nrows + chunks - 1) / chunks;
    const dim3 grid{unsigned((ld + 1023) / 1024), unsigned(chunks), 1u};
    if (elem_bytes == 4)
        hipLaunchKernelGGL(k_matvec_t<float>, grid, dim3(256), 0, s, static_cast<const float*>(Q),
                           nrows, ld, rpc, x, part, skip);
    else
        hipLaunchKernelGGL(k_matvec_t<double>, grid, dim3(256), 0, s, static_cast<const double*>(Q),
                           nrows, ld, rpc, x, part, skip);
    sum_parts(nrows, chunks, ld, part, y, s, skip);
    return hipGetLastError();
}

hipError_t launch_matvec_t_sym(const void* Q, int elem_bytes, int planes, int64_t nel, int64_t ldp,
                               const double* x, double* part, int64_t chunks, double* y, hipStream_t s,
                               const int32_t* skip)
{
    if ((planes != 5 && planes != 6) || ldp % 256 != 0 || chunks < 1) return hipErrorInvalidValue;
    const int64_t epc = (nel + chunks - 1) / chunks;
    const int64_t ld = 3 * ldp;
    const dim3 grid{unsigned((ldp / 2 + 255) / 256), unsigned(chunks), 1u};
    if (elem_bytes == 4) {
        const float* q = static_cast<const float*>(Q);
        if (planes == 5)
            hipLaunchKernelGGL((k_matvec_t_sym<float, 5>), grid, dim3(256), 0, s, q, nel, ldp, epc, x, part, ld, skip);
        else
            hipLaunchKernelGGL((k_matvec_t_sym<float, 6>), grid, dim3(256), 0, s, q, nel, ldp, epc, x, part, ld, skip);
    } else {
        const double* q = static_cast<const double*>(Q);
        if (planes == 5)
            hipLaunchKernelGGL((k_matvec_t_sym<double, 5>), grid, dim3(256), 0, s, q, nel, ldp, epc, x, part, ld, skip);
        else
            hipLaunchKernelGGL((k_matvec_t_sym<double, 6>), grid, dim3(256), 0, s, q, nel, ldp, epc, x, part, ld, skip);
    }
    sum_parts(3 * nel, chunks, ld, part, y, s, skip);
    return hipGetLastError();
}

hipError_t launch_adj_scale(int64_t n, const double* mats, const double* lam, double* mu, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_scale, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, n, mats, lam, mu);
    return hipGetLastError();
}

hipError_t launch_adj_step_dev(int64_t n, const double* mats, const double* rhs, const double* qdiag, const double* y,
                               const double* lam, double* F, double* partials, const HistBufs& hb,
                               RelaxDevState* st, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_step_dev, dim3(unsigned(relax_blocks(n))), dim3(kRelaxLanes), 0, s, n,
                       TransposedLaw{mats, rhs, qdiag, y}, lam, F, partials, hb, st);
    return hipGetLastError();
}

hipError_t launch_adj_update_dev(int64_t n, const double* mats, double* lam, double* mu, const double* F,
                                 const HistBufs& hb, double* lam_out, const RelaxDevState* st, hipStream_t s)
{
    hipLaunchKernelGGL(k_adj_update_dev, dim3(unsigned(relax_blocks(n))), dim3(kRelaxLanes), 0, s, n, mats, lam, mu, F,
                       hb, lam_out, st);
    return hipGetLastError();
}

}  // namespace rh
