// rh_kernels.hip -- gfx950 kernels: interaction-matrix assembly, field
// evaluation, the relaxation's matrix pass and per-element update, and
// current-source fields.
//
// Mapping (wave64): in the assembly and field kernels each lane owns one
// observation point (a matrix row's collocation point, or a field point) and
// every lane of the workgroup sweeps the same source elements, so element
// records are read at wave-uniform addresses (from LDS where a sweep is long
// enough to stage them, otherwise through the scalar cache; no
// per-lane gathers) and the per-element branches are uniform.  These kernels
// are bound by FP64 transcendental/VALU throughput.  The matrix pass streams
// the matrix once per iteration with 16-byte non-temporal loads and FP64
// accumulation; it is bound by HBM bandwidth.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "rh_current.hpp"
#include "rh_eval.hpp"
#include "rh_far.hpp"
#include "rh_geom.hpp"
#include "rh_kernels.hpp"
#include "rh_relax_step.hpp"
#include "rh_mesh.hpp"

namespace rh {

namespace {

__host__ __device__ __forceinline__ ModelView view(const DevModel& m)
{
    return ModelView{m.kind, m.off, m.data, m.copy_off, m.copies, m.charged, m.koff[1]};
}

// Field-only tetrahedron records for magnetization M (one lane per tetrahedron).
__global__ __launch_bounds__(256) void k_charge_tets(DevModel m, const double* __restrict__ M,
                                                     double* __restrict__ out)
{
    const int64_t k = m.koff[1] + int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (k >= m.koff[2]) return;
    const int64_t j = m.kidx[k];
    const double mm[3] = {M[3 * j], M[3 * j + 1], M[3 * j + 2]};
    charge_tet(m.data + m.off[j], mm, out + kChargedTet * (k - m.koff[1]));
}

// Far-form records of the tetrahedra (one lane each).
__global__ __launch_bounds__(256) void k_far_records(DevModel m, double* __restrict__ out)
{
    const int64_t k = m.koff[1] + int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (k >= m.koff[2]) return;
    far_tet_record(m.data + m.off[m.kidx[k]], out + kFarTet * (k - m.koff[1]));
}

// Far-form records of the hexahedra among the general polyhedra, one wave each,
// at the places that `at` gives; an element that does not fit the topology has
// none.
__global__ __launch_bounds__(64) void k_hex_records(DevModel m, double* __restrict__ out, int32_t* __restrict__ at)
{
    __shared__ double rec[kHexIn], o[kHex];
    __shared__ int id[8];
    __shared__ int ok;
    const int64_t j = m.kidx[m.koff[2] + blockIdx.x];
    const int64_t q = at[j];
    if (q < 0) return;
    const double* src = m.data + m.off[j];
    for (int i = threadIdx.x; i < kHexIn; i += 64) rec[i] = src[i];
    __syncthreads();
    if (threadIdx.x == 0) ok = hex_vertices(rec, id) ? 1 : 0;
    __syncthreads();
    bool fits = ok;
    if (fits && threadIdx.x < 12) fits = hex_edge_record(rec, id, threadIdx.x, o);
    else if (fits && threadIdx.x < 17) fits = hex_face_record(rec, id, threadIdx.x - 12, o);
    if (__any(!fits)) {
        if (threadIdx.x == 0) at[j] = -1;
        return;
    }
    __syncthreads();
    if (threadIdx.x == 0) hex_close_record(rec, id, o);
    __syncthreads();
    for (int i = threadIdx.x; i < kHex; i += 64) out[kHex * q + i] = o[i];
}

template <class T>
__device__ __forceinline__ void store_out(T* p, double v) { *p = T(v); }

// ---------------------------------------------------------------- assembly
// Rows of elements [r0, r1) into Q (Q holds row 3*r0 first); block columns
// are the elements kidx[k0 .. k1) of one kind slot.  A workgroup's four waves
// own the same 64 row elements (one per lane) and split the sources of a tile
// between them, sweeping uniform records; the lanes' 3x3 blocks of the tile's
// S sources are staged in one LDS tile, and the 256 threads write its rows as
// contiguous segments of 128 bytes (symmetric-block planes: 16 sources in FP64,
// 32 in FP32) or 192 bytes (row-major blocks: 8 and 16 sources).  Sources
// whose columns are not consecutive (mixed kinds) are stored directly.
//
// Measured with the integrals left out, the stores alone take (8,000 rows,
// FP64 planes) 2.09 ms in 32-byte segments, 1.03 in 64-byte and 0.72 in
// 128-byte ones, which fill whole lines.  With one wave per tile 128-byte
// segments leave LDS for one wave per SIMD; four waves to a tile allow three.
// Tetrahedra take the far form of rh_far.hpp, staged through LDS, where every
// lane is far (84 % of the sources a wave of the C-yoke meets, 92 % on the
// 24,000-tetrahedron yoke).  Measured: C-yoke FP64 2.09 -> 1.35 ms; 23,999
// tetrahedra mixed 14.05 -> 8.4 ms; 1,500 blocks x 4 copies mixed 259 -> 240 us.
// What bounds it now: vector issue about half of the time, the rest the four
// waves' wait for the one that met near sources, and the stores' 0.72 ms.
//
// Symmetric-block layout (PK = 5 or 6): without transform copies and row
// transforms every block is the symmetric tensor Q(x_i) of source j, so an
// element row is stored as PK planes (xx, xy, xz, yy, yz[, zz]) of ld values,
// plane k holding entry k of the blocks (i, 0 .. n-1); with PK = 5 the zz
// entry is -(xx + yy), exact for a collocation point outside the source.  A
// block with a trace beyond 1/4 (a collocation point inside another element)
// sets *flag, and the caller stores the matrix with 6 planes instead.
#ifndef RH_ASM_S64
#define RH_ASM_S64 8
#endif
#ifndef RH_ASM_S32
#define RH_ASM_S32 16
#endif
#ifndef RH_ASM_P64
#define RH_ASM_P64 16
#endif
#ifndef RH_ASM_P32
#define RH_ASM_P32 32
#endif
template <class OUT, int PK>
struct AsmTile {
    static constexpr int RPE = PK ? PK : 3;  // stored rows per element row
    static constexpr int VPS = PK ? 1 : 3;   // values per source in a stored row
    static constexpr int S = PK ? ((sizeof(OUT) == 8) ? RH_ASM_P64 : RH_ASM_P32)
                                : ((sizeof(OUT) == 8) ? RH_ASM_S64 : RH_ASM_S32);  // sources per tile
    static constexpr int U = VPS * S * int(sizeof(OUT)) / 8;  // 8-byte units per row segment
    static constexpr int EPU = 8 / int(sizeof(OUT));          // elements per 8-byte unit
    // LDS row stride (elements): row-major tiles pad a unit against bank
    // conflicts; plane tiles are unpadded with the units of the rows of lane l
    // stored at unit index u ^ (l & SWZ) instead
    static constexpr int W = (PK ? U : U + 1) * EPU;
    static constexpr int SWZ = PK ? U - 1 : 0;
    static_assert(!PK || (U & (U - 1)) == 0, "plane tiles swizzle a power-of-two number of units");
    // element index of element c of tile row r (rows RPE l .. RPE l + RPE - 1 belong to lane l)
    __device__ static int at(int r, int c) { return r * W + (((c / EPU) ^ ((r / RPE) & SWZ)) * EPU + c % EPU); }
};

// occupancy floor (waves per SIMD): tetrahedra 3 (the LDS tiles allow 3), the
// other kinds 2 (their integrals need more than 168 registers)
template <int KIND, bool SYM>
constexpr int asm_waves() { return KIND == 1 ? (SYM ? 2 : 3) : 2; }
// far-form tetrahedron records staged at a time
constexpr int kFarChunk = 16;
static_assert(kFarTet % 2 == 0, "16-byte loads of whole records");
// FAR32: far blocks in FP32 arithmetic, near ones in FP64 (block_Q_mixed).
// PK: 0 row-major 3x3 blocks, 5 or 6 the symmetric-block planes (then ld is
// the plane stride and SYM, ROWT are false).
template <class R, bool SYM, bool ROWT, class OUT, int KIND, bool FAR32 = false, int PK = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(asm_waves<KIND, SYM>()))) void
k_assemble(DevModel m, OUT* __restrict__ Q, int64_t ld, double* __restrict__ qdiag, int64_t jt, int64_t r0, int64_t r1,
           int32_t* __restrict__ flag)
{
    static_assert(PK == 0 || (!SYM && !ROWT), "the symmetric-block layout needs lab-frame blocks");
    using TL = AsmTile<OUT, PK>;
    constexpr int S = TL::S, W = TL::W, RPE = TL::RPE, VPS = TL::VPS;
    static_assert(S % 4 == 0 && S <= 32, "a quarter of the tile's sources per wave, one bit each");
    __shared__ __align__(16) OUT tile[RPE * 64 * W];
    // tetrahedra: the far records of the next CH sources, fetched one chunk
    // ahead into registers.  (Read through the scalar cache a record's 620
    // bytes cost six dependent batches of scalar loads, each a miss of its
    // own wave: 2.8 ms on the C-yoke with one wave per tile, against 2.1
    // without the far form.)
    constexpr bool kFar = KIND == 1;
    constexpr int CH = S < kFarChunk ? S : kFarChunk;
    constexpr int kLoads = (CH * kFarTet / 2 + 255) / 256;
    __shared__ __align__(16) double fsrc[kFar ? CH * kFarTet : 2];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int64_t i0 = r0 + int64_t(blockIdx.x) * 64;
    const int64_t i = i0 + lane;
    const bool live = i < r1;
    const int nrow = int((r1 - i0 < 64) ? (r1 - i0) : 64);
    const int64_t kend = m.koff[KIND + 1];
    const int64_t k0 = m.koff[KIND] + int64_t(blockIdx.y) * jt;
    const int64_t k1 = (k0 + jt < kend) ? (k0 + jt) : kend;
    const ModelView mv = view(m);
    const int64_t ic = live ? i : i0;  // idle lanes evaluate row i0 and store nothing
    const double x[3] = {m.colloc[3 * ic], m.colloc[3 * ic + 1], m.colloc[3 * ic + 2]};
    double rt[9];
    if (ROWT)
        for (int k = 0; k < 9; k++) rt[k] = m.rowt[9 * ic + k];
    OUT* row = Q + (RPE * (ic - r0)) * ld;
    bool traced = false;
    double2 ahead[kFar ? kLoads : 1];
    auto fetch = [&](int64_t k) {
        if constexpr (kFar) {
            const double2* src = reinterpret_cast<const double2*>(m.far_tet + kFarTet * (k - m.koff[1]));
            const int cnt = int((k1 - k < CH) ? (k1 - k) : CH) * (kFarTet / 2);
#pragma unroll
            for (int t = 0; t < kLoads; t++)
                if (int(threadIdx.x) + 256 * t < cnt) ahead[t] = src[threadIdx.x + 256 * t];
        }
    };
    auto chunk = [&](int64_t k) {
        if constexpr (kFar) {
            __syncthreads();  // the previous chunk has been consumed
            double2* dst = reinterpret_cast<double2*>(fsrc);
#pragma unroll
            for (int t = 0; t < kLoads; t++)
                if (int(threadIdx.x) + 256 * t < CH * (kFarTet / 2)) dst[threadIdx.x + 256 * t] = ahead[t];
            __syncthreads();
            if (k + CH < k1) fetch(k + CH);
        }
    };
    if constexpr (kFar) {
#pragma unroll
        for (int t = 0; t < kLoads; t++) ahead[t] = double2{0.0, 0.0};
        fetch(k0);
    }
    for (int64_t kb = k0; kb < k1; kb += S) {
        const int cnt = int((k1 - kb < S) ? (k1 - kb) : S);
        const int64_t jb = m.kidx[kb];
        const bool run = (m.kidx[kb + cnt - 1] - jb == cnt - 1);  // consecutive columns
        // a lane's stored values of source s: into the tile, or straight to its row
        auto put = [&](int s, const double (&v)[RPE * VPS]) {
            if (run) {
#pragma unroll
                for (int a = 0; a < RPE; a++)
#pragma unroll
                    for (int b = 0; b < VPS; b++) tile[TL::at(RPE * lane + a, VPS * s + b)] = OUT(v[VPS * a + b]);
            } else if (live) {
                OUT* o = row + VPS * m.kidx[kb + s];
#pragma unroll
                for (int a = 0; a < RPE; a++)
#pragma unroll
                    for (int b = 0; b < VPS; b++) store_out(o + a * ld + b, v[VPS * a + b]);
            }
        };
        // the block q of source s (element j): row transform, self block, storage
        auto finish = [&](int s, int64_t j, double (&q)[9]) {
            if (ROWT) {
                double t[9];
                for (int a = 0; a < 3; a++)
                    for (int b = 0; b < 3; b++)
                        t[3 * a + b] = rt[3 * a] * q[b] + rt[3 * a + 1] * q[3 + b] + rt[3 * a + 2] * q[6 + b];
                for (int k = 0; k < 9; k++) q[k] = t[k];
            }
            if (live && j == i) {
                for (int k = 0; k < 9; k++) {
                    qdiag[9 * i + k] = q[k];
                    q[k] = 0.0;
                }
            }
            // stored values: the 3x3 block row by row, or the planes
            double v[RPE * VPS];
            if constexpr (PK == 0) {
#pragma unroll
                for (int k = 0; k < 9; k++) v[k] = q[k];
            } else {
                if (PK == 5) traced |= fabs(q[0] + q[4] + q[8]) > 0.25;
                v[0] = q[0];
                v[1] = 0.5 * (q[1] + q[3]);
                v[2] = 0.5 * (q[2] + q[6]);
                v[3] = q[4];
                v[4] = 0.5 * (q[5] + q[7]);
                if constexpr (PK == 6) v[5] = q[8];
            }
            put(s, v);
        };
        if constexpr (kFar && SYM) {
            // tetrahedra with transform copies: copy by copy, far or not
#pragma unroll 1
            for (int c = 0; c < cnt; c += CH) {
                chunk(kb + c);
#pragma unroll 1
                for (int t = 0; t < CH / 4; t++) {
                    const int f = wave * (CH / 4) + t, s = c + f;
                    if (s >= cnt) break;
                    const int64_t j = m.kidx[kb + s];
                    double q[9];
#pragma unroll
                    for (int k = 0; k < 9; k++) q[k] = 0.0;
#pragma unroll 1
                    for (int64_t cc = m.copy_off[j]; cc < m.copy_off[j + 1]; cc++) {
                        const double* cp = m.copies + 24 * cc;
                        double xl[3], g[5];
                        apply_inv(cp, x, xl);
                        double zz = 0.0;
                        if (!far_tet_eval<FAR32>(fsrc + kFarTet * f, xl, g))
                            zz = near_tet_eval<FAR32>(fsrc + kFarTet * f, xl, g) ? -1.0 : 0.0;
                        zz -= g[0] + g[3];
                        const double l[9] = {g[0], g[1], g[2], g[1], g[3], g[4], g[2], g[4], zz};
                        const double* F = cp + 12;
#pragma unroll
                        for (int a = 0; a < 3; a++)
#pragma unroll
                            for (int b = 0; b < 3; b++)
                                q[3 * a + b] += F[3 * a] * l[b] + F[3 * a + 1] * l[3 + b] + F[3 * a + 2] * l[6 + b];
                    }
                    finish(s, j, q);
                }
            }
        } else if constexpr (kFar) {
            // stores a tetrahedron's block: xx, xy, xz, yy, yz and zz
            auto put6 = [&](int s, const double (&q)[5], double zz) {
                double v[RPE * VPS];
                if constexpr (PK == 0) {
                    v[0] = q[0];
                    v[1] = v[3] = q[1];
                    v[2] = v[6] = q[2];
                    v[4] = q[3];
                    v[5] = v[7] = q[4];
                    v[8] = zz;
                } else {
#pragma unroll
                    for (int k = 0; k < 5; k++) v[k] = q[k];
                    if constexpr (PK == 6) v[5] = zz;
                }
                put(s, v);
            };
#pragma unroll 1
            for (int c = 0; c < cnt; c += CH) {
                chunk(kb + c);
                // far sources first; the others' bits are set and they follow
                // after the loop, where the far form's registers are free
                uint32_t near = 0;
#pragma unroll 1
                for (int t = 0; t < CH / 4; t++) {
                    const int f = wave * (CH / 4) + t, s = c + f;
                    if (s >= cnt) break;
                    double q[5];
                    if (far_tet_eval<FAR32>(fsrc + kFarTet * f, x, q))
                        put6(s, q, -(q[0] + q[3]));
                    else
                        near |= 1u << f;
                }
#pragma unroll 1
                for (; near; near &= near - 1) {
                    const int f = __builtin_ctz(near), s = c + f;
                    double q[5];
                    const bool in = near_tet_eval<FAR32>(fsrc + kFarTet * f, x, q);
                    double zz = -(q[0] + q[3]) - (in ? 1.0 : 0.0);
                    if (live && m.kidx[kb + s] == i) {
                        const double d[9] = {q[0], q[1], q[2], q[1], q[3], q[4], q[2], q[4], zz};
                        for (int k = 0; k < 9; k++) qdiag[9 * i + k] = d[k];
                        for (int k = 0; k < 5; k++) q[k] = 0.0;
                        zz = 0.0;
                    } else if (PK == 5) {
                        traced |= in;
                    }
                    put6(s, q, zz);
                }
            }
        } else {
#pragma unroll 1
            for (int s = wave * (S / 4); s < (wave + 1) * (S / 4) && s < cnt; s++) {
                const int64_t j = m.kidx[kb + s];
                double q[9];
                if constexpr (FAR32)
                    block_Q_mixed<SYM, KIND>(mv, j, x, q);
                else
                    block_Q<R, SYM, KIND>(mv, j, x, q);
                finish(s, j, q);
            }
        }
        if (run) {
            __syncthreads();
            OUT* base = Q + (RPE * (i0 - r0)) * ld + VPS * jb;
            constexpr int U = TL::U, RP = 256 / U;  // rows per pass
            constexpr int TR = RPE * 64;             // stored rows of a full tile
            if (cnt == S && nrow == 64 && ((VPS * jb * int64_t(sizeof(OUT))) & 7) == 0) {
                // full tile: 8-byte units, RP rows of U units per pass, offsets
                // in 32 bits from a uniform base (the tile spans < 2^32 bytes)
                const int lr = threadIdx.x / U, lc = threadIdx.x - U * lr;
                if (lr < RP) {
                    constexpr int WU = W / TL::EPU;
                    const uint64_t* src = reinterpret_cast<const uint64_t*>(tile);
                    // unit lc of tile row r
                    auto unit = [&](int r) { return src[r * WU + (lc ^ ((r / RPE) & TL::SWZ))]; };
                    char* dst = reinterpret_cast<char*>(base);  // uniform, advanced per pass
                    const int64_t step = int64_t(RP) * ld * int64_t(sizeof(OUT));
                    const uint32_t off = uint32_t(lr) * uint32_t(ld * sizeof(OUT)) + uint32_t(8 * lc);
                    constexpr int full = TR / RP;  // passes with every thread's row in the tile
                    constexpr int G = full % 5 == 0 ? 5 : (full % 4 == 0 ? 4 : 3);  // reads in flight
#pragma unroll 1
                    for (int it = 0; it < full / G * G; it += G) {
                        uint64_t u[G];
#pragma unroll
                        for (int k = 0; k < G; k++) u[k] = unit(lr + RP * (it + k));
#pragma unroll
                        for (int k = 0; k < G; k++) {
                            *reinterpret_cast<uint64_t*>(dst + off) = u[k];
                            dst += step;
                        }
                    }
#pragma unroll
                    for (int it = full / G * G; it < full; it++) {
                        *reinterpret_cast<uint64_t*>(dst + off) = unit(lr + RP * it);
                        dst += step;
                    }
                    if (RP * full + lr < TR) *reinterpret_cast<uint64_t*>(dst + off) = unit(lr + RP * full);
                }
            } else {
                // partial tile: the RPE*nrow stored rows, VPS*cnt values each
                const int cols = VPS * cnt, total = RPE * nrow * cols;
                const int step_r = 256 / cols, step_c = 256 - step_r * cols;
                int r = threadIdx.x / cols, c = threadIdx.x - r * cols;
                for (int e = threadIdx.x; e < total; e += 256) {
                    base[int64_t(r) * ld + c] = tile[TL::at(r, c)];
                    c += step_c;
                    r += step_r;
                    if (c >= cols) {
                        c -= cols;
                        r++;
                    }
                }
            }
            __syncthreads();
        }
    }
    if (PK == 5 && live && traced) *flag = 1;
}

template <bool SYM, bool ROWT, class OUT, int PK = 0>
hipError_t asm_dispatch(const DevModel& m, OUT* Q, int64_t ld, double* qdiag, int64_t r0, int64_t r1,
                        hipStream_t s, bool far32, int32_t* flag)
{
    if (r1 <= r0) return hipSuccess;
    const int64_t gx = (r1 - r0 + 63) / 64;
    for (int slot = 0; slot < 3; slot++) {
        const int64_t cnt = m.koff[slot + 1] - m.koff[slot];
        if (cnt == 0) continue;
        // enough workgroups to fill 256 CUs several times over; column tiles
        // are whole LDS tiles
        constexpr int S = AsmTile<OUT, PK>::S;
        const int64_t gy_target = std::max<int64_t>(1, (4096 + gx - 1) / gx);
        int64_t jt = std::max<int64_t>(4, (cnt + gy_target - 1) / gy_target);
        jt = std::min<int64_t>((jt + S - 1) / S * S, 256);
        const dim3 grid{unsigned(gx), unsigned((cnt + jt - 1) / jt), 1u};
        // FP32 storage: far blocks in FP32 arithmetic (general polyhedra stay FP64)
        constexpr bool mixed = sizeof(OUT) == 4;
        if (slot == 0 && mixed && far32)
            hipLaunchKernelGGL((k_assemble<double, SYM, ROWT, OUT, 0, mixed, PK>), grid, dim3(256), 0, s, m, Q, ld, qdiag, jt, r0, r1, flag);
        else if (slot == 0)
            hipLaunchKernelGGL((k_assemble<double, SYM, ROWT, OUT, 0, false, PK>), grid, dim3(256), 0, s, m, Q, ld, qdiag, jt, r0, r1, flag);
        else if (slot == 1 && mixed && far32)
            hipLaunchKernelGGL((k_assemble<double, SYM, ROWT, OUT, 1, mixed, PK>), grid, dim3(256), 0, s, m, Q, ld, qdiag, jt, r0, r1, flag);
        else if (slot == 1)
            hipLaunchKernelGGL((k_assemble<double, SYM, ROWT, OUT, 1, false, PK>), grid, dim3(256), 0, s, m, Q, ld, qdiag, jt, r0, r1, flag);
        else
            hipLaunchKernelGGL((k_assemble<double, SYM, ROWT, OUT, 2, false, PK>), grid, dim3(256), 0, s, m, Q, ld, qdiag, jt, r0, r1, flag);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ---------------------------------------------------------------- field
// Sums the elements kidx[koff[KIND] + y*js ...] of one kind slot; slice
// `slice0 + blockIdx.y` of the partial buffer (or B/H directly).
// The FP32 sweep runs as two launches over the same grid: kPassFar (FP32,
// the elements no lane of the wave is near) stores the sums, kPassNear (FP64,
// the others) adds to them.
template <int PASS>
__device__ __forceinline__ void field_store(double* __restrict__ o, const double b[3], const double h[3])
{
    for (int k = 0; k < 3; k++) {
        if (PASS == kPassNear) {
            o[k] += b[k];
            o[3 + k] += h[k];
        } else {
            o[k] = b[k];
            o[3 + k] = h[k];
        }
    }
}
template <int PASS>
__device__ __forceinline__ void field_store(double* __restrict__ B, double* __restrict__ H, int64_t p,
                                            const double b[3], const double h[3])
{
    for (int k = 0; k < 3; k++) {
        if (B) B[3 * p + k] = (PASS == kPassNear) ? B[3 * p + k] + b[k] : b[k];
        if (H) H[3 * p + k] = (PASS == kPassNear) ? H[3 * p + k] + h[k] : h[k];
    }
}

// Blocks without transform copies: the workgroup copies kRecTile records and
// magnetizations to LDS first.  Read from memory they are a chain of three
// scalar loads (list, offset, record) per element, which two waves a SIMD do
// not hide: a host call of 10,000 points on 512 blocks 167 us by that chain,
// 163 from LDS.  More waves a SIMD (3 or 4, the near form spilling) 171 and 184.
constexpr int kRecTile = 64;
constexpr int kRecStage = 6 + 3;
// General polyhedra (FP64): hexahedron records and magnetizations likewise.
// 2,048 points and 1,000 hexahedra 329 us by eval_gen, 134 now.
constexpr int kHexTile = 16;
constexpr int kHexStage = kHex + 3;

template <class R, bool SYM, int KIND, int PASS>
__global__ __launch_bounds__(256) void k_field(DevModel m, const double* __restrict__ M,
                                               const double* __restrict__ pts, int64_t np,
                                               int64_t js, int64_t slice0, double* __restrict__ B,
                                               double* __restrict__ H, double* __restrict__ part)
{
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const bool live = p < np;
    const int64_t kend = m.koff[KIND + 1];
    const int64_t k0 = m.koff[KIND] + int64_t(blockIdx.y) * js;
    const int64_t k1 = (k0 + js < kend) ? (k0 + js) : kend;
    double x[3] = {0, 0, 0};
    if (live) {
        x[0] = pts[3 * p];
        x[1] = pts[3 * p + 1];
        x[2] = pts[3 * p + 2];
    }
    double b[3] = {0, 0, 0}, h[3] = {0, 0, 0};
    if constexpr (KIND == 0 && !SYM) {
        __shared__ double tile[kRecTile * kRecStage];
        for (int64_t base = k0; base < k1; base += kRecTile) {
            const int cnt = int((k1 - base < kRecTile) ? (k1 - base) : kRecTile);
            __syncthreads();  // the previous tile has been consumed
            if (int(threadIdx.x) < cnt) {
                const int64_t j = m.kidx[base + threadIdx.x];
                const double* rec = m.data + m.off[j];
                double* o = tile + kRecStage * threadIdx.x;
                for (int k = 0; k < 6; k++) o[k] = rec[k];
                for (int k = 0; k < 3; k++) o[6 + k] = M[3 * j + k];
            }
            __syncthreads();
            if (!live) continue;
#pragma unroll 1
            for (int q = 0; q < cnt; q++) {
                const double* rec = tile + kRecStage * q;
                const double mm[3] = {rec[6], rec[7], rec[8]};
                double hl[3];
                bool in;
                if (!elem_H<R, KIND, PASS>(EK_REC, rec, nullptr, mm, x, hl, in)) continue;
                for (int k = 0; k < 3; k++) {
                    h[k] += hl[k];
                    b[k] += hl[k] + (in ? mm[k] : 0.0);
                }
            }
        }
        if (!live) return;
    } else if constexpr (KIND == 2 && PASS == kPassAll) {
        static_assert(sizeof(R) == 8, "the single-precision sweep is two passes");
        __shared__ double tile[kHexTile * kHexStage];
        __shared__ int32_t elem[kHexTile], at[kHexTile];
        for (int64_t base = k0; base < k1; base += kHexTile) {
            const int cnt = int((k1 - base < kHexTile) ? (k1 - base) : kHexTile);
            __syncthreads();  // the previous tile has been consumed
            if (int(threadIdx.x) < cnt) {
                const int32_t j = m.kidx[base + threadIdx.x];
                elem[threadIdx.x] = j;
                at[threadIdx.x] = m.hex_at[j];
                for (int k = 0; k < 3; k++) tile[kHexStage * threadIdx.x + kHex + k] = M[3 * int64_t(j) + k];
            }
            __syncthreads();
            for (int i = threadIdx.x; i < cnt * kHex; i += 256) {
                const int q = i / kHex, k = i - kHex * q;
                if (at[q] >= 0) tile[kHexStage * q + k] = m.hex[int64_t(kHex) * at[q] + k];
            }
            __syncthreads();
            if (!live) continue;
#pragma unroll 1
            for (int q = 0; q < cnt; q++) {
                const double* rec = tile + kHexStage * q;
                const double mm[3] = {rec[kHex], rec[kHex + 1], rec[kHex + 2]};
                const int64_t j = __builtin_amdgcn_readfirstlane(elem[q]);
                const double* er = m.data + m.off[j];
                auto H_at = [&](const double* xl, double* hl) {
                    double q6[6];
                    const bool in = gen_block(at[q] >= 0 ? rec : nullptr, er, xl, q6);
                    hl[0] = q6[0] * mm[0] + q6[3] * mm[1] + q6[4] * mm[2];
                    hl[1] = q6[3] * mm[0] + q6[1] * mm[1] + q6[5] * mm[2];
                    hl[2] = q6[4] * mm[0] + q6[5] * mm[1] + q6[2] * mm[2];
                    return in;
                };
                double hl[3];
                if (!SYM) {
                    const bool in = H_at(x, hl);
                    for (int k = 0; k < 3; k++) {
                        h[k] += hl[k];
                        b[k] += hl[k] + (in ? mm[k] : 0.0);
                    }
                    continue;
                }
                for (int64_t c = m.copy_off[j]; c < m.copy_off[j + 1]; c++) {
                    const double* cp = m.copies + 24 * c;
                    double xl[3], hg[3], bg[3];
                    apply_inv(cp, x, xl);
                    const bool in = H_at(xl, hl);
                    const double bl[3] = {hl[0] + (in ? mm[0] : 0.0), hl[1] + (in ? mm[1] : 0.0),
                                          hl[2] + (in ? mm[2] : 0.0)};
                    mat3_vec(cp + 12, hl, hg);
                    mat3_vec(cp + 12, bl, bg);
                    for (int k = 0; k < 3; k++) {
                        h[k] += hg[k];
                        b[k] += bg[k];
                    }
                }
            }
        }
        if (!live) return;
    } else {
        if (!live) return;
        field_add<R, SYM, KIND, PASS>(view(m), M, m.kidx, k0, k1, x, b, h);
    }
    if (part)
        field_store<PASS>(part + ((slice0 + int64_t(blockIdx.y)) * np + p) * 6, b, h);
    else
        field_store<PASS>(B, H, p, b, h);
}

// Tetrahedron field sweep over charged records staged in LDS: the workgroup
// copies kTetTile records (86 doubles each) with coalesced 16-byte loads, and
// every lane then reads them at wave-uniform LDS addresses (broadcast, no bank
// conflicts) while it evaluates its own point.  Staging keeps the record out of
// scalar registers, whose pressure otherwise spills through VGPR lanes.
constexpr int kTetTile = 32;
// occupancy floor for the tetrahedron sweep (waves per SIMD): bounds
// the VGPRs the scheduler may use for hoisted LDS reads
#ifndef RH_TET_WAVES
#define RH_TET_WAVES 3
#endif
// mesh sweep with N points per lane: occupancy floor (waves per SIMD).  Two
// points share a record's LDS reads, branches and votes and give each other
// independent instructions; on the C-yoke (FP64, 1M points) two points at 3
// waves (155 VGPRs, no spill) take 35.7 ms and at 4 waves 0.2 ms more, one point
// at 4 to 6 waves 40-47 ms; FP32 on the Halbach ring (250,007 points) two
// points 37.5 ms at 4 waves and 39.7 at 3, one point 39.4 ms at 5.
#ifndef RH_MESH_WAVES32
#define RH_MESH_WAVES32 4
#endif
#ifndef RH_MESH_WAVES
#define RH_MESH_WAVES 3
#endif
template <class R, int N>
constexpr int mesh_waves() { return N == 1 ? 4 : (sizeof(R) == 4 ? RH_MESH_WAVES32 : RH_MESH_WAVES); }
// records per LDS tile (at most 64: one bit of a mask each; even, for the
// pairwise unrolled loops)
constexpr int kMeshStage = 64;

template <class R, bool SYM, int PASS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RH_TET_WAVES))) void k_field_tet(DevModel m, const double* __restrict__ pts,
                                                   int64_t np, int64_t js, int64_t slice0,
                                                   double* __restrict__ B, double* __restrict__ H,
                                                   double* __restrict__ part)
{
    __shared__ __align__(16) double tile[kTetTile * kChargedTet];
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const bool live = p < np;
    const int64_t ntet = m.koff[2] - m.koff[1];
    const int64_t t0 = int64_t(blockIdx.y) * js;
    const int64_t t1 = (t0 + js < ntet) ? (t0 + js) : ntet;
    double x[3] = {0.0, 0.0, 0.0};
    if (live) {
        x[0] = pts[3 * p];
        x[1] = pts[3 * p + 1];
        x[2] = pts[3 * p + 2];
    }
    double b[3] = {0, 0, 0}, h[3] = {0, 0, 0};
    for (int64_t base = t0; base < t1; base += kTetTile) {
        const int cnt = int((t1 - base < kTetTile) ? (t1 - base) : kTetTile);
        const double2* src = reinterpret_cast<const double2*>(m.charged + kChargedTet * base);
        double2* dst = reinterpret_cast<double2*>(tile);
        __syncthreads();  // the previous tile has been consumed
        for (int i = threadIdx.x; i < cnt * (kChargedTet / 2); i += 256) dst[i] = src[i];
        __syncthreads();
        if (!live) continue;
#pragma unroll 1
        for (int q = 0; q < cnt; q++) {
            const double* rec = tile + kChargedTet * q;
            const double mm[3] = {rec[kChargedM], rec[kChargedM + 1], rec[kChargedM + 2]};
            if (!SYM) {
                double hl[3];
                if (PASS != kPassAll && tet_near32(rec, x) != (PASS == kPassNear)) continue;
                const bool in = field_tet<R>(rec, x, hl);
                for (int k = 0; k < 3; k++) {
                    h[k] += hl[k];
                    b[k] += hl[k] + (in ? mm[k] : 0.0);
                }
                continue;
            }
            const int64_t j = m.kidx[m.koff[1] + base + q];
            for (int64_t c = m.copy_off[j]; c < m.copy_off[j + 1]; c++) {
                const double* cp = m.copies + 24 * c;
                double xl[3], hl[3], hg[3], bg[3];
                apply_inv(cp, x, xl);
                if (PASS != kPassAll && tet_near32(rec, xl) != (PASS == kPassNear)) continue;
                const bool in = field_tet<R>(rec, xl, hl);
                const double bl[3] = {hl[0] + (in ? mm[0] : 0.0), hl[1] + (in ? mm[1] : 0.0),
                                      hl[2] + (in ? mm[2] : 0.0)};
                mat3_vec(cp + 12, hl, hg);
                mat3_vec(cp + 12, bl, bg);
                for (int k = 0; k < 3; k++) {
                    h[k] += hg[k];
                    b[k] += bg[k];
                }
            }
        }
    }
    if (!live) return;
    if (part)
        field_store<PASS>(part + ((slice0 + int64_t(blockIdx.y)) * np + p) * 6, b, h);
    else
        field_store<PASS>(B, H, p, b, h);
}

// ---------------------------------------------------------------- mesh form
// Charged records of the mesh form for magnetization M (one lane per entity).
__global__ __launch_bounds__(256) void k_mesh_charge_edges(MeshDev md, const double* __restrict__ M, bool pack32)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= md.ne) return;
    double w[3] = {0.0, 0.0, 0.0};
    for (int64_t k = md.edge_inc_off[i]; k < md.edge_inc_off[i + 1]; k++) {
        const int64_t j = md.edge_inc_elem[k];
        const double* W = md.edge_inc_w + 9 * k;  // F_c W_e, row-major
        const double m0 = M[3 * j], m1 = M[3 * j + 1], m2 = M[3 * j + 2];
        w[0] += W[0] * m0 + W[1] * m1 + W[2] * m2;
        w[1] += W[3] * m0 + W[4] * m1 + W[5] * m2;
        w[2] += W[6] * m0 + W[7] * m1 + W[8] * m2;
    }
    mesh_charge_edge(md.edge_geo + kMeshEdgeGeo * i, w, pack32, md.ch_edge + kMeshEdge * i);
}

__global__ __launch_bounds__(256) void k_mesh_charge_faces(MeshDev md, const double* __restrict__ M, bool pack32)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= md.nf) return;
    const double* g = md.face_geo + kMeshFaceGeo * i;
    double s = 0.0;
    for (int64_t k = md.face_inc_off[i]; k < md.face_inc_off[i + 1]; k++) {
        const int64_t j = md.face_inc_elem[k];
        const double* v = md.face_inc_v + 3 * k;
        s += v[0] * M[3 * j] + v[1] * M[3 * j + 1] + v[2] * M[3 * j + 2];
    }
    // owned edges were charged before, on the same stream
    mesh_charge_face(g, s, md.face_edge + 3 * i, md.edge_geo, md.ch_edge, pack32, md.ch_face + kMeshFace * i);
}

__global__ __launch_bounds__(256) void k_mesh_charge_in(MeshDev md, const double* __restrict__ M)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= md.ni) return;
    const int64_t j = md.in_elem[i];
    const double* g = md.in_geo + (1 + 4 * kMeshPlanes) * i;
    double* o = md.ch_in + kMeshIn * i;
    const double* F = md.in_F + 9 * i;  // the copy's field transform
    const double m0 = M[3 * j], m1 = M[3 * j + 1], m2 = M[3 * j + 2];
    o[0] = g[0];
    o[1] = F[0] * m0 + F[1] * m1 + F[2] * m2;
    o[2] = F[3] * m0 + F[4] * m1 + F[5] * m2;
    o[3] = F[6] * m0 + F[7] * m1 + F[8] * m2;
    for (int k = 0; k < 4 * kMeshPlanes; k++) o[4 + k] = g[1 + k];
}

// Field sweep of the mesh form: slice blockIdx.y of the unique edges no face
// owns, the unique faces and the inside tiles.  Every lane evaluates the same
// record for its own N points; records are staged through LDS in tiles of
// kMeshStage and read there at wave-uniform addresses (broadcast), their
// branch flags through the scalar cache.
//
// Bound by FP64 vector issue: 119 instructions per wave of points and
// tetrahedron on the C-yoke (185 with logarithm-ratio edges, dot products and
// one point per lane), 80 % of the issue slots.  1M points: 35.7 ms against
// 49.3; FP32 on the 20,000-element ring, 250,007 points: 35.4 ms against 45.8.
// Reading the records through the scalar cache instead of LDS freed the vector
// registers but left each wave waiting on scalar loads: 52 ms.
//
// FP32: the records of a chunk that the wave is near (mesh32_near) are marked
// in `defer` and evaluated in FP64 after the chunk's loop, where the loop's
// carried values are dead, so the FP64 code does not add to the loop's
// registers.
template <class R, int N>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(mesh_waves<R, N>()))) void
k_field_mesh(DevModel m, const double* __restrict__ pts, int64_t np, int64_t S, int64_t slice0,
             double* __restrict__ B, double* __restrict__ H, double* __restrict__ part)
{
    constexpr bool f32 = sizeof(R) == 4;
    using Vtx = MeshVtxN<R, N>;
    __shared__ __align__(16) double tile[kMeshStage * kMeshFace];
    const MeshDev& md = m.mesh;
    // a wave's 64 N points are consecutive
    const int64_t p = int64_t(blockIdx.x) * (256 * N) + (threadIdx.x >> 6) * (64 * N) + (threadIdx.x & 63);
    const bool live = p < np;
    const int64_t y = blockIdx.y;
    double x[N][3];
#pragma unroll
    for (int i = 0; i < N; i++) {
        // a point past the end repeats the lane's first one, unstored
        const int64_t q = (p + 64 * i < np) ? p + 64 * i : p;
        for (int k = 0; k < 3; k++) x[i][k] = live ? pts[3 * q + k] : 0.0;
    }
    // records [base, base + cnt) of `size` doubles each into the tile
    auto stage = [&](const double* __restrict__ rec, int cnt, int size) {
        const double2* src = reinterpret_cast<const double2*>(rec);
        double2* dst = reinterpret_cast<double2*>(tile);
        __syncthreads();  // the previous tile has been consumed
        for (int i = threadIdx.x; i < cnt * (size / 2); i += 256) dst[i] = src[i];
        __syncthreads();
    };
    double h[N][3];
#pragma unroll
    for (int i = 0; i < N; i++) h[i][0] = h[i][1] = h[i][2] = 0.0;
    auto add = [&](const R (&v)[N], const double* __restrict__ w) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            h[i][0] += double(v[i]) * w[0];
            h[i][1] += double(v[i]) * w[1];
            h[i][2] += double(v[i]) * w[2];
        }
    };
    // FP32: whether a point of the wave is near the record with these vertices
    auto near32 = [&](const Vtx* const (&v)[4], int nv, float thr) {
        float d = float(v[0]->d[0]);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int i = 0; i < N; i++)
                if (k < nv) d = fminf(d, float(v[k]->d[i]));
        return mesh32_near(d, thr);
    };
    // leading coefficients of the far tiers, kept in vector registers
    double a_top = kAtan32Top, e_top = kEdge6Top;
    if constexpr (!f32) asm("" : "+v"(a_top), "+v"(e_top));
    // an edge from its ends and the sum of their distances: + L_e w_e, e its
    // 2 len and w
    auto edge_term = [&](const Vtx& u, const Vtx& v, const R (&suv)[N], const double* __restrict__ e, R len2) {
        R L[N];
        edge_L2(u.r, u.d, v.r, v.d, suv, len2, e_top, L);
        add(L, e + 1);
    };
    // unique edges that no face owns, along paths: a continued edge takes its
    // first vertex's offset and distance from the previous edge.  The loop is
    // unrolled by two with the vertex slots P, Q swapping roles, so the
    // carried values stay in place (no register copies per edge).
    {
        Vtx P{}, Q{};
        const int64_t e0 = md.ne_free * y / S, e1 = md.ne_free * (y + 1) / S;
        const MeshFlags flags = mesh_flags(md.edge_flag);
        uint64_t defer = 0;
        auto edge = [&](int64_t g, int q, Vtx& a, Vtx& b) {
            const double* rec = tile + kMeshEdge * q;
            if (!(flags[g] & kMeshCont) || g == e0) mesh_vtx<R, N>(rec, x, a);
            mesh_vtx<R, N>(rec + 3, x, b);
            if constexpr (f32) {
                const float* f = reinterpret_cast<const float*>(rec + 6);
                const Vtx* const v[4] = {&a, &b, &b, &b};
                if (near32(v, 2, f[1])) {
                    defer |= uint64_t(1) << q;
                    return;
                }
                R s[N];
                mesh_sum<R, N>(a, b, s);
                edge_term(a, b, s, rec + 9, f[0]);
            } else {
                R s[N];
                mesh_sum<R, N>(a, b, s);
                edge_term(a, b, s, rec + 9, rec[9]);
            }
        };
        for (int64_t base = e0; base < e1; base += kMeshStage) {
            const int cnt = int((e1 - base < kMeshStage) ? (e1 - base) : kMeshStage);
            stage(md.ch_edge + kMeshEdge * base, cnt, kMeshEdge);
            if (!live) continue;
            int q = 0;
#pragma unroll 1
            for (; q + 2 <= cnt; q += 2) {
                edge(base + q, q, P, Q);
                edge(base + q + 1, q + 1, Q, P);
            }
            if (q < cnt) edge(base + q, q, P, Q);  // the last edge of the slice
            if constexpr (f32) {
                for (; defer; defer &= defer - 1) {
                    const double* rec = tile + kMeshEdge * __builtin_ctzll(defer);
#pragma unroll
                    for (int i = 0; i < N; i++) {
                        const double L = mesh_edge_L_near(rec, x[i]);
                        for (int k = 0; k < 3; k++) h[i][k] += L * rec[10 + k];
                    }
                }
            }
        }
    }
    // unique faces: - Omega_f g_f, triangles along strips: a continued
    // triangle takes its first two vertices (and the sum of their distances)
    // from the previous one.  Unrolled by three with the slots A, B, C
    // rotating.  A triangle also evaluates the edges it owns from the offsets
    // and distances of its vertices.
    {
        // this slice's faces: triangles [f0, ft), then quadrilaterals [fq, f1)
        const int64_t f0 = md.nf * y / S, f1 = md.nf * (y + 1) / S;
        const int64_t ft = f1 < md.nf_tri ? f1 : md.nf_tri, fq = f0 > md.nf_tri ? f0 : md.nf_tri;
        const MeshFlags flags = mesh_flags(md.face_flag);
        uint64_t defer = 0;
        // FP64 for the records of the tile from `base` that the wave is near
        auto deferred = [&](int64_t base) {
            if constexpr (f32) {
                for (; defer; defer &= defer - 1) {
                    const int q = __builtin_ctzll(defer);
                    const double* rec = tile + kMeshFace * q;
                    const int flag = flags[base + q];
#pragma unroll
                    for (int i = 0; i < N; i++) {
                        const MeshFace64 f = mesh_face_near(rec, flag, x[i]);
                        h[i][0] += f.h0 + f.om * rec[18];
                        h[i][1] += f.h1 + f.om * rec[19];
                        h[i][2] += f.h2 + f.om * rec[20];
                    }
                }
            }
        };
        auto owned = [&](const Vtx& u, const Vtx& v, const R (&suv)[N], const double* __restrict__ e) {
            edge_term(u, v, suv, e, R(e[0]));
        };
        {
            Vtx A{}, Bv{}, C{};
            R sAB[N] = {}, sBC[N] = {}, sCA[N] = {};
            auto tri = [&](int64_t g, int q, Vtx& a, Vtx& b, Vtx& c, R (&sab)[N], R (&sbc)[N]) {
                const double* rec = tile + kMeshFace * q;
                const int flag = flags[g];
                if (!(flag & kMeshCont) || g == f0) {
                    mesh_vtx<R, N>(rec, x, a);
                    mesh_vtx<R, N>(rec + 3, x, b);
                    mesh_sum<R, N>(a, b, sab);
                }
                mesh_vtx<R, N>(rec + 6, x, c);
                mesh_sum<R, N>(b, c, sbc);
                if constexpr (f32) {
                    // a near record only sets its bit; the carried values
                    // (b, c, sbc) are in place either way
                    const Vtx* const v[4] = {&a, &b, &c, &c};
                    if (near32(v, 3, reinterpret_cast<const float*>(rec + kMeshFaceEdges + 13)[0])) {
                        defer |= uint64_t(1) << q;
                        return;
                    }
                }
                R sca[N], om[N];
                mesh_sum<R, N>(c, a, sca);
                mesh_tri_half_omega<R, N>(a, b, c, sab, sbc, sca, rec, a_top, om);
                add(om, rec + 18);
                if (flag & 1) owned(a, b, sab, rec + kMeshFaceEdges);
                if (flag & 2) owned(b, c, sbc, rec + kMeshFaceEdges + 4);
                if (flag & 4) owned(c, a, sca, rec + kMeshFaceEdges + 8);
            };
            // tiles hold whole turns of the slots
            constexpr int kTri = kMeshStage / 3 * 3;
            for (int64_t base = f0; base < ft; base += kTri) {
                const int cnt = int((ft - base < kTri) ? (ft - base) : kTri);
                stage(md.ch_face + kMeshFace * base, cnt, kMeshFace);
                if (!live) continue;
                int q = 0;
#pragma unroll 1
                for (; q + 3 <= cnt; q += 3) {
                    tri(base + q, q, A, Bv, C, sAB, sBC);
                    tri(base + q + 1, q + 1, Bv, C, A, sBC, sCA);
                    tri(base + q + 2, q + 2, C, A, Bv, sCA, sAB);
                }
                // the last triangles of the slice
                if (q < cnt) tri(base + q, q, A, Bv, C, sAB, sBC);
                if (q + 1 < cnt) tri(base + q + 1, q + 1, Bv, C, A, sBC, sCA);
                deferred(base);
            }
        }
        {
            Vtx QA{}, QB{}, QC{}, QD{};
            R sQAB[N] = {}, sQCD[N] = {};
            // a quadrilateral with the sides (v0,v1), (v1,v2), (v2,v3) it
            // owns, along strips: a continued quadrilateral takes v0, v1 and
            // their sum from the previous one's v2, v3 (slots a, b, sab)
            auto quad = [&](int64_t g, int q, Vtx& a, Vtx& b, Vtx& c, Vtx& d, R (&sab)[N], R (&scd)[N]) {
                const double* rec = tile + kMeshFace * q;
                const int flag = flags[g];
                if (!(flag & kMeshCont) || g == fq) {
                    mesh_vtx<R, N>(rec, x, a);
                    mesh_vtx<R, N>(rec + 3, x, b);
                    mesh_sum<R, N>(a, b, sab);
                }
                mesh_vtx<R, N>(rec + 6, x, c);
                mesh_vtx<R, N>(rec + 9, x, d);
                mesh_sum<R, N>(c, d, scd);
                if constexpr (f32) {
                    const Vtx* const v[4] = {&a, &b, &c, &d};
                    if (near32(v, 4, reinterpret_cast<const float*>(rec + kMeshFaceEdges + 13)[0])) {
                        defer |= uint64_t(1) << q;
                        return;
                    }
                }
                R sbc[N], om[N];
                mesh_sum<R, N>(b, c, sbc);
                mesh_quad_half_omega<R, N>(a, b, c, d, sab, sbc, scd, rec, a_top, om);
                add(om, rec + 18);
                if (flag & 1) owned(a, b, sab, rec + kMeshFaceEdges);
                if (flag & 2) owned(b, c, sbc, rec + kMeshFaceEdges + 4);
                if (flag & 4) owned(c, d, scd, rec + kMeshFaceEdges + 8);
            };
            for (int64_t base = fq; base < f1; base += kMeshStage) {
                const int cnt = int((f1 - base < kMeshStage) ? (f1 - base) : kMeshStage);
                stage(md.ch_face + kMeshFace * base, cnt, kMeshFace);
                if (!live) continue;
                int q = 0;
#pragma unroll 1
                for (; q + 2 <= cnt; q += 2) {
                    quad(base + q, q, QA, QB, QC, QD, sQAB, sQCD);
                    quad(base + q + 1, q + 1, QC, QD, QA, QB, sQCD, sQAB);
                }
                if (q < cnt) quad(base + q, q, QA, QB, QC, QD, sQAB, sQCD);
                deferred(base);
            }
        }
    }
    if (!live) return;
    // inside tests: B gets the magnetization of the element holding the
    // point.  Tiles whose bounding box holds no point of the wave are skipped
    // (wave-uniform vote).
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int64_t pi = p + 64 * i;
        if (pi >= np) break;
        double min[3] = {0.0, 0.0, 0.0};
        const int64_t t0 = md.ntiles * y / S, t1 = md.ntiles * (y + 1) / S;
        for (int64_t t = t0; t < t1; t++) {
            const double* bx = md.tile_box + 6 * t;
            const bool near = x[i][0] >= bx[0] && x[i][1] >= bx[1] && x[i][2] >= bx[2] && x[i][0] <= bx[3] &&
                              x[i][1] <= bx[4] && x[i][2] <= bx[5];
            if (!rh_any(near)) continue;
            const int64_t base = t * kMeshTile;
            const int cnt = int((md.ni - base < kMeshTile) ? (md.ni - base) : kMeshTile);
            for (int q = 0; q < cnt; q++) {
                const double* rec = md.ch_in + kMeshIn * (base + q);
                if (near && mesh_inside(rec, x[i]))
                    for (int k = 0; k < 3; k++) min[k] += rec[1 + k];
            }
        }
        double* o = part ? part + ((slice0 + y) * np + pi) * 6 : nullptr;
        for (int k = 0; k < 3; k++) {
            const double hk = h[i][k] * kInv4Pi;
            if (o) {
                o[k] = hk + min[k];
                o[3 + k] = hk;
            } else {
                if (B) B[3 * pi + k] = hk + min[k];
                if (H) H[3 * pi + k] = hk;
            }
        }
    }
}

// Sums the `splits` partial rows of 6 np values (B and H of each point) in a
// fixed order: a workgroup owns 256/G columns, G threads take every G-th row
// of a column and the first adds their G sums.  With one thread per point a
// sweep of 64 points over 1,790 slices of the 8,000-tetrahedron yoke spent
// 0.5 ms here, in one thread's chain of additions; G by the number of rows.
template <int G>
__global__ __launch_bounds__(256) void k_field_reduce(int64_t np, int64_t splits,
                                                      const double* __restrict__ part,
                                                      double* __restrict__ B, double* __restrict__ H)
{
    constexpr int C = 256 / G;
    __shared__ double red[G > 1 ? 256 : 1];
    const int col = threadIdx.x % C, g = threadIdx.x / C;
    const int64_t c = int64_t(blockIdx.x) * C + col, w = 6 * np;
    double acc = 0.0;
    if (c < w) {
#pragma unroll 4
        for (int64_t s = g; s < splits; s += G) acc += part[s * w + c];
    }
    if constexpr (G > 1) {
        red[threadIdx.x] = acc;
        __syncthreads();
        if (g == 0) {
#pragma unroll
            for (int k = 1; k < G; k++) acc += red[k * C + col];
        }
    }
    if (g != 0 || c >= w) return;
    const int64_t p = c / 6;
    const int k = int(c - 6 * p);
    if (k < 3) {
        if (B) B[3 * p + k] = acc;
    } else {
        if (H) H[3 * p + k - 3] = acc;
    }
}

// ---------------------------------------------------------------- matrix pass
typedef float nf4 __attribute__((ext_vector_type(4)));
typedef double nd2 __attribute__((ext_vector_type(2)));
template <int RW>
__global__ __launch_bounds__(256) void k_matvec_f32(const float* __restrict__ Q, int64_t nrows,
                                                    int64_t ld, const double* __restrict__ x,
                                                    const double* __restrict__ add,
                                                    double* __restrict__ y,
                                                    const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const int lane = threadIdx.x & 63;
    const int64_t r0 = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * RW;
    if (r0 >= nrows) return;
    double acc[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) acc[r] = 0.0;
    const nf4* rows[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) {
        const int64_t rr = (r0 + r < nrows) ? (r0 + r) : r0;
        rows[r] = reinterpret_cast<const nf4*>(Q + rr * ld);
    }
    const int64_t nv = ld / 4;  // float4 per row (ld multiple of 256)
    const nd2* x2 = reinterpret_cast<const nd2*>(x);
    for (int64_t c = lane; c < nv; c += 64) {
        const nd2 xa = x2[2 * c], xb = x2[2 * c + 1];
#pragma unroll
        for (int r = 0; r < RW; r++) {
            const nf4 q = __builtin_nontemporal_load(rows[r] + c);
            acc[r] += double(q.x) * xa.x + double(q.y) * xa.y + double(q.z) * xb.x + double(q.w) * xb.y;
        }
    }
#pragma unroll
    for (int r = 0; r < RW; r++) {
        const double v = wave_sum(acc[r]);
        if (lane == 0 && r0 + r < nrows) y[r0 + r] = v + (add ? add[r0 + r] : 0.0);
    }
}

template <int RW>
__global__ __launch_bounds__(256) void k_matvec_f64(const double* __restrict__ Q, int64_t nrows,
                                                    int64_t ld, const double* __restrict__ x,
                                                    const double* __restrict__ add,
                                                    double* __restrict__ y,
                                                    const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const int lane = threadIdx.x & 63;
    const int64_t r0 = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * RW;
    if (r0 >= nrows) return;
    double acc[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) acc[r] = 0.0;
    const nd2* rows[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) {
        const int64_t rr = (r0 + r < nrows) ? (r0 + r) : r0;
        rows[r] = reinterpret_cast<const nd2*>(Q + rr * ld);
    }
    const int64_t nv = ld / 2;
    const nd2* x2 = reinterpret_cast<const nd2*>(x);
#ifdef RH_MV_UNROLL
#pragma unroll RH_MV_UNROLL
#endif
    for (int64_t c = lane; c < nv; c += 64) {
        const nd2 xa = x2[c];
#pragma unroll
        for (int r = 0; r < RW; r++) {
            const nd2 q = __builtin_nontemporal_load(rows[r] + c);
            acc[r] += q.x * xa.x + q.y * xa.y;
        }
    }
#pragma unroll
    for (int r = 0; r < RW; r++) {
        const double v = wave_sum(acc[r]);
        if (lane == 0 && r0 + r < nrows) y[r0 + r] = v + (add ? add[r0 + r] : 0.0);
    }
}

// Matrix pass over the symmetric-block layout: ER element rows per wave, their
// P planes (xx, xy, xz, yy, yz[, zz]) streamed with 16-byte non-temporal loads
// (two column elements per lane in FP64, four in FP32), the iterate read once
// per column chunk as the interleaved (x, y, z) triples of those columns and
// shared by the ER rows; FP64 accumulation.
// element rows per wave: on the 40,000-tetrahedron yoke (5 planes) 4 rows
// measured 9.57 ms FP64 / 4.87 ms FP32 per pass, 2 rows 9.75 / 5.04, 1 row
// 10.70 / 6.18 (the iterate's reads per matrix byte fall as 1/rows); a
// twofold unroll of the column loop gained nothing
#ifndef RH_MVS_ER
#define RH_MVS_ER 4
#endif
#ifndef RH_MVS_UNROLL
#define RH_MVS_UNROLL 1
#endif
template <int P, int ER>
__global__ __launch_bounds__(256) void k_matvec_sym_f64(const double* __restrict__ Q, int64_t nel,
                                                        int64_t ldp, const double* __restrict__ x,
                                                        const double* __restrict__ add,
                                                        double* __restrict__ y,
                                                        const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const int lane = threadIdx.x & 63;
    const int64_t i0 = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * ER;
    if (i0 >= nel) return;
    const nd2* pl[ER][P];
#pragma unroll
    for (int r = 0; r < ER; r++) {
        const int64_t i = (i0 + r < nel) ? (i0 + r) : i0;  // rows past the end repeat row i0, unstored
#pragma unroll
        for (int k = 0; k < P; k++) pl[r][k] = reinterpret_cast<const nd2*>(Q + (i * P + k) * ldp);
    }
    const nd2* x2 = reinterpret_cast<const nd2*>(x);
    double h[ER][3];
#pragma unroll
    for (int r = 0; r < ER; r++) h[r][0] = h[r][1] = h[r][2] = 0.0;
    const int64_t nv = ldp / 2;
#pragma unroll RH_MVS_UNROLL
    for (int64_t c = lane; c < nv; c += 64) {
        nd2 q[ER][P];
#pragma unroll
        for (int r = 0; r < ER; r++)
#pragma unroll
            for (int k = 0; k < P; k++) q[r][k] = __builtin_nontemporal_load(pl[r][k] + c);
        // columns 2c and 2c+1: (a.x, a.y, b.x) and (b.y, d.x, d.y)
        const nd2 a = x2[3 * c], b = x2[3 * c + 1], d = x2[3 * c + 2];
#pragma unroll
        for (int r = 0; r < ER; r++) {
            const nd2* v = q[r];
            const nd2 zz = (P == 6) ? v[P - 1] : -(v[0] + v[3]);
            h[r][0] += v[0].x * a.x + v[1].x * a.y + v[2].x * b.x + v[0].y * b.y + v[1].y * d.x + v[2].y * d.y;
            h[r][1] += v[1].x * a.x + v[3].x * a.y + v[4].x * b.x + v[1].y * b.y + v[3].y * d.x + v[4].y * d.y;
            h[r][2] += v[2].x * a.x + v[4].x * a.y + zz.x * b.x + v[2].y * b.y + v[4].y * d.x + zz.y * d.y;
        }
    }
#pragma unroll
    for (int r = 0; r < ER; r++) {
        const double hx = wave_sum(h[r][0]), hy = wave_sum(h[r][1]), hz = wave_sum(h[r][2]);
        const int64_t i = i0 + r;
        if (lane == 0 && i < nel) {
            y[3 * i] = hx + (add ? add[3 * i] : 0.0);
            y[3 * i + 1] = hy + (add ? add[3 * i + 1] : 0.0);
            y[3 * i + 2] = hz + (add ? add[3 * i + 2] : 0.0);
        }
    }
}

template <int P, int ER>
__global__ __launch_bounds__(256) void k_matvec_sym_f32(const float* __restrict__ Q, int64_t nel,
                                                        int64_t ldp, const double* __restrict__ x,
                                                        const double* __restrict__ add,
                                                        double* __restrict__ y,
                                                        const int32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const int lane = threadIdx.x & 63;
    const int64_t i0 = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * ER;
    if (i0 >= nel) return;
    const nf4* pl[ER][P];
#pragma unroll
    for (int r = 0; r < ER; r++) {
        const int64_t i = (i0 + r < nel) ? (i0 + r) : i0;  // rows past the end repeat row i0, unstored
#pragma unroll
        for (int k = 0; k < P; k++) pl[r][k] = reinterpret_cast<const nf4*>(Q + (i * P + k) * ldp);
    }
    const nd2* x2 = reinterpret_cast<const nd2*>(x);
    double h[ER][3];
#pragma unroll
    for (int r = 0; r < ER; r++) h[r][0] = h[r][1] = h[r][2] = 0.0;
    const int64_t nv = ldp / 4;
#pragma unroll RH_MVS_UNROLL
    for (int64_t c = lane; c < nv; c += 64) {
        nf4 q[ER][P];
#pragma unroll
        for (int r = 0; r < ER; r++)
#pragma unroll
            for (int k = 0; k < P; k++) q[r][k] = __builtin_nontemporal_load(pl[r][k] + c);
        // columns 4c .. 4c+3: twelve doubles of x
        nd2 m[6];
#pragma unroll
        for (int k = 0; k < 6; k++) m[k] = x2[6 * c + k];
        const double mv[12] = {m[0].x, m[0].y, m[1].x, m[1].y, m[2].x, m[2].y,
                               m[3].x, m[3].y, m[4].x, m[4].y, m[5].x, m[5].y};
#pragma unroll
        for (int r = 0; r < ER; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const double xx = q[r][0][e], xy = q[r][1][e], xz = q[r][2][e], yy = q[r][3][e],
                             yz = q[r][4][e];
                const double zz = (P == 6) ? double(q[r][P - 1][e]) : -(xx + yy);
                const double mx = mv[3 * e], my = mv[3 * e + 1], mz = mv[3 * e + 2];
                h[r][0] += xx * mx + xy * my + xz * mz;
                h[r][1] += xy * mx + yy * my + yz * mz;
                h[r][2] += xz * mx + yz * my + zz * mz;
            }
    }
#pragma unroll
    for (int r = 0; r < ER; r++) {
        const double hx = wave_sum(h[r][0]), hy = wave_sum(h[r][1]), hz = wave_sum(h[r][2]);
        const int64_t i = i0 + r;
        if (lane == 0 && i < nel) {
            y[3 * i] = hx + (add ? add[3 * i] : 0.0);
            y[3 * i + 1] = hy + (add ? add[3 * i + 1] : 0.0);
            y[3 * i + 2] = hz + (add ? add[3 * i + 2] : 0.0);
        }
    }
}

// ---------------------------------------------------------------- relaxation update
__device__ __forceinline__ void inv3d(const double* m, double* o)
{
    const double c0 = m[4] * m[8] - m[5] * m[7], c1 = m[2] * m[7] - m[1] * m[8],
                 c2 = m[1] * m[5] - m[2] * m[4];
    const double c3 = m[5] * m[6] - m[3] * m[8], c4 = m[0] * m[8] - m[2] * m[6],
                 c5 = m[2] * m[3] - m[0] * m[5];
    const double c6 = m[3] * m[7] - m[4] * m[6], c7 = m[1] * m[6] - m[0] * m[7],
                 c8 = m[0] * m[4] - m[1] * m[3];
    const double inv = 1.0 / (m[0] * c0 + m[1] * c3 + m[2] * c6);
    o[0] = c0 * inv; o[1] = c1 * inv; o[2] = c2 * inv;
    o[3] = c3 * inv; o[4] = c4 * inv; o[5] = c5 * inv;
    o[6] = c6 * inv; o[7] = c7 * inv; o[8] = c8 * inv;
}

// H = (I - A)^{-1} b with A = chi_s * Q (iso) or Q * K (aniso).
__device__ __forceinline__ void solve_IminusA(const double* A, const double* b, double* H)
{
    double m[9];
    for (int k = 0; k < 9; k++) m[k] = -A[k];
    m[0] += 1.0; m[4] += 1.0; m[8] += 1.0;
    double inv[9];
    inv3d(m, inv);
    mat3_vec(inv, b, H);
}

// e^x - 1 for x <= 0, to about 1 ulp: x = k ln 2 + r, e^r - 1 = r + r^2 P(r)
// with P a degree-10 Chebyshev interpolant on |r| <= ln(2)/2 (8.6e-19,
// relative), then 2^k (e^r - 1) + (2^k - 1), whose second part is exact.
__device__ __forceinline__ double expm1_neg(double x)
{
    x = (x < -40.0) ? -40.0 : x;  // e^-40 is below half an ulp of 1
    const double k = rint(x * 1.4426950408889634);
    const double r = fma(-k, kLn2Lo, fma(-k, kLn2Hi, x));
    double p = 2.0914686968086876e-09;
    p = fma(p, r, 2.5105217004720745e-08);
    p = fma(p, r, 2.75572736431103e-07);
    p = fma(p, r, 2.7557255400206422e-06);
    p = fma(p, r, 2.4801587325547743e-05);
    p = fma(p, r, 0.00019841269874820627);
    p = fma(p, r, 0.0013888888888883748);
    p = fma(p, r, 0.008333333333326136);
    p = fma(p, r, 0.04166666666666667);
    p = fma(p, r, 0.1666666666666667);
    p = fma(p, r, 0.5);
    const double e = fma(r * r, p, r), s = ldexp(1.0, int(k));
    return fma(s, e, s - 1.0);
}

// secant susceptibility f(h)/h of the tanh-sum law (radmater.h:644-657), h >= 0
__device__ __forceinline__ double frm_chi(const double* mat, double h)
{
    const int nt = int(mat[1]);
    double chi = 0.0;
    for (int t = 0; t < nt; t++) {
        const double ms = mat[2 + t], ks = mat[5 + t];
        if (ms == 0.0) continue;
        if (h > 0.0) {
            const double u = rh_div(ks * h, ms);
            const double e = expm1_neg(-2.0 * fabs(u));
            chi += (u < 1e-8) ? ks : ms * copysign(rh_div(-e, 2.0 + e), u) / h;
        } else {
            chi += ks;
        }
    }
    return chi;
}

// |M|(h) of a tabulated law (node triples x, y, d): cubic Hermite between
// nodes, y[0] below the first, the last slope beyond the last
// (radmater.cpp:619-646)
__device__ __forceinline__ double tab_f(const double* t, int L, double h)
{
    if (h < t[0]) return t[1];
    if (h >= t[3 * (L - 1)]) return t[3 * (L - 1) + 1] + (h - t[3 * (L - 1)]) * t[3 * (L - 1) + 2];
    int lo = 0, hi = L - 1;  // t[3 lo] <= h < t[3 hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (t[3 * mid] <= h) lo = mid;
        else hi = mid;
    }
    const double* a = t + 3 * lo;
    const double s = a[3] - a[0], u = h - a[0];
    const double sl = (a[4] - a[1]) / s;
    const double c2 = (3.0 * sl - 2.0 * a[2] - a[5]) / s;
    const double c3 = (-2.0 * sl + a[2] + a[5]) / (s * s);
    return a[1] + u * (a[2] + u * (c2 + u * c3));
}

// secant susceptibility |M|(h)/h of an isotropic nonlinear law (kind 2: tanh
// sum, kind 3: table)
__device__ __forceinline__ double law_chi(const double* mat, const double* tab, double h)
{
    if (int(mat[0]) == 3) {
        const double* t = tab + 3 * int64_t(mat[1]);
        return (h > 0.0) ? tab_f(t, int(mat[2]), h) / h : t[2];
    }
    return frm_chi(mat, h);
}

// |M|(h) and d|M|/dh of an isotropic nonlinear law (kind 2 tanh sum, kind 3
// table), h > 0.
__device__ __forceinline__ void law_f_df(const double* mat, const double* tab, double h, double& f,
                                         double& df)
{
    if (int(mat[0]) == 3) {
        const double* t = tab + 3 * int64_t(mat[1]);
        const int L = int(mat[2]);
        if (h < t[0]) {
            f = t[1];
            df = 0.0;
            return;
        }
        if (h >= t[3 * (L - 1)]) {
            f = t[3 * (L - 1) + 1] + (h - t[3 * (L - 1)]) * t[3 * (L - 1) + 2];
            df = t[3 * (L - 1) + 2];
            return;
        }
        int lo = 0, hi = L - 1;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (t[3 * mid] <= h) lo = mid;
            else hi = mid;
        }
        const double* a = t + 3 * lo;
        const double sg = a[3] - a[0], u = h - a[0];
        const double sl = (a[4] - a[1]) / sg;
        const double c2 = (3.0 * sl - 2.0 * a[2] - a[5]) / sg;
        const double c3 = (-2.0 * sl + a[2] + a[5]) / (sg * sg);
        f = a[1] + u * (a[2] + u * (c2 + u * c3));
        df = a[2] + u * (2.0 * c2 + 3.0 * c3 * u);
        return;
    }
    // The three terms side by side (an absent one has ks = 0 and adds 0).  An
    // element's solve is a chain of about nine evaluations on one lane, so
    // their length is the relaxation step's time: with the library's expm1 and
    // four IEEE divisions a term a step of 8,000 elements took 38 us, with
    // these 31.
    const int nt = int(mat[1]);
    f = 0.0;
    df = 0.0;
#pragma unroll
    for (int t = 0; t < 3; t++) {
        const bool on = t < nt && mat[2 + t] != 0.0;
        const double ms = on ? mat[2 + t] : 1.0, ks = on ? mat[5 + t] : 0.0;
        const double u = rh_div(ks * h, ms);
        // tanh u and sech^2 u from one expm1: with e = exp(-2|u|) - 1,
        // tanh|u| = -e / (2 + e) and sech^2 u = 4 (1 + e) / (2 + e)^2
        const double e = expm1_neg(-2.0 * fabs(u));
        const double q = rh_rcp(2.0 + e);
        f = fma(ms, copysign(-e * q, u), f);
        df = fma(ks, 4.0 * (1.0 + e) * (q * q), df);
    }
}

__device__ void local_solve(const double* mat, const double* q, const double* heff, double* Mp,
                            double* Hl, const double* tab, double warm)
{
    const int kind = int(mat[0]);
    const double* mr = mat + 13;
    double qmr[3];
    mat3_vec(q, mr, qmr);
    const double b[3] = {heff[0] + qmr[0], heff[1] + qmr[1], heff[2] + qmr[2]};
    if (kind == 0) {
        double A[9];
        for (int k = 0; k < 9; k++) A[k] = mat[1] * q[k];
        solve_IminusA(A, b, Hl);
        for (int k = 0; k < 3; k++) Mp[k] = mat[1] * Hl[k] + mr[k];
        return;
    }
    if (kind == 1) {
        const double* K = mat + 4;
        double A[9];
        for (int a = 0; a < 3; a++)
            for (int c = 0; c < 3; c++)
                A[3 * a + c] = q[3 * a] * K[c] + q[3 * a + 1] * K[3 + c] + q[3 * a + 2] * K[6 + c];
        solve_IminusA(A, b, Hl);
        double kh[3];
        mat3_vec(K, Hl, kh);
        for (int k = 0; k < 3; k++) Mp[k] = kh[k] + mr[k];
        return;
    }
    // nonlinear isotropic: find h = |H(h)|, H(h) = (I - chi(h) Q)^{-1} b with
    // the secant susceptibility chi(h) = |M|(h)/h.  Safeguarded Newton on
    // g(h) = |H(h)| - h inside a bracket g(lo) > 0 > g(hi), started from the
    // previous iteration's |H| (warm) when it lies in the bracket; where a
    // Newton step leaves the bracket, false position, and bisection after two
    // false-position steps in a row.
    const double bn = sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
    if (!(bn > 0.0)) {
        Hl[0] = Hl[1] = Hl[2] = 0.0;
        for (int k = 0; k < 3; k++) Mp[k] = mr[k];
        return;
    }
    const double chi0 = law_chi(mat, tab, 0.0);
    // |H(h)| into the return value, H(h) into Hv, dg/dh into *dg (if given)
    auto phi = [&](double h, double* Hv, double* dg) -> double {
        double chi = chi0, dchi = 0.0;
        if (h > 0.0) {
            double f, df;
            law_f_df(mat, tab, h, f, df);
            chi = f / h;
            dchi = (df - chi) / h;
        }
        double A[9];
        for (int k = 0; k < 9; k++) A[k] = -chi * q[k];
        A[0] += 1.0;
        A[4] += 1.0;
        A[8] += 1.0;
        double Ai[9];
        inv3d(A, Ai);
        mat3_vec(Ai, b, Hv);
        const double hv = sqrt(Hv[0] * Hv[0] + Hv[1] * Hv[1] + Hv[2] * Hv[2]);
        if (dg) {
            double qh[3], dH[3];
            mat3_vec(q, Hv, qh);
            mat3_vec(Ai, qh, dH);
            *dg = (hv > 0.0 ? dchi * (Hv[0] * dH[0] + Hv[1] * dH[1] + Hv[2] * dH[2]) / hv : 0.0) - 1.0;
        }
        return hv;
    };
    double Hv[3];
    double lo = 0.0, glo = phi(0.0, Hv, nullptr);
    double hi = bn, ghi = phi(hi, Hv, nullptr) - hi;
    for (int k = 0; k < 60 && ghi > 0.0; k++) {
        lo = hi;
        glo = ghi;
        hi *= 2.0;
        ghi = phi(hi, Hv, nullptr) - hi;
    }
    double h;
    if (!(glo > 0.0) || !(ghi < 0.0)) {
        h = (glo <= 0.0) ? lo : hi;
    } else {
        h = (warm > lo && warm < hi) ? warm : (lo * ghi - hi * glo) / (ghi - glo);
        int fp = 0;
        for (int it = 0; it < 60; it++) {
            double dg;
            const double g = phi(h, Hv, &dg) - h;
            if (g == 0.0) break;
            if (g > 0.0) {
                lo = h;
                glo = g;
            } else {
                hi = h;
                ghi = g;
            }
            double hn = (dg < 0.0) ? h - g / dg : -1.0;
            if (hn > lo && hn < hi) {
                fp = 0;
            } else {
                hn = (fp < 2) ? (lo * ghi - hi * glo) / (ghi - glo) : 0.5 * (lo + hi);
                fp = (fp < 2) ? fp + 1 : 0;
                if (!(hn > lo && hn < hi)) hn = 0.5 * (lo + hi);
            }
            const bool done = fabs(hn - h) <= 1e-15 * bn || hi - lo <= 1e-15 * bn;
            h = hn;
            if (done) break;
        }
    }
    phi(h, Hv, nullptr);
    const double hn = sqrt(Hv[0] * Hv[0] + Hv[1] * Hv[1] + Hv[2] * Hv[2]);
    const double chi = law_chi(mat, tab, hn);
    for (int k = 0; k < 3; k++) {
        Hl[k] = Hv[k];
        Mp[k] = chi * Hv[k] + mr[k];
    }
}

// FP64 defect of the stored-matrix field: out = hext + rowT*H64 - y - Qii M,
// with H64 the FP64 field of all elements at the collocation points (lab
// frame) and y the stored-matrix product (diagonal blocks excluded).
__global__ __launch_bounds__(256) void k_refine_defect(int64_t n, const double* __restrict__ H64,
                                                       const double* __restrict__ rowt,
                                                       const double* __restrict__ y,
                                                       const double* __restrict__ qdiag,
                                                       const double* __restrict__ M,
                                                       const double* __restrict__ hext,
                                                       double* __restrict__ out)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    double h[3] = {H64[3 * i], H64[3 * i + 1], H64[3 * i + 2]};
    if (rowt) {
        const double* t = rowt + 9 * i;
        const double g[3] = {h[0], h[1], h[2]};
        for (int k = 0; k < 3; k++) h[k] = t[3 * k] * g[0] + t[3 * k + 1] * g[1] + t[3 * k + 2] * g[2];
    }
    const double* D = qdiag + 9 * i;
    const double m[3] = {M[3 * i], M[3 * i + 1], M[3 * i + 2]};
    for (int k = 0; k < 3; k++)
        out[3 * i + k] = hext[3 * i + k] + (h[k] - y[3 * i + k]) -
                         (D[3 * k] * m[0] + D[3 * k + 1] * m[1] + D[3 * k + 2] * m[2]);
}

__global__ __launch_bounds__(kRelaxLanes) void k_relax_update(int64_t n, const double* __restrict__ mats,
                                                              const double* __restrict__ tab,
                                                              const double* __restrict__ hext,
                                                              const double* __restrict__ qdiag,
                                                              const double* __restrict__ y,
                                                              const double* __restrict__ M,
                                                              double* __restrict__ F,
                                                              double* __restrict__ Hout,
                                                              double* __restrict__ partials)
{
    __shared__ double red[3][kRelaxLanes];
    const int64_t i = int64_t(blockIdx.x) * kRelaxLanes + threadIdx.x;
    double f2 = 0.0, mm = 0.0, hh = 0.0;
    if (i < n) {
        const double heff[3] = {y[3 * i] + hext[3 * i], y[3 * i + 1] + hext[3 * i + 1],
                                y[3 * i + 2] + hext[3 * i + 2]};
        // the previous local field's magnitude starts the nonlinear solve
        const double warm = sqrt(Hout[3 * i] * Hout[3 * i] + Hout[3 * i + 1] * Hout[3 * i + 1] +
                                 Hout[3 * i + 2] * Hout[3 * i + 2]);
        double mp[3], hl[3];
        local_solve(mats + 16 * i, qdiag + 9 * i, heff, mp, hl, tab, warm);
        for (int k = 0; k < 3; k++) {
            const double d = mp[k] - M[3 * i + k];
            F[3 * i + k] = d;
            Hout[3 * i + k] = hl[k];
            f2 += d * d;
        }
        mm = sqrt(mp[0] * mp[0] + mp[1] * mp[1] + mp[2] * mp[2]);
        hh = sqrt(hl[0] * hl[0] + hl[1] * hl[1] + hl[2] * hl[2]);
    }
    red[0][threadIdx.x] = f2;
    red[1][threadIdx.x] = mm;
    red[2][threadIdx.x] = hh;
    __syncthreads();
    for (int st = kRelaxLanes / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            red[0][threadIdx.x] += red[0][threadIdx.x + st];
            red[1][threadIdx.x] = fmax(red[1][threadIdx.x], red[1][threadIdx.x + st]);
            red[2][threadIdx.x] = fmax(red[2][threadIdx.x], red[2][threadIdx.x + st]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partials[3 * blockIdx.x] = red[0][0];
        partials[3 * blockIdx.x + 1] = red[1][0];
        partials[3 * blockIdx.x + 2] = red[2][0];
    }
}

// ---------------------------------------------------------------- Newton-Krylov
// Material law at the total field of the current magnetization: H = y + Qii M
// + hext, F = M_mat(H) - M, tangent D = dM_mat/dH (D = mp hh^T + sc (I - hh^T)
// for isotropic laws, hh = H/|H|, sc = |M|/|H|, mp = d|M|/d|H|; chi0 I at
// H = 0; chi I or K for linear laws) and the block preconditioner
// P = (I - D Qii)^{-1}.  partials per block: [sum |F|^2, max |M_mat|, max |H|].
__global__ __launch_bounds__(kRelaxLanes) void k_nk_material(int64_t n, const double* __restrict__ mats,
                                                     const double* __restrict__ tab,
                                                     const double* __restrict__ hext,
                                                     const double* __restrict__ qdiag,
                                                     const double* __restrict__ y,
                                                     const double* __restrict__ M,
                                                     double* __restrict__ F, double* __restrict__ D,
                                                     double* __restrict__ P, double* __restrict__ Hout,
                                                     double* __restrict__ partials)
{
    __shared__ double red[3][kRelaxLanes];
    const int64_t i = int64_t(blockIdx.x) * kRelaxLanes + threadIdx.x;
    double f2 = 0.0, mm = 0.0, hh = 0.0;
    if (i < n) {
        const double* mat = mats + 16 * i;
        const double* q = qdiag + 9 * i;
        const double m[3] = {M[3 * i], M[3 * i + 1], M[3 * i + 2]};
        double qm[3];
        mat3_vec(q, m, qm);
        double H[3];
        for (int k = 0; k < 3; k++) H[k] = y[3 * i + k] + qm[k] + hext[3 * i + k];
        const int kind = int(mat[0]);
        double d[9], mn[3];
        if (kind == 1) {
            for (int k = 0; k < 9; k++) d[k] = mat[4 + k];
            mat3_vec(d, H, mn);
        } else {
            double sc, mp;
            const double h = sqrt(H[0] * H[0] + H[1] * H[1] + H[2] * H[2]);
            if (kind == 0) {
                sc = mp = mat[1];
            } else if (h > 1e-300) {
                double f, df;
                law_f_df(mat, tab, h, f, df);
                sc = f / h;
                mp = df;
            } else {
                sc = mp = law_chi(mat, tab, 0.0);
            }
            const double e[3] = {h > 1e-300 ? H[0] / h : 0.0, h > 1e-300 ? H[1] / h : 0.0,
                                 h > 1e-300 ? H[2] / h : 0.0};
            for (int a = 0; a < 3; a++)
                for (int b = 0; b < 3; b++) d[3 * a + b] = (mp - sc) * e[a] * e[b] + (a == b ? sc : 0.0);
            for (int k = 0; k < 3; k++) mn[k] = sc * H[k];
        }
        for (int k = 0; k < 3; k++) mn[k] += mat[13 + k];
        // P = (I - D Qii)^{-1}
        double a[9];
        for (int r = 0; r < 3; r++)
            for (int c = 0; c < 3; c++)
                a[3 * r + c] = (r == c ? 1.0 : 0.0) -
                               (d[3 * r] * q[c] + d[3 * r + 1] * q[3 + c] + d[3 * r + 2] * q[6 + c]);
        double pinv[9];
        inv3d(a, pinv);
        for (int k = 0; k < 9; k++) {
            D[9 * i + k] = d[k];
            P[9 * i + k] = pinv[k];
        }
        for (int k = 0; k < 3; k++) {
            const double fk = mn[k] - m[k];
            F[3 * i + k] = fk;
            Hout[3 * i + k] = H[k];
            f2 += fk * fk;
        }
        mm = sqrt(mn[0] * mn[0] + mn[1] * mn[1] + mn[2] * mn[2]);
        hh = sqrt(H[0] * H[0] + H[1] * H[1] + H[2] * H[2]);
    }
    red[0][threadIdx.x] = f2;
    red[1][threadIdx.x] = mm;
    red[2][threadIdx.x] = hh;
    __syncthreads();
    for (int st = kRelaxLanes / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            red[0][threadIdx.x] += red[0][threadIdx.x + st];
            red[1][threadIdx.x] = fmax(red[1][threadIdx.x], red[1][threadIdx.x + st]);
            red[2][threadIdx.x] = fmax(red[2][threadIdx.x], red[2][threadIdx.x + st]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partials[3 * blockIdx.x] = red[0][0];
        partials[3 * blockIdx.x + 1] = red[1][0];
        partials[3 * blockIdx.x + 2] = red[2][0];
    }
}

// z = P v per element (3x3 blocks).
__global__ __launch_bounds__(256) void k_nk_prec(int64_t n, const double* __restrict__ P,
                                                 const double* __restrict__ v, double* __restrict__ z)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const double x[3] = {v[3 * i], v[3 * i + 1], v[3 * i + 2]};
    double o[3];
    mat3_vec(P + 9 * i, x, o);
    for (int k = 0; k < 3; k++) z[3 * i + k] = o[k];
}

// w = z - D (y + Qii z): the Newton operator (I - D Q) applied to z, with
// y = offdiag(Q) z from the matrix pass.
__global__ __launch_bounds__(256) void k_nk_apply(int64_t n, const double* __restrict__ D,
                                                  const double* __restrict__ qdiag,
                                                  const double* __restrict__ z,
                                                  const double* __restrict__ y, double* __restrict__ w)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const double zz[3] = {z[3 * i], z[3 * i + 1], z[3 * i + 2]};
    double qz[3];
    mat3_vec(qdiag + 9 * i, zz, qz);
    const double g[3] = {y[3 * i] + qz[0], y[3 * i + 1] + qz[1], y[3 * i + 2] + qz[2]};
    double dg[3];
    mat3_vec(D + 9 * i, g, dg);
    for (int k = 0; k < 3; k++) w[3 * i + k] = zz[k] - dg[k];
}

// Dot products of w with nv basis vectors (V, leading dimension ldv) and with
// itself: grid (chunks, nv + 1), partials[j * chunks + chunk].
__global__ __launch_bounds__(256) void k_mdot(int nv, const double* __restrict__ V, int64_t ldv,
                                              const double* __restrict__ w, int64_t len,
                                              double* __restrict__ partials)
{
    __shared__ double red[4];
    const int j = blockIdx.y;
    const double* a = (j < nv) ? V + int64_t(j) * ldv : w;
    double acc = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < len; i += int64_t(gridDim.x) * 256)
        acc += a[i] * w[i];
    const double v = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partials[int64_t(j) * gridDim.x + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// out = cb * base + sum_j c_j V_j (base may be null; out may alias base).
__global__ __launch_bounds__(256) void k_vcomb(int nv, const double* __restrict__ V, int64_t ldv,
                                               Coef64 c, const double* base, double cb, int64_t len,
                                               double* out)
{
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < len; i += int64_t(gridDim.x) * 256) {
        double acc = base ? cb * base[i] : 0.0;
        for (int j = 0; j < nv; j++) acc += c.c[j] * V[int64_t(j) * ldv + i];
        out[i] = acc;
    }
}

// ---------------------------------------------------------------- vector helpers
struct CombPack {
    const double* v[kCombMax];
    double c[kCombMax];
};

__global__ __launch_bounds__(256) void k_lincomb(int nv, CombPack pk, int64_t len,
                                                 double* __restrict__ y)
{
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < len;
         i += int64_t(gridDim.x) * 256) {
        double acc = 0.0;
        for (int k = 0; k < nv; k++) acc += pk.c[k] * pk.v[k][i];
        y[i] = acc;
    }
}

// The element update of the relaxation: H_i = (I - Q_ii K)^{-1} (y + hext + ...)
// by the element's material law, started from the previous local field.
struct MaterialLaw {
    const double *mats, *tab, *hext, *qdiag, *y;
    double* Hout;
    __device__ __forceinline__ void operator()(int64_t i, double* mp, double& hh) const
    {
        double hl[3];
        const double heff[3] = {y[3 * i] + hext[3 * i], y[3 * i + 1] + hext[3 * i + 1],
                                y[3 * i + 2] + hext[3 * i + 2]};
        const double warm = sqrt(Hout[3 * i] * Hout[3 * i] + Hout[3 * i + 1] * Hout[3 * i + 1] +
                                 Hout[3 * i + 2] * Hout[3 * i + 2]);
        local_solve(mats + 16 * i, qdiag + 9 * i, heff, mp, hl, tab, warm);
        for (int k = 0; k < 3; k++) Hout[3 * i + k] = hl[k];
        hh = sqrt(hl[0] * hl[0] + hl[1] * hl[1] + hl[2] * hl[2]);
    }
};

__global__ __launch_bounds__(kRelaxLanes) void k_relax_step(int64_t n, const double* __restrict__ mats,
                                                            const double* __restrict__ tab,
                                                            const double* __restrict__ hext,
                                                            const double* __restrict__ qdiag,
                                                            const double* __restrict__ y,
                                                            const double* __restrict__ M,
                                                            double* __restrict__ F,
                                                            double* __restrict__ Hout,
                                                            double* __restrict__ partials, HistPack hp)
{
    relax_step_block(n, MaterialLaw{mats, tab, hext, qdiag, y, Hout}, M, F, partials, hp.Fp, hp.xp, hp.dFw, hp.dXw,
                     hp.dF, hp.nh);
}

// The same step in the device-driven loop (history slots from the state); the
// last block to finish runs the Anderson step on the partials of all blocks.
__global__ __launch_bounds__(kRelaxLanes) void k_relax_step_dev(int64_t n, const double* __restrict__ mats,
                                                                const double* __restrict__ tab,
                                                                const double* __restrict__ hext,
                                                                const double* __restrict__ qdiag,
                                                                const double* __restrict__ y,
                                                                const double* __restrict__ M,
                                                                double* __restrict__ F,
                                                                double* __restrict__ Hout,
                                                                double* __restrict__ partials, HistBufs hb,
                                                                RelaxDevState* __restrict__ st)
{
    relax_step_dev(n, MaterialLaw{mats, tab, hext, qdiag, y, Hout}, M, F, partials, hb, st);
}

// The update of the device-driven loop (grid-stride over the 3n components).
__global__ __launch_bounds__(256) void k_update_dev(int64_t n3, double* __restrict__ x,
                                                    const double* __restrict__ F, HistBufs hb,
                                                    double* __restrict__ M_out,
                                                    const RelaxDevState* __restrict__ st)
{
    const int done = st->done;
    if (done == 2) return;
    const UpdateCoef c(st);
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n3; i += int64_t(gridDim.x) * 256) {
        if (done == 1) M_out[i] = x[i] + F[i];
        else x[i] = c.apply(x[i], F, hb, i);
    }
}

// ---------------------------------------------------------------- currents
__global__ __launch_bounds__(256) void k_current(int64_t ns, const int32_t* __restrict__ kind,
                                                 const double* __restrict__ par,
                                                 const double* __restrict__ cp,
                                                 const double* __restrict__ pts, int64_t np,
                                                 double* __restrict__ B)
{
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (p >= np) return;
    const double x[3] = {pts[3 * p], pts[3 * p + 1], pts[3 * p + 2]};
    double b[3] = {0, 0, 0};
    for (int64_t s = 0; s < ns; s++) current_add(kind[s], par + 12 * s, cp + 24 * s, x, b);
    for (int k = 0; k < 3; k++) B[3 * p + k] += b[k];
}

}  // namespace

// ---------------------------------------------------------------- launchers
int64_t far_tet_doubles(int64_t ntet) { return kFarTet * ntet; }
int64_t hex_doubles(int64_t nhex) { return kHex * nhex; }

hipError_t launch_far_tets(const DevModel& m, double* tet, hipStream_t s)
{
    const int64_t ntet = m.koff[2] - m.koff[1];
    if (ntet > 0) hipLaunchKernelGGL(k_far_records, dim3(unsigned((ntet + 255) / 256)), dim3(256), 0, s, m, tet);
    return hipGetLastError();
}

hipError_t launch_hexes(const DevModel& m, double* hex, int32_t* hex_at, hipStream_t s)
{
    const int64_t ngen = m.koff[3] - m.koff[2];
    if (ngen > 0) hipLaunchKernelGGL(k_hex_records, dim3(unsigned(ngen)), dim3(64), 0, s, m, hex, hex_at);
    return hipGetLastError();
}

hipError_t launch_assemble(const DevModel& m, void* Q, int elem_bytes, int64_t ld, double* qdiag,
                           int64_t r0, int64_t r1, hipStream_t s, bool far32, int planes, int32_t* flag)
{
    if (m.n == 0 || r1 <= r0) return hipSuccess;
    if (planes != 0 && (m.sym || !m.rowt_identity || (planes != 5 && planes != 6) || (planes == 5 && !flag)))
        return hipErrorInvalidValue;
    if (elem_bytes == 4) {
        float* q = static_cast<float*>(Q);
        if (planes == 5) return asm_dispatch<false, false, float, 5>(m, q, ld, qdiag, r0, r1, s, far32, flag);
        if (planes == 6) return asm_dispatch<false, false, float, 6>(m, q, ld, qdiag, r0, r1, s, far32, flag);
        if (!m.sym && m.rowt_identity) return asm_dispatch<false, false>(m, q, ld, qdiag, r0, r1, s, far32, flag);
        if (m.rowt_identity) return asm_dispatch<true, false>(m, q, ld, qdiag, r0, r1, s, far32, flag);
        return asm_dispatch<true, true>(m, q, ld, qdiag, r0, r1, s, far32, flag);
    }
    double* q = static_cast<double*>(Q);
    if (planes == 5) return asm_dispatch<false, false, double, 5>(m, q, ld, qdiag, r0, r1, s, false, flag);
    if (planes == 6) return asm_dispatch<false, false, double, 6>(m, q, ld, qdiag, r0, r1, s, false, flag);
    if (!m.sym && m.rowt_identity) return asm_dispatch<false, false>(m, q, ld, qdiag, r0, r1, s, false, flag);
    if (m.rowt_identity) return asm_dispatch<true, false>(m, q, ld, qdiag, r0, r1, s, false, flag);
    return asm_dispatch<true, true>(m, q, ld, qdiag, r0, r1, s, false, flag);
}

namespace {
// element splits for one kind slot: enough workgroups to fill the chip
int64_t slot_splits(int64_t np, int64_t cnt, int64_t per_block = 256, int64_t least = 16)
{
    if (cnt == 0) return 0;
    const int64_t blocks = (np + per_block - 1) / per_block;
    if (blocks >= 2048 || cnt < 64) return 1;
    int64_t sp = (2048 + blocks - 1) / blocks;
    sp = std::min<int64_t>(sp, std::max<int64_t>(1, cnt / least));
    return std::max<int64_t>(1, sp);
}

template <class R, bool SYM, int KIND>
void field_slot(const DevModel& m, const double* M, const double* pts, int64_t np, int64_t splits,
                int64_t slice0, double* B, double* H, double* part, hipStream_t s)
{
    const int64_t cnt = m.koff[KIND + 1] - m.koff[KIND];
    int64_t js = (cnt + splits - 1) / splits;
    const dim3 grid{unsigned((np + 255) / 256), unsigned(splits), 1u};
    constexpr bool f32 = sizeof(R) == 4;
    if (KIND == 1 && m.charged) {
        js = (js + kTetTile - 1) / kTetTile * kTetTile;
        if constexpr (f32) {
            hipLaunchKernelGGL((k_field_tet<float, SYM, kPassFar>), grid, dim3(256), 0, s, m, pts, np, js,
                               slice0, B, H, part);
            hipLaunchKernelGGL((k_field_tet<double, SYM, kPassNear>), grid, dim3(256), 0, s, m, pts, np, js,
                               slice0, B, H, part);
        } else {
            hipLaunchKernelGGL((k_field_tet<double, SYM, kPassAll>), grid, dim3(256), 0, s, m, pts, np, js,
                               slice0, B, H, part);
        }
        return;
    }
    if constexpr (f32) {
        hipLaunchKernelGGL((k_field<float, SYM, KIND, kPassFar>), grid, dim3(256), 0, s, m, M, pts, np, js,
                           slice0, B, H, part);
        hipLaunchKernelGGL((k_field<double, SYM, KIND, kPassNear>), grid, dim3(256), 0, s, m, M, pts, np, js,
                           slice0, B, H, part);
    } else {
        hipLaunchKernelGGL((k_field<double, SYM, KIND, kPassAll>), grid, dim3(256), 0, s, m, M, pts, np, js,
                           slice0, B, H, part);
    }
}

bool mesh_on(const DevModel& m) { return m.use_mesh && m.mesh.active; }

// Points per lane of the mesh sweep.  Two from 1e8 (point, entity) pairs on:
// below that a sweep is too short to fill the chip with half as many waves and
// its latency decides.  Measured (FP64, us, one / two points per lane):
// 1,000 points on the 8,000-tetrahedron yoke (2.9e7 pairs) 142 / 171, 8,000
// points (2.3e8) 441 / 409, 32,000 points 1,513 / 1,317; 8,000 points on the
// 1,000-tetrahedron yoke (2.9e7) 135 / 152; 1,000 points on the 20,000-element
// ring (1.3e8) 344 / 327.
int64_t mesh_points(const DevModel& m, int64_t np)
{
    return double(np) * double(m.mesh.ne + m.mesh.nf) >= 1e8 ? 2 : 1;
}

// slices per kind slot (0 blocks, 1 tetrahedra, 2 general polyhedra); in the
// mesh form slot 1 carries the whole mesh and slot 2 is empty
void slot_plan(const DevModel& m, int64_t np, int64_t sp[3], int64_t work_cap)
{
    sp[0] = slot_splits(np, m.koff[1] - m.koff[0]);
    if (mesh_on(m)) {
        sp[1] = slot_splits(np, m.mesh.ne + m.mesh.nf, 256 * mesh_points(m, np));
        sp[2] = 0;
    } else {
        sp[1] = slot_splits(np, m.koff[2] - m.koff[1]);
        // slices of 8: the near elements of a point lie side by side, and a slice
        // of 16 of them is the sweep's longest wave (2,048 points, 1,000
        // hexahedra: 191 us with 16, 128 with 8)
        sp[2] = slot_splits(np, m.koff[3] - m.koff[2], 256, 8);
    }
    if (work_cap < 0) return;
    // halve the largest split count until the partials fit or every slot is
    // down to one split
    for (;;) {
        const int64_t total = sp[0] + sp[1] + sp[2];
        if (total <= 1 || 6 * np * total <= work_cap) return;
        int big = 0;
        for (int k = 1; k < 3; k++)
            if (sp[k] > sp[big]) big = k;
        if (sp[big] <= 1) return;
        sp[big] = (sp[big] + 1) / 2;
    }
}

template <class R, bool SYM>
hipError_t field_all(const DevModel& m, const double* M, const double* pts, int64_t np, double* B,
                     double* H, double* work, int64_t work_cap, hipStream_t s)
{
    int64_t sp[3];
    slot_plan(m, np, sp, work_cap);
    if (work_cap >= 0 && sp[0] + sp[1] + sp[2] > 1 && 6 * np * (sp[0] + sp[1] + sp[2]) > work_cap)
        return hipErrorInvalidValue;
    const int64_t total = sp[0] + sp[1] + sp[2];
    double* part = (total > 1) ? work : nullptr;
    int64_t slice0 = 0;
    if (sp[0]) field_slot<R, SYM, 0>(m, M, pts, np, sp[0], slice0, B, H, part, s);
    slice0 += sp[0];
    if (sp[1] && mesh_on(m)) {
        const int64_t per = 256 * mesh_points(m, np);
        const dim3 grid{unsigned((np + per - 1) / per), unsigned(sp[1]), 1u};
        if (mesh_points(m, np) == 2)
            hipLaunchKernelGGL((k_field_mesh<R, 2>), grid, dim3(256), 0, s, m, pts, np, sp[1], slice0, B, H, part);
        else
            hipLaunchKernelGGL((k_field_mesh<R, 1>), grid, dim3(256), 0, s, m, pts, np, sp[1], slice0, B, H, part);
    } else if (sp[1]) {
        field_slot<R, SYM, 1>(m, M, pts, np, sp[1], slice0, B, H, part, s);
    }
    slice0 += sp[1];
    if (sp[2]) field_slot<R, SYM, 2>(m, M, pts, np, sp[2], slice0, B, H, part, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || total <= 1) return e;
    // about 16 rows per thread: fewer threads per column read longer lines,
    // more shorten the chain of additions
    auto reduce = [&](auto g) {
        constexpr int G = decltype(g)::value;
        const int64_t cols = 256 / G;
        hipLaunchKernelGGL(k_field_reduce<G>, dim3(unsigned((6 * np + cols - 1) / cols)), dim3(256), 0, s, np, total,
                           part, B, H);
    };
    if (total <= 16) reduce(std::integral_constant<int, 1>{});
    else if (total <= 64) reduce(std::integral_constant<int, 4>{});
    else if (total <= 256) reduce(std::integral_constant<int, 16>{});
    else reduce(std::integral_constant<int, 64>{});
    return hipGetLastError();
}
}  // namespace

int64_t field_slices(const DevModel& m, int64_t np, int64_t work_cap)
{
    int64_t sp[3];
    slot_plan(m, np, sp, work_cap);
    return std::max<int64_t>(1, sp[0] + sp[1] + sp[2]);
}

hipError_t launch_field(const DevModel& m0, const double* M, const double* pts, int64_t np,
                        double* B, double* H, double* work, double* charged, bool fp32,
                        hipStream_t s, int64_t work_cap)
{
    if (np == 0) return hipSuccess;
    if (m0.n == 0) {
        if (B) (void)hipMemsetAsync(B, 0, size_t(3 * np) * sizeof(double), s);
        if (H) (void)hipMemsetAsync(H, 0, size_t(3 * np) * sizeof(double), s);
        return hipGetLastError();
    }
    DevModel m = m0;
    const int64_t ntet = m.koff[2] - m.koff[1];
    if (mesh_on(m)) {
        const MeshDev& md = m.mesh;
        if (md.ne)
            hipLaunchKernelGGL(k_mesh_charge_edges, dim3(unsigned((md.ne + 255) / 256)), dim3(256), 0, s,
                               md, M, fp32);
        if (md.nf)
            hipLaunchKernelGGL(k_mesh_charge_faces, dim3(unsigned((md.nf + 255) / 256)), dim3(256), 0, s,
                               md, M, fp32);
        if (md.ni)
            hipLaunchKernelGGL(k_mesh_charge_in, dim3(unsigned((md.ni + 255) / 256)), dim3(256), 0, s, md,
                               M);
    } else if (ntet > 0 && charged) {
        hipLaunchKernelGGL(k_charge_tets, dim3(unsigned((ntet + 255) / 256)), dim3(256), 0, s, m, M,
                           charged);
        m.charged = charged;
    }
    if (fp32) return m.sym ? field_all<float, true>(m, M, pts, np, B, H, work, work_cap, s)
                           : field_all<float, false>(m, M, pts, np, B, H, work, work_cap, s);
    return m.sym ? field_all<double, true>(m, M, pts, np, B, H, work, work_cap, s)
                 : field_all<double, false>(m, M, pts, np, B, H, work, work_cap, s);
}

hipError_t launch_matvec(const void* Q, int elem_bytes, int64_t nrows, int64_t ld, const double* x,
                         const double* add, double* y, hipStream_t s, const int32_t* skip)
{
    if (nrows <= 0) return hipSuccess;
// rows per wave of the matrix pass: on the C-yoke (24,000 x 24,064) 4 rows
// measured 0.668 ms FP64 / 0.358 ms FP32, 2 rows 0.695 / 0.394, 8 rows
// 0.870 / 0.487; unrolling the column loop (RH_MV_UNROLL) gained nothing
#ifndef RH_MV_RW
#define RH_MV_RW 4
#endif
    constexpr int RW = RH_MV_RW;
    const int64_t waves = (nrows + RW - 1) / RW;
    const int64_t blocks = (waves + 3) / 4;
    if (elem_bytes == 4)
        hipLaunchKernelGGL((k_matvec_f32<RW>), dim3(unsigned(blocks)), dim3(256), 0, s,
                           static_cast<const float*>(Q), nrows, ld, x, add, y, skip);
    else
        hipLaunchKernelGGL((k_matvec_f64<RW>), dim3(unsigned(blocks)), dim3(256), 0, s,
                           static_cast<const double*>(Q), nrows, ld, x, add, y, skip);
    return hipGetLastError();
}

hipError_t launch_matvec_sym(const void* Q, int elem_bytes, int planes, int64_t nel, int64_t ldp,
                             const double* x, const double* add, double* y, hipStream_t s,
                             const int32_t* skip)
{
    if (nel <= 0) return hipSuccess;
    if ((planes != 5 && planes != 6) || ldp % 256 != 0) return hipErrorInvalidValue;
    constexpr int ER = RH_MVS_ER;
    const int64_t waves = (nel + ER - 1) / ER;
    const dim3 grid{unsigned((waves + 3) / 4), 1u, 1u};
    if (elem_bytes == 4) {
        const float* q = static_cast<const float*>(Q);
        if (planes == 5)
            hipLaunchKernelGGL((k_matvec_sym_f32<5, ER>), grid, dim3(256), 0, s, q, nel, ldp, x, add, y, skip);
        else
            hipLaunchKernelGGL((k_matvec_sym_f32<6, ER>), grid, dim3(256), 0, s, q, nel, ldp, x, add, y, skip);
    } else {
        const double* q = static_cast<const double*>(Q);
        if (planes == 5)
            hipLaunchKernelGGL((k_matvec_sym_f64<5, ER>), grid, dim3(256), 0, s, q, nel, ldp, x, add, y, skip);
        else
            hipLaunchKernelGGL((k_matvec_sym_f64<6, ER>), grid, dim3(256), 0, s, q, nel, ldp, x, add, y, skip);
    }
    return hipGetLastError();
}

int64_t relax_blocks(int64_t n) { return (n + kRelaxLanes - 1) / kRelaxLanes; }

hipError_t launch_relax_update(int64_t n, const double* mats, const double* tab, const double* hext,
                               const double* qdiag, const double* y, const double* M, double* F,
                               double* Hout, double* partials, hipStream_t s)
{
    hipLaunchKernelGGL(k_relax_update, dim3(unsigned(relax_blocks(n))), dim3(kRelaxLanes), 0, s, n, mats,
                       tab, hext, qdiag, y, M, F, Hout, partials);
    return hipGetLastError();
}

hipError_t launch_relax_step(int64_t n, const double* mats, const double* tab, const double* hext,
                             const double* qdiag, const double* y, const double* M, double* F,
                             double* Hout, double* partials, const HistPack& hp, hipStream_t s)
{
    if (hp.nh < 0 || hp.nh > kHistMax || (hp.nh > 0 && !hp.dFw)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_relax_step, dim3(unsigned(relax_blocks(n))), dim3(kRelaxLanes), 0, s, n, mats, tab,
                       hext, qdiag, y, M, F, Hout, partials, hp);
    return hipGetLastError();
}

hipError_t launch_relax_step_dev(int64_t n, const double* mats, const double* tab, const double* hext,
                                 const double* qdiag, const double* y, const double* M, double* F,
                                 double* Hout, double* partials, const HistBufs& hb, RelaxDevState* st,
                                 hipStream_t s)
{
    hipLaunchKernelGGL(k_relax_step_dev, dim3(unsigned(relax_blocks(n))), dim3(kRelaxLanes), 0, s, n, mats, tab,
                       hext, qdiag, y, M, F, Hout, partials, hb, st);
    return hipGetLastError();
}

hipError_t launch_update_dev(int64_t n3, double* x, const double* F, const HistBufs& hb, double* M_out,
                             const RelaxDevState* st, hipStream_t s)
{
    const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(4096, (n3 + 255) / 256));
    hipLaunchKernelGGL(k_update_dev, dim3(unsigned(blocks)), dim3(256), 0, s, n3, x, F, hb, M_out, st);
    return hipGetLastError();
}

hipError_t launch_refine_defect(int64_t n, const double* H64, const double* rowt, const double* y,
                                const double* qdiag, const double* M, const double* hext,
                                double* out, hipStream_t s)
{
    hipLaunchKernelGGL(k_refine_defect, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, n, H64, rowt,
                       y, qdiag, M, hext, out);
    return hipGetLastError();
}

hipError_t launch_nk_material(int64_t n, const double* mats, const double* tab, const double* hext,
                              const double* qdiag, const double* y, const double* M, double* F, double* D,
                              double* P, double* Hout, double* partials, hipStream_t s)
{
    hipLaunchKernelGGL(k_nk_material, dim3(unsigned(relax_blocks(n))), dim3(kRelaxLanes), 0, s, n, mats, tab, hext,
                       qdiag, y, M, F, D, P, Hout, partials);
    return hipGetLastError();
}

hipError_t launch_nk_prec(int64_t n, const double* P, const double* v, double* z, hipStream_t s)
{
    hipLaunchKernelGGL(k_nk_prec, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, n, P, v, z);
    return hipGetLastError();
}

hipError_t launch_nk_apply(int64_t n, const double* D, const double* qdiag, const double* z, const double* y,
                           double* w, hipStream_t s)
{
    hipLaunchKernelGGL(k_nk_apply, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, n, D, qdiag, z, y, w);
    return hipGetLastError();
}

hipError_t launch_mdot(int nv, const double* V, int64_t ldv, const double* w, int64_t len, double* partials,
                       hipStream_t s)
{
    if (nv < 0 || nv > kCoefMax) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mdot, dim3(unsigned(dot_blocks(len)), unsigned(nv + 1)), dim3(256), 0, s, nv, V, ldv,
                       w, len, partials);
    return hipGetLastError();
}

hipError_t launch_vcomb(int nv, const double* V, int64_t ldv, const double* c, const double* base, double cb,
                        int64_t len, double* out, hipStream_t s)
{
    if (nv < 0 || nv > kCoefMax) return hipErrorInvalidValue;
    Coef64 cc{};
    for (int j = 0; j < nv; j++) cc.c[j] = c[j];
    const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(4096, (len + 255) / 256));
    hipLaunchKernelGGL(k_vcomb, dim3(unsigned(blocks)), dim3(256), 0, s, nv, V, ldv, cc, base, cb, len, out);
    return hipGetLastError();
}

int64_t dot_blocks(int64_t len) { return std::max<int64_t>(1, std::min<int64_t>(128, (len + 511) / 512)); }

hipError_t launch_lincomb(int nv, const double* const* v, const double* c, int64_t len, double* y,
                          hipStream_t s)
{
    if (nv < 1 || nv > kCombMax) return hipErrorInvalidValue;
    CombPack pk;
    for (int k = 0; k < nv; k++) {
        pk.v[k] = v[k];
        pk.c[k] = c[k];
    }
    const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(4096, (len + 255) / 256));
    hipLaunchKernelGGL(k_lincomb, dim3(unsigned(blocks)), dim3(256), 0, s, nv, pk, len, y);
    return hipGetLastError();
}

hipError_t launch_current(int64_t ns, const int32_t* kind, const double* par, const double* cp,
                          const double* pts, int64_t np, double* B, hipStream_t s)
{
    if (np == 0 || ns == 0) return hipSuccess;
    hipLaunchKernelGGL(k_current, dim3(unsigned((np + 255) / 256)), dim3(256), 0, s, ns, kind, par,
                       cp, pts, np, B);
    return hipGetLastError();
}

}  // namespace rh
