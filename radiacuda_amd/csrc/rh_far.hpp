// rh_far.hpp -- interaction blocks of elements that are far from every point
// of a wave, or from a lane's own point (blocks) (device only).
//
// With S = Ra + Rb the sum of an edge's end distances, its integral is
// 2 atanh(len / S) and a triangle's half solid angle has the tangent
// 2 r0 . (r1 x r2) / (S01 S12 S20 - R2 l01^2 - R1 l02^2 - R0 l12^2)
// (rh_mesh.hpp), so a tetrahedron costs 4 offsets and roots, 6 sums and 9
// divisions with short polynomials: about 270 issue slots against 750 for the
// form that also holds next to the element (eval_tet: logarithms of
// cancellation-free ratios, octant-reduced arctangents, selects).  Every term
// keeps a relative error of a few ulp, where a logarithm of a ratio near 1
// carries an absolute one, so far blocks are also the more accurate ones.
//
// Far means S >= 4 len for every edge and every lane.  Then every vertex is at
// least 1.5 longest edges away, every face is seen under less than 0.23 sr
// (half the angle has a tangent below 0.12), and X = 2 len / S <= 1/2, inside
// the polynomials' ranges; the point is outside the element, so that the
// fourth solid angle is minus the sum of the other three and the tensor is
// traceless.  Against 64-bit sums the C-yoke's blocks carry 2.3e-15 of their
// norm (5.5e-15 by the general form), FP32 far blocks 5.4e-7 (8.0e-7).
#pragma once

#include "rh_math.hpp"

namespace rh {

// Record of a tetrahedron for the far form (built from its element record):
// vertices (12), W xx xy xz yy yz of the 6 edges (30), -2 (n_f n_f^T -
// n_3 n_3^T) xx xy xz yy yz of faces 0-2 (15), then the geometry that the
// integrals are formed from: 2 len (6), len^2 (6), 4 area n of faces 0-2 (9),
// and the same 21 values as floats for the FP32 integrals (whose vertex
// offsets and weighted sums stay in FP64), and n_3 (3).
constexpr int kFarW = 12, kFarT = 42, kFarG = 57;
constexpr int kFarGeo = 6 + 6 + 9;
constexpr int kFarG32 = kFarG + kFarGeo;                    // 78
constexpr int kFarN3 = kFarG32 + (kFarGeo + 1) / 2;         // 89
constexpr int kFarTet = kFarN3 + 3;                         // 92 doubles

#ifdef __HIPCC__
__device__ __forceinline__ void far_tet_record(const double* __restrict__ rec, double* __restrict__ o)
{
    for (int k = 0; k < 12; k++) o[k] = rec[k];
    double* g = o + kFarG;
    for (int e = 0; e < 6; e++) {
        const double* E = rec + 12 + kTetEdge * e;
        g[e] = 2.0 * E[3];
        // W is stored xx yy zz xy xz yz
        double* w = o + kFarW + 5 * e;
        w[0] = E[4];
        w[1] = E[7];
        w[2] = E[8];
        w[3] = E[5];
        w[4] = E[9];
        const double* a = rec + 3 * kTetEdgeA[e];
        const double* b = rec + 3 * kTetEdgeB[e];
        g[6 + e] = sq3(b[0] - a[0], b[1] - a[1], b[2] - a[2]);
    }
    const double* F = rec + 12 + 6 * kTetEdge;
    const double* n3 = F + 3 * kTetFaceRec;
    for (int f = 0; f < 3; f++) {
        const double* n = F + kTetFaceRec * f;
        for (int k = 0; k < 3; k++) g[12 + 3 * f + k] = 2.0 * n[3] * n[k];
        double* t = o + kFarT + 5 * f;
        t[0] = -2.0 * (n[0] * n[0] - n3[0] * n3[0]);
        t[1] = -2.0 * (n[0] * n[1] - n3[0] * n3[1]);
        t[2] = -2.0 * (n[0] * n[2] - n3[0] * n3[2]);
        t[3] = -2.0 * (n[1] * n[1] - n3[1] * n3[1]);
        t[4] = -2.0 * (n[1] * n[2] - n3[1] * n3[2]);
    }
    float* f = reinterpret_cast<float*>(o + kFarG32);
    for (int k = 0; k < kFarGeo; k++) f[k] = float(g[k]);
    f[kFarGeo] = 0.0f;
    for (int k = 0; k < 3; k++) o[kFarN3 + k] = n3[k];
}
template <class R>
__device__ __forceinline__ const R* far_geo(const double* __restrict__ rec)
{
    if constexpr (sizeof(R) == 4) return reinterpret_cast<const float*>(rec + kFarG32);
    else return rec + kFarG;
}

// 2 atanh(X/2) for X <= 1/2 and atan(t) for |t| <= tan(pi/16), no branches.
__device__ __forceinline__ double far_atanh2(double X)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double u = X * X;
    double p = d_edge2_p[7];
#pragma unroll
    for (int k = 6; k >= 0; k--) p = fma(p, u, d_edge2_p[k]);
    return fma(X * u, p, X);
#else
    return X;
#endif
}
__device__ __forceinline__ float far_atanh2(float X)
{
    // the degree-3 interpolant on X <= 1/2 (8e-10 relative)
    const float u = X * X;
    float p = fmaf(0.000481864669f, u, 0.00222449683f);
    p = fmaf(p, u, 0.0125003858f);
    p = fmaf(p, u, 0.0833333303f);
    return fmaf(X * u, p, X);
}
__device__ __forceinline__ double far_atan(double t)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double u = t * t;
    double p = d_atan16_p[6];
#pragma unroll
    for (int k = 5; k >= 0; k--) p = fma(p, u, d_atan16_p[k]);
    return fma(t * u, p, t);
#else
    return t;
#endif
}
__device__ __forceinline__ float far_atan(float t)
{
    const float u = t * t;
    const float p = fmaf(fmaf(-0.13649502f, u, 0.19990657f), u, -0.33333313f);
    return fmaf(t * u, p, t);
}
__device__ __forceinline__ float rh_div(float y, float d) { return y * rh_rcp(d); }

// Distances of the vertices of a far record from p and their pair sums;
// whether every lane of the wave is far.
template <class R>
struct FarTet {
    V3<R> r[4];
    R d[4], S[6];
};
template <class R>
__device__ __forceinline__ bool far_tet_open(const double* __restrict__ rec, const double p[3], FarTet<R>& t)
{
    const R* g = far_geo<R>(rec);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        t.r[k] = rel<R>(rec + 3 * k, p);
        t.d[k] = rh_sqrt(dot(t.r[k], t.r[k]));
    }
    bool far = true;
#pragma unroll
    for (int e = 0; e < 6; e++) {
        t.S[e] = t.d[kTetEdgeA[e]] + t.d[kTetEdgeB[e]];
        far &= (t.S[e] >= R(2) * g[e]);
    }
    return rh_all(far);
}

// q5 = acc / (4 pi), kept as products: what is formed from the entries (zz, in
// the layouts that store it) is then the same in every kernel, whatever the
// compiler would contract.
__device__ __forceinline__ void far_scale(const double (&acc)[5], double q5[5])
{
#pragma unroll
    for (int k = 0; k < 5; k++) {
        q5[k] = kInv4Pi * acc[k];
#ifdef __HIP_DEVICE_COMPILE__
        asm("" : "+v"(q5[k]));
#endif
    }
}

// The block's xx, xy, xz, yy, yz (zz = -(xx + yy)).
template <class R>
__device__ __forceinline__ void far_tet_block(const double* __restrict__ rec, const FarTet<R>& t, double q5[5])
{
    const R* g = far_geo<R>(rec);
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < 6; e++) {
        const double L = double(far_atanh2(rh_div(g[e], t.S[e])));
#pragma unroll
        for (int k = 0; k < 5; k++) acc[k] += L * rec[kFarW + 5 * e + k];
    }
    // edge of a vertex pair
    constexpr int kEdge[4][4] = {{-1, 0, 1, 2}, {0, -1, 3, 4}, {1, 3, -1, 5}, {2, 4, 5, -1}};
#pragma unroll
    for (int f = 0; f < 3; f++) {
        const int a = kTetFace[f][0], b = kTetFace[f][1], c = kTetFace[f][2];
        const int ab = kEdge[a][b], bc = kEdge[b][c], ca = kEdge[c][a];
        const R* n = g + 12 + 3 * f;
        const R im = dot(t.r[a], v3(n[0], n[1], n[2]));
        const R re = (t.S[ab] * t.S[bc]) * t.S[ca] - (t.d[c] * g[6 + ab] + t.d[b] * g[6 + ca] + t.d[a] * g[6 + bc]);
        const double om = double(far_atan(rh_div(im, re)));
#pragma unroll
        for (int k = 0; k < 5; k++) acc[k] += om * rec[kFarT + 5 * f + k];
    }
    far_scale(acc, q5);
}

// The same block for a wave that is not far from the tetrahedron (its own
// element among them): one edge and one face at a time, each with the tier its
// wave needs (edge_L2, rh_atan2_wave), so that it sets neither the kernel's
// registers nor, taken by 6 to 16 % of the waves, its time.  Returns whether
// the point is inside (zz is then -(xx + yy) - 1): the signs of the four plane
// distances, as in eval_tet.
template <class R>
__device__ __forceinline__ bool near_tet_block(const double* __restrict__ rec, const double p[3], double q5[5])
{
    const R* g = far_geo<R>(rec);
    auto vtx = [&](int k, V3<R>& r, R& d) {
        r = rel<R>(rec + 3 * k, p);
        d = rh_sqrt(dot(r, r));
    };
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int e = 0; e < 6; e++) {
        // edges (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
        const int a = (e < 3) ? 0 : (e < 5 ? 1 : 2), b = (e < 3) ? e + 1 : (e < 5 ? e - 1 : 3);
        V3<R> ra[1], rb[1];
        R da[1], db[1], S[1], L[1];
        vtx(a, ra[0], da[0]);
        vtx(b, rb[0], db[0]);
        S[0] = da[0] + db[0];
        edge_L2(ra, da, rb, db, S, g[e], kEdge6Top, L);
        for (int k = 0; k < 5; k++) acc[k] += double(L[0]) * rec[kFarW + 5 * e + k];
    }
    bool inside = true;
#pragma unroll 1
    for (int f = 0; f < 3; f++) {
        // faces (1,2,3) (0,3,2) (0,1,3): squared edges opposite a, b, c
        const int a = (f == 0) ? 1 : 0, b = (f == 0) ? 2 : (f == 1 ? 3 : 1), c = (f == 1) ? 2 : 3;
        const int ab = (f == 0) ? 3 : (f == 1 ? 2 : 0), bc = (f == 2) ? 4 : 5, ca = (f == 0) ? 4 : (f == 1 ? 1 : 2);
        V3<R> ra, rb, rc;
        R da, db, dc, om[1];
        vtx(a, ra, da);
        vtx(b, rb, db);
        vtx(c, rc, dc);
        const R* n = g + 12 + 3 * f;
        const R im[1] = {dot(ra, v3(n[0], n[1], n[2]))};
        const R re[1] = {((da + db) * (db + dc)) * (dc + da) - (dc * g[6 + ab] + db * g[6 + ca] + da * g[6 + bc])};
        inside = inside && (im[0] > R(0));
        rh_atan2_wave(im, re, kAtan32Top, om);
        for (int k = 0; k < 5; k++) acc[k] += double(om[0]) * rec[kFarT + 5 * f + k];
    }
    const double* n = rec + kFarN3;
    {
        const V3<R> r0 = rel<R>(rec, p);  // face 3 holds vertex 0
        inside = inside && (dot(r0, v3(R(n[0]), R(n[1]), R(n[2]))) > R(0));
    }
    // the solid angles sum to 4 pi inside: the fourth face's share of it
    const double in4 = inside ? 4.0 * kPi : 0.0;
    acc[0] -= in4 * n[0] * n[0];
    acc[1] -= in4 * n[0] * n[1];
    acc[2] -= in4 * n[0] * n[2];
    acc[3] -= in4 * n[1] * n[1];
    acc[4] -= in4 * n[1] * n[2];
    far_scale(acc, q5);
    return inside;
}

// Block (rectangular parallelepiped) at points whose eight corner distances
// are all at least twice the longest edge.  An off-diagonal entry is a signed
// sum of four edge integrals 2 atanh(len/S): pairs combine as
// atanh a - atanh b = atanh((a - b)/(1 - a b)), so that each entry takes one
// division and one short polynomial.  A face's two triangles have the same
// numerator z len len' (no cancellation) and the denominators above; the
// tangents of an axis' two faces combine as complex factors, and outside the
// block the third diagonal entry is minus the sum of the other two.  About
// 300 issue slots against 1,100 for the form that also holds at the block
// (eval_rec: cancellation-free ratios, octant-reduced arctangents): 10,000
// points of a line past 512 blocks 190 -> 104 us, the rest of it the waves that
// hold a near point; four copies each of 1,500 blocks assembled in mixed
// precision 260 -> 182 us with a 14th of the error (3.4e-6 -> 2.4e-7).
//
// A lane's far test depends on its own point only and far lanes always take
// this form, so a block does not depend on the lanes that share its wave.
//
// X, Y, Z: corner coordinates relative to the point, w: edge lengths.
template <class R>
__device__ __forceinline__ void far_rec_block(const R (&X)[2], const R (&Y)[2], const R (&Z)[2], const R (&D)[2][2][2],
                                              const R (&w)[3], double q6[6])
{
    // sums of end distances of the edges along x, y, z
    R Sx[2][2], Sy[2][2], Sz[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            Sx[i][j] = D[0][i][j] + D[1][i][j];
            Sy[i][j] = D[i][0][j] + D[i][1][j];
            Sz[i][j] = D[i][j][0] + D[i][j][1];
        }
    // sum of s_i s_j 2 atanh(len / S_ij), s_0 = -1, s_1 = +1
    auto edges = [](const R (&S)[2][2], R len) {
        const R l2 = len * len;
        const R nA = len * (S[0][1] - S[0][0]), dA = S[0][0] * S[0][1] - l2;
        const R nB = len * (S[1][1] - S[1][0]), dB = S[1][0] * S[1][1] - l2;
        return double(far_atanh2(rh_div(R(2) * (nA * dB - nB * dA), dA * dB - nA * nB)));
    };
    // half the solid angles of the two faces across axis `x`, corners (j, k):
    // height h, edge lengths a (along j) and b, distances d[j][k], edge sums
    // along j at k and along k at j.  The faces' outward normals are -x, +x.
    auto faces = [](const R (&h)[2], R a, R b, const R (&d)[2][2][2], const R (&Sj)[2][2], const R (&Sk)[2][2]) {
        R re[2], im[2];
        const R a2 = a * a, b2 = b * b, c2 = a2 + b2;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const R g = d[i][0][0] + d[i][1][1];  // ends of the shared diagonal
            // triangles (00, 10, 11) and (00, 01, 11)
            const R r1 = (Sj[i][0] * Sk[i][1]) * g - (d[i][1][1] * a2 + d[i][0][0] * b2 + d[i][1][0] * c2);
            const R r2 = (Sk[i][0] * Sj[i][1]) * g - (d[i][1][1] * b2 + d[i][0][0] * a2 + d[i][0][1] * c2);
            const R z = R(i ? 2 : -2) * h[i] * (a * b);
            re[i] = r1 * r2 - z * z;
            im[i] = z * (r1 + r2);
        }
        return double(far_atan(rh_div(re[0] * im[1] + im[0] * re[1], re[0] * re[1] - im[0] * im[1])));
    };
    const double om0 = faces(X, w[1], w[2], D, {{Sy[0][0], Sy[0][1]}, {Sy[1][0], Sy[1][1]}},
                             {{Sz[0][0], Sz[0][1]}, {Sz[1][0], Sz[1][1]}});
    R E[2][2][2];  // distances with y first: [j][i][k]
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++) E[j][i][k] = D[i][j][k];
    const double om1 = faces(Y, w[0], w[2], E, {{Sx[0][0], Sx[0][1]}, {Sx[1][0], Sx[1][1]}},
                             {{Sz[0][0], Sz[1][0]}, {Sz[0][1], Sz[1][1]}});
    double acc[5] = {-2.0 * om0, edges(Sz, w[2]), edges(Sy, w[1]), -2.0 * om1, edges(Sx, w[0])}, q5[5];
    far_scale(acc, q5);
    q6[0] = q5[0];
    q6[1] = q5[3];
    q6[2] = -(q5[0] + q5[3]);
    q6[3] = q5[1];
    q6[4] = q5[2];
    q6[5] = q5[4];
}

// Q of a block at p (element frame); returns whether p is inside.
template <class R>
__device__ __forceinline__ bool rec_block(const double* __restrict__ rec, const double p[3], double q6[6])
{
    const double c[3] = {rec[0] - p[0], rec[1] - p[1], rec[2] - p[2]};
    // FP32: lengths in units of a power of two near the distance (exact), since
    // the faces' factors are of the 12th degree in them
    double u = 1.0;
    if (sizeof(R) == 4) u = ldexp(1.0, -(__builtin_amdgcn_frexp_exp(sq3(c[0], c[1], c[2])) >> 1));
    R x[3][2], w[3], D[2][2][2];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        x[k][0] = R(u * (c[k] - rec[3 + k]));
        x[k][1] = R(u * (c[k] + rec[3 + k]));
        w[k] = R(2.0 * u * rec[3 + k]);
    }
    const R wm = fmax(fmax(w[0], w[1]), w[2]);
    R least = R(INFINITY);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                D[i][j][k] = rh_sqrt(x[0][i] * x[0][i] + x[1][j] * x[1][j] + x[2][k] * x[2][k]);
                least = fmin(least, D[i][j][k]);
            }
    const bool far = least >= R(2) * wm;
    bool in = false;
    if (rh_any(far)) far_rec_block(x[0], x[1], x[2], D, w, q6);
    if (rh_any(!far)) {
        double qn[6];
        in = eval_rec<R>(rec, p, qn) && !far;
#pragma unroll
        for (int k = 0; k < 6; k++) q6[k] = far ? q6[k] : qn[k];
    }
    return in;
}
#endif

}  // namespace rh
