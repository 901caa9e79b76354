// rh_far.hpp -- interaction blocks of elements that are far from every point
// of a wave, or from a lane's own point (blocks, hexahedra).
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
// Far means S >= 4 len for every edge and every lane.  The cosine between the
// directions of two vertices is then (R0^2 + R1^2 - len^2)/(2 R0 R1) >=
// 15/16 - 1/16 = 7/8.  All vertices lie within one half-space of directions, so
// that the point is outside the element, the fourth solid angle is minus the
// sum of the other three and the tensor is traceless.  A face's half angle has
// the tangent |u0 . (u1 x u2)| / (1 + u0.u1 + u1.u2 + u2.u0) of its vertices'
// directions u, at most sqrt(1 - 3 c^2 + 2 c^3) / (1 + 3 c) = 0.058 at c = 7/8
// (a face is seen under less than 0.115 sr), and X = 2 len / S <= 1/2: both
// inside the polynomials' ranges.  The two ends of the longest edge are at
// least 1.5 of it away, and any other vertex at least 1.2 (R2 >= 0.6 R0 by its
// own edge).  Against 64-bit sums the C-yoke's blocks carry 2.3e-15 of their
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

// Record of a hexahedron (a general polyhedron of six quadrilaterals) for the
// far form, its vertices renumbered to one topology: 0-3 around a face, 4 + i
// across from i.  Vertices (24), W xx xy xz yy yz of the 12 edges (60), 2 len
// (12), len^2 (12), -2 (n_f n_f^T - n_5 n_5^T) of faces 0-4 (25), for each of
// these n and four times the areas of its two triangles (25) and the squared
// diagonal between them (5), the squared limit distance and n_5.
constexpr int kHexW = 24, kHexL = 84, kHexL2 = 96, kHexT = 108, kHexF = 133, kHexD2 = 158, kHexR2 = 163, kHexN5 = 164,
              kHex = 168;

// vertex k of face f, edges' ends, edges and their order around a face
constexpr int kHexFace[6][4] = {{0, 1, 2, 3}, {0, 1, 5, 4}, {1, 2, 6, 5}, {2, 3, 7, 6}, {3, 0, 4, 7}, {4, 5, 6, 7}};
constexpr int kHexEdgeA[12] = {0, 1, 2, 3, 4, 5, 6, 7, 0, 1, 2, 3};
constexpr int kHexEdgeB[12] = {1, 2, 3, 0, 5, 6, 7, 4, 4, 5, 6, 7};
constexpr int kHexFaceEdge[5][4] = {{0, 1, 2, 3}, {0, 9, 4, 8}, {1, 10, 5, 9}, {2, 11, 6, 10}, {3, 8, 7, 11}};

// Its parts from an element record of 8 vertices, 12 edges, 6 faces and 24
// face corners; false if they are not a hexahedron's.
constexpr int kHexIn = kGenHdr + 24 + 12 * kGenEdge + 6 * kGenFace + 24;
constexpr int kHexInE = kGenHdr + 24, kHexInF = kHexInE + 12 * kGenEdge, kHexInV = kHexInF + 6 * kGenFace;
RH_FORM bool hex_vertices(const double* rec, int* id)
{
    const double *ed = rec + kHexInE, *fc = rec + kHexInF, *fv = rec + kHexInV;
    for (int f = 0; f < 6; f++)
        if (int(fc[kGenFace * f + 4]) != 4) return false;
    for (int i = 0; i < 4; i++) id[i] = int(fv[int(fc[3]) + i]);
    for (int i = 0; i < 4; i++) {
        id[4 + i] = -1;
        for (int e = 0; e < 12; e++) {
            const int a = int(ed[kGenEdge * e]), b = int(ed[kGenEdge * e + 1]);
            const int c = (a == id[i]) ? b : (b == id[i] ? a : -1);
            if (c >= 0 && c != id[0] && c != id[1] && c != id[2] && c != id[3]) id[4 + i] = c;
        }
        if (id[4 + i] < 0) return false;
    }
    return true;
}
RH_FORM bool hex_edge_record(const double* rec, const int* id, int e, double* o)
{
    const double *vt = rec + kGenHdr, *ed = rec + kHexInE;
    const int a = id[e < 8 ? e : e - 8], b = id[e < 8 ? (e & 4) + ((e + 1) & 3) : e - 4];
    int q = 0;
    for (; q < 12; q++) {
        const int c = int(ed[kGenEdge * q]), d = int(ed[kGenEdge * q + 1]);
        if ((c == a && d == b) || (c == b && d == a)) break;
    }
    if (q == 12) return false;
    const double* E = ed + kGenEdge * q;
    double* w = o + kHexW + 5 * e;  // stored xx yy zz xy xz yz
    w[0] = E[6];
    w[1] = E[9];
    w[2] = E[10];
    w[3] = E[7];
    w[4] = E[11];
    o[kHexL + e] = 2.0 * E[5];
    o[kHexL2 + e] = sq3(vt[3 * b] - vt[3 * a], vt[3 * b + 1] - vt[3 * a + 1], vt[3 * b + 2] - vt[3 * a + 2]);
    return true;
}
// the normal of face f in the order of kHexFace, null if it is no face
RH_FORM const double* hex_normal(const double* rec, const int* id, int f)
{
    const double *fc = rec + kHexInF, *fv = rec + kHexInV;
    const int i = f - 1, j = f & 3;
    unsigned want;
    if (f == 0 || f == 5) want = (1u << id[f ? 4 : 0]) | (1u << id[f ? 5 : 1]) | (1u << id[f ? 6 : 2]) | (1u << id[f ? 7 : 3]);
    else want = (1u << id[i]) | (1u << id[j]) | (1u << id[4 + i]) | (1u << id[4 + j]);
    for (int q = 0; q < 6; q++) {
        unsigned got = 0;
        for (int k = 0; k < 4; k++) got |= 1u << int(fv[int(fc[kGenFace * q + 3]) + k]);
        if (got == want) return fc + kGenFace * q;
    }
    return nullptr;
}
RH_FORM bool hex_face_record(const double* rec, const int* id, int f, double* o)
{
    const double* vt = rec + kGenHdr;
    const double *n = hex_normal(rec, id, f), *m = hex_normal(rec, id, 5);
    if (!n || !m) return false;
    double* t = o + kHexT + 5 * f;
    t[0] = -2.0 * (n[0] * n[0] - m[0] * m[0]);
    t[1] = -2.0 * (n[0] * n[1] - m[0] * m[1]);
    t[2] = -2.0 * (n[0] * n[2] - m[0] * m[2]);
    t[3] = -2.0 * (n[1] * n[1] - m[1] * m[1]);
    t[4] = -2.0 * (n[1] * n[2] - m[1] * m[2]);
    const int i = f - 1, j = f & 3;
    const double* a = vt + 3 * id[f == 0 ? 0 : i];
    auto side = [&](int k) { return v3(vt[3 * k] - a[0], vt[3 * k + 1] - a[1], vt[3 * k + 2] - a[2]); };
    const V3<double> e1 = side(id[f == 0 ? 1 : j]), e2 = side(id[f == 0 ? 2 : 4 + j]), e3 = side(id[f == 0 ? 3 : 4 + i]);
    const V3<double> c1 = cross(e1, e2), c2 = cross(e2, e3);
    double* g = o + kHexF + 5 * f;
    for (int c = 0; c < 3; c++) g[c] = n[c];
    g[3] = 2.0 * sqrt(dot(c1, c1));
    g[4] = 2.0 * sqrt(dot(c2, c2));
    o[kHexD2 + f] = dot(e2, e2);
    return true;
}
RH_FORM void hex_close_record(const double* rec, const int* id, double* o)
{
    for (int k = 0; k < 8; k++)
        for (int c = 0; c < 3; c++) o[3 * k + c] = rec[kGenHdr + 3 * id[k] + c];
    double l2 = 0.0;
    for (int e = 0; e < 12; e++) l2 = fmax(l2, o[kHexL2 + e]);
    o[kHexR2] = 4.0 * l2;
    const double* n = hex_normal(rec, id, 5);
    for (int c = 0; c < 3; c++) o[kHexN5 + c] = n[c];
    o[kHex - 1] = 0.0;
}

RH_FORM void far_tet_record(const double* __restrict__ rec, double* __restrict__ o)
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
RH_FORM const R* far_geo(const double* __restrict__ rec)
{
    if constexpr (sizeof(R) == 4) return reinterpret_cast<const float*>(rec + kFarG32);
    else return rec + kFarG;
}

// 2 atanh(X/2) for X <= 1/2 and atan(t) for |t| <= tan(pi/16), no branches.
RH_FORM double far_atanh2(double X)
{
    const double u = X * X;
    double p = d_edge2_p[7];
#pragma unroll
    for (int k = 6; k >= 0; k--) p = fma(p, u, d_edge2_p[k]);
    return fma(X * u, p, X);
}
RH_FORM float far_atanh2(float X)
{
    // the degree-3 interpolant on X <= 1/2 (8e-10 relative)
    const float u = X * X;
    float p = fmaf(0.000481864669f, u, 0.00222449683f);
    p = fmaf(p, u, 0.0125003858f);
    p = fmaf(p, u, 0.0833333303f);
    return fmaf(X * u, p, X);
}
RH_FORM double far_atan(double t)
{
    const double u = t * t;
    double p = d_atan16_p[6];
#pragma unroll
    for (int k = 5; k >= 0; k--) p = fma(p, u, d_atan16_p[k]);
    return fma(t * u, p, t);
}
RH_FORM float far_atan(float t)
{
    const float u = t * t;
    const float p = fmaf(fmaf(-0.13649502f, u, 0.19990657f), u, -0.33333313f);
    return fmaf(t * u, p, t);
}
RH_FORM float rh_div(float y, float d) { return y * rh_rcp(d); }

// Distances of the vertices of a far record from p and their pair sums;
// whether every lane of the wave is far.
template <class R>
struct FarTet {
    V3<R> r[4];
    R d[4], S[6];
};
template <class R>
RH_FORM bool far_tet_open(const double* __restrict__ rec, const double p[3], FarTet<R>& t)
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
RH_FORM void far_scale(const double (&acc)[5], double q5[5])
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
RH_FORM void far_tet_block(const double* __restrict__ rec, const FarTet<R>& t, double q5[5])
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
RH_FORM bool near_tet_block(const double* __restrict__ rec, const double p[3], double q5[5])
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
        // faces (1,2,3) (0,3,2) (0,1,3)
        const int a = (f == 0) ? 1 : 0, b = (f == 0) ? 2 : (f == 1 ? 3 : 1), c = (f == 1) ? 2 : 3;
        V3<R> ra, rb, rc;
        R da, db, dc, om[1];
        vtx(a, ra, da);
        vtx(b, rb, db);
        vtx(c, rc, dc);
        const R* n = g + 12 + 3 * f;
        const R im[1] = {dot(ra, v3(n[0], n[1], n[2]))};
        const R re[1] = {tri_re2(ra, da, rb, db, rc, dc)};
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
RH_FORM void far_rec_block(const R (&X)[2], const R (&Y)[2], const R (&Z)[2], const R (&D)[2][2][2],
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
RH_FORM bool rec_block(const double* __restrict__ rec, const double p[3], double q6[6])
{
    const double c[3] = {rec[0] - p[0], rec[1] - p[1], rec[2] - p[2]};
    // FP32: lengths in units of a power of two near the distance (exact), since
    // the faces' factors are of the 12th degree in them
    double u = 1.0;
    if (sizeof(R) == 4) {
        double mant;
        int ex;
        rh_frexp(sq3(c[0], c[1], c[2]), mant, ex);
        u = ldexp(1.0, -(ex >> 1));
    }
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

// Keeps a record's reads from being hoisted past here: in one block of code the
// scheduler would load all 164 values first, into registers that it then spills.
#ifdef __HIP_DEVICE_COMPILE__
#define FAR_GROUP()                   \
    do {                              \
        asm volatile("" ::: "memory"); \
        __builtin_amdgcn_sched_barrier(0); \
    } while (0)
#else
#define FAR_GROUP()
#endif

// The block at points near a hexahedron: one edge and one face at a time from
// the record, each with the tier its wave needs, as near_tet_block.  All six
// solid angles are formed, from the corners' triple products (which keep their
// digits next to a corner, where a plane distance times the area does not), and
// half[0] is their sum, halved: 2 pi inside, 0 outside.  At a point on a face
// that face's angle is one of its two limits, by the sign of a rounded or a
// zero triple product, and the others stand; five angles closed by the plane
// tests' answer were off by 4 pi there.
RH_FORM bool near_hex_block(const double* __restrict__ h, const double p[3], double q5[5], double half[1])
{
    auto vtx = [&](int k, V3<double>& r, double& d) {
        r = rel<double>(h + 3 * k, p);
        d = rh_sqrt(dot(r, r));
    };
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int e = 0; e < 12; e++) {
        const int a = e & 7, top = e & 4;
        const int b = (e < 8) ? top + ((e + 1) & 3) : e - 4;
        V3<double> ra[1], rb[1];
        double da[1], db[1], S[1], L[1];
        vtx(e < 8 ? a : e - 8, ra[0], da[0]);
        vtx(b, rb[0], db[0]);
        S[0] = da[0] + db[0];
        edge_L2(ra, da, rb, db, S, h[kHexL + e], kEdge6Top, L);
        for (int k = 0; k < 5; k++) acc[k] += L[0] * h[kHexW + 5 * e + k];
    }
    bool inside = true;
    const double* n5 = h + kHexN5;
    half[0] = 0.0;
#pragma unroll 1
    for (int f = 0; f < 6; f++) {
        // corners as in kHexFace: outward for face 0, inward for the others
        const int i = f - 1, j = f & 3;
        const int a = (f == 0) ? 0 : (f == 5 ? 4 : i), b = (f == 0) ? 1 : (f == 5 ? 5 : j);
        const int c = (f == 0) ? 2 : (f == 5 ? 6 : 4 + j), e = (f == 0) ? 3 : (f == 5 ? 7 : 4 + i);
        V3<double> ra, rb, rc, re;
        double da, db, dc, de, om[1], i1, r1, i2, r2;
        vtx(a, ra, da);
        vtx(b, rb, db);
        vtx(c, rc, dc);
        vtx(e, re, de);
        const double* n = (f == 5) ? n5 : h + kHexF + 5 * f;
        inside = inside && (dot(ra, v3(n[0], n[1], n[2])) > 0.0);
        tri_factor(ra, da, rb, db, rc, dc, r1, i1);
        tri_factor(ra, da, rc, dc, re, de, r2, i2);
        const double s = (f == 0) ? 1.0 : -1.0;
        const double im[1] = {s * (r1 * i2 + r2 * i1)}, rr[1] = {r1 * r2 - i1 * i2};
        rh_atan2_wave(im, rr, kAtan32Top, om);
        half[0] += om[0];
        if (f == 5) break;
        for (int k = 0; k < 5; k++) acc[k] += om[0] * h[kHexT + 5 * f + k];
    }
    // the records' weights are the faces' less the sixth's
    const double w = 2.0 * half[0];
    acc[0] -= w * n5[0] * n5[0];
    acc[1] -= w * n5[0] * n5[1];
    acc[2] -= w * n5[0] * n5[2];
    acc[3] -= w * n5[1] * n5[1];
    acc[4] -= w * n5[1] * n5[2];
    far_scale(acc, q5);
    return inside;
}

// General polyhedron at p (element frame); h: its hexahedron record, null if it
// is none (then by eval_gen).  Points whose distances from all corners are at
// least two longest edges take the far form: 8 offsets and roots, 12 short edge
// integrals, and for each of five faces two triangle denominators and one short
// arctangent, about 600 issue slots against 3,000 for eval_gen, which forms
// both ends of every edge and every face's corners anew and reads its record
// through chains of scalar loads (36,000 cycles where few waves hide them).
// The far test is each lane's own, as for blocks.
RH_FORM bool gen_block(const double* __restrict__ h, const double* __restrict__ rec,
                                          const double p[3], double q6[6])
{
    if (!h) return eval_gen<double>(rec, p, q6);
    V3<double> r[8];
    double d[8], least = INFINITY;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        r[k] = rel<double>(h + 3 * k, p);
        const double d2 = dot(r[k], r[k]);
        least = fmin(least, d2);
        d[k] = rh_sqrt(d2);
    }
    const bool far = least >= h[kHexR2];
    FAR_GROUP();
    double q5[5];
    if (rh_any(far)) {
        double S[12], acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int e = 0; e < 12; e++) {
            S[e] = d[kHexEdgeA[e]] + d[kHexEdgeB[e]];
            const double L = far_atanh2(rh_div(h[kHexL + e], S[e]));
#pragma unroll
            for (int k = 0; k < 5; k++) acc[k] += L * h[kHexW + 5 * e + k];
            if ((e & 1) == 1) FAR_GROUP();
        }
#pragma unroll
        for (int f = 0; f < 5; f++) {
            const int a = kHexFace[f][0], b = kHexFace[f][1], c = kHexFace[f][2], e = kHexFace[f][3];
            const int ab = kHexFaceEdge[f][0], bc = kHexFaceEdge[f][1], ce = kHexFaceEdge[f][2], ea = kHexFaceEdge[f][3];
            const double* g = h + kHexF + 5 * f;
            const double D = d[a] + d[c], D2 = h[kHexD2 + f], z = dot(r[a], v3(g[0], g[1], g[2]));
            const double r1 = (S[ab] * S[bc]) * D - (d[c] * h[kHexL2 + ab] + d[b] * D2 + d[a] * h[kHexL2 + bc]);
            const double r2 = (S[ea] * S[ce]) * D - (d[a] * h[kHexL2 + ce] + d[e] * D2 + d[c] * h[kHexL2 + ea]);
            const double i1 = z * g[3], i2 = z * g[4];
            const double om = far_atan(rh_div(r1 * i2 + r2 * i1, r1 * r2 - i1 * i2));
#pragma unroll
            for (int k = 0; k < 5; k++) acc[k] += om * h[kHexT + 5 * f + k];
            FAR_GROUP();
        }
        far_scale(acc, q5);
    }
    double half = 0.0;  // the solid angles' sum, halved
    bool in = false;
    if (rh_any(!far)) {
        double qn[5], hn[1];
        in = near_hex_block(h, p, qn, hn) && !far;
        half = far ? 0.0 : hn[0];
#pragma unroll
        for (int k = 0; k < 5; k++) q5[k] = far ? q5[k] : qn[k];
    }
    q6[0] = q5[0];
    q6[1] = q5[3];
    q6[2] = -(q5[0] + q5[3]) - 2.0 * kInv4Pi * half;
    q6[3] = q5[1];
    q6[4] = q5[2];
    q6[5] = q5[4];
    return in;
}

}  // namespace rh
