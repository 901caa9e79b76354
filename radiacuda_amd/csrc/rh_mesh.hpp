// rh_mesh.hpp -- field of a conforming polyhedral mesh as line terms on its
// unique edges and charge sheets on its unique faces.
//
// Summed over the elements of a mesh, the per-element form
//     4 pi H = sum_e L_e W_e M - sum_f Omega_f (n_f . M) n_f
// regroups by mesh entity.  L_e depends only on the edge and the point, so
// every edge is evaluated once with the net weight w_e = sum_{elements at e}
// W_{e,j} M_j.  A face shared by two elements appears with opposite outward
// normals and opposite signed solid angles, so it is evaluated once with the
// net charge g_f = n_f sum_j s_j (n_f . M_j), s_j = +-1 the orientation of
// element j's copy of the face.  The sum is the same; on the C-yoke mesh the
// work per tetrahedron drops from 6 logs and 3 atan2 to about 1.4 and 2.2.
// B = H + M of the element containing the point, found by plane tests.
#pragma once

#include "rh_math.hpp"

namespace rh {

// Charged edge record: a(3), b(3), t(3), 2 len, w(3), 0 (edge_flag, an array
// beside the records, tells whether a is the previous record's b).  The FP32 sweep's records hold 2 len and the near
// distance as floats in slot 6 (the near pass reads slot 9).
constexpr int kMeshEdge = 14;
// Charged face record: v0..v3 (12), n(3), 4*area(v0,v1,v2), 4*area(v0,v2,v3),
// nv, -2 g(3), 0 (face_flag tells the owned sides and whether a triangle's v0,
// v1 are the previous record's v1, v2, or a quadrilateral's the previous
// record's v2, v3), then the edges the face owns: for the sides
// (v0,v1), (v1,v2), (v2,v0) of a triangle or (v0,v1), (v1,v2), (v2,v3) of a
// quadrilateral in turn 2 len and w(3) (slots 22-33); slot 35: the FP32
// sweep's near distance (a float); slots 36-40: the squared distances of
// (v0,v1), (v1,v2), (v0,v2), (v2,v3), (v0,v3) (the last two of
// quadrilaterals; FP32 records: five floats from slot 36).  A face's vertices
// may come in either direction of its loop: its solid angle below takes the
// fan triangles' triple products from n and their areas, not from the order.
// Constant factors are charged into the records, so that the sweep spends no
// instruction on them: lengths are doubled (edge_L2), the charge is -2 g
// (the sweep adds half the solid angle), and a triangle's n is scaled by
// 4*area.  (The host build's mesh_edge_L and mesh_face_omega read records
// with plain len, n, 2*area and g.)
constexpr int kMeshFace = 42;
constexpr int kMeshFaceEdges = 22;
constexpr int kMeshFaceLen2 = 36;
// Inside-test record: nplanes, M(3), up to 8 planes (n(3), d) with outward n:
// inside iff n.p < d for every plane.
constexpr int kMeshPlanes = 8;
constexpr int kMeshIn = 4 + 4 * kMeshPlanes;  // 36
// Geometry-only sizes (host arrays the charged records are built from).
constexpr int kMeshEdgeGeo = 10;  // a, b, t, len
constexpr int kMeshFaceGeo = 18;  // v0..v3, n, a1, a2, nv

// L_e of one charged edge at p.
template <class R>
RH_HD double mesh_edge_L(const double* __restrict__ rec, const double p[3])
{
    const V3<R> ra = rel<R>(rec, p), rb = rel<R>(rec + 3, p);
    const R Ra = rh_sqrt(dot(ra, ra)), Rb = rh_sqrt(dot(rb, rb));
    return double(edge_L(ra, Ra, rb, Rb, R(rec[9])));
}

// Signed solid angle of one charged face at p: the fan triangles (v0,v1,v2)
// and (v0,v2,v3) multiplied as complex numbers, one atan2 per face.
template <class R>
RH_HD double mesh_face_omega(const double* __restrict__ rec, const double p[3])
{
    const V3<R> r0 = rel<R>(rec, p), r1 = rel<R>(rec + 3, p), r2 = rel<R>(rec + 6, p);
    const R R0 = rh_sqrt(dot(r0, r0)), R1 = rh_sqrt(dot(r1, r1)), R2 = rh_sqrt(dot(r2, r2));
    const V3<R> n = v3(R(rec[12]), R(rec[13]), R(rec[14]));
    const R h = dot(r0, n);  // r0 . n, the same for every fan triangle
    R im = R(rec[15]) * h;
    R re = R0 * R1 * R2 + dot(r0, r1) * R2 + dot(r0, r2) * R1 + dot(r1, r2) * R0;
    if (rec[17] > 3.5) {
        const V3<R> r3 = rel<R>(rec + 9, p);
        const R R3 = rh_sqrt(dot(r3, r3));
        const R im2 = R(rec[16]) * h;
        const R re2 = R0 * R2 * R3 + dot(r0, r2) * R3 + dot(r0, r3) * R2 + dot(r2, r3) * R0;
        const R pr = re * re2 - im * im2;
        const R pi = re * im2 + im * re2;
        re = pr;
        im = pi;
    }
    return 2.0 * double(rh_atan2_wave(im, re));
}

#ifdef __HIPCC__
// What the sweep has to know of a record before it reads the record itself is
// read through the scalar cache (the address is the same in every lane), so
// that its branches wait for no vector instruction.
typedef const __attribute__((address_space(4))) int* MeshFlags;
__device__ __forceinline__ MeshFlags mesh_flags(const int32_t* p) { return (MeshFlags)(uintptr_t)p; }
#endif
// Flags of a face or edge record: bits 0-2 the sides a face owns, bit 3 the
// record continues the previous one (faces: code 1 or 3).
constexpr int kMeshCont = 8;

// A vertex relative to the observation point and its distance.
template <class R>
struct MeshVtx {
    V3<R> r;
    R d;
};
template <class R>
RH_HD MeshVtx<R> mesh_vtx(const double* __restrict__ v, const double p[3])
{
    const V3<R> r = rel<R>(v, p);
    return MeshVtx<R>{r, rh_sqrt(dot(r, r))};
}
// The same for the N points of a lane.
template <class R, int N>
struct MeshVtxN {
    V3<R> r[N];
    R d[N];
};

// FP32 sweep records: the geometry the lanes use in FP32 is stored as floats
// when the records are charged (edge slot 6: 2 len, near distance; face slots
// 12-14: n(3), the two doubled areas), so the sweep converts none of it per
// record; vertices (offsets are formed in FP64) and the weights w and g (the
// sums are accumulated in FP64) stay FP64.
template <class R>
struct MeshGeo {
    R n0, n1, n2, a1, a2, l01, l12, l02, l23, l03;
};
template <class R>
RH_FORM MeshGeo<R> mesh_geo(const double* __restrict__ rec)
{
    if constexpr (sizeof(R) == 4) {
        const float* f = reinterpret_cast<const float*>(rec + 12);
        const float* l = reinterpret_cast<const float*>(rec + kMeshFaceLen2);
        return MeshGeo<R>{f[0], f[1], f[2], f[3], f[4], l[0], l[1], l[2], l[3], l[4]};
    } else {
        const double* l = rec + kMeshFaceLen2;
        return MeshGeo<R>{rec[12], rec[13], rec[14], rec[15], rec[16], l[0], l[1], l[2], l[3], l[4]};
    }
}

template <class R, int N>
RH_FORM void mesh_vtx(const double* __restrict__ v, const double (&p)[N][3], MeshVtxN<R, N>& o)
{
#pragma unroll
    for (int i = 0; i < N; i++) {
        o.r[i] = rel<R>(v, p[i]);
        o.d[i] = rh_sqrt(dot(o.r[i], o.r[i]));
    }
}
// S = Ra + Rb
template <class R, int N>
RH_FORM void mesh_sum(const MeshVtxN<R, N>& a, const MeshVtxN<R, N>& b, R (&o)[N])
{
#pragma unroll
    for (int i = 0; i < N; i++) o[i] = a.d[i] + b.d[i];
}

// Half the signed solid angle of a charged triangle from the offset of its
// first vertex, the distances and their sums.  The formula of Van Oosterom and
// Strackee, tan(Omega/2) = r0 . (r1 x r2) / (R0 R1 R2 + (r0.r1) R2 + (r2.r0) R1
// + (r1.r2) R0), with r_i . r_j = (R_i^2 + R_j^2 - l_ij^2) / 2: the denominator
// is ((R0+R1)(R1+R2)(R2+R0) - R2 l01^2 - R1 l02^2 - R0 l12^2) / 2: no dot
// product is formed, and the sums are those that the edges' integrals divide
// by.  Next to a vertex the difference cancels.  FP64: a wave whose points all
// have |im| < re / 32, the shortest arctangent's range, and a subtracted part t
// below re (from about one edge away; the angle then carries less than a unit
// of 1.1e-16, absolute) takes it, by one vote 32 |im| + t < re that costs what
// the range alone would; any other wave forms the dot products (tri_re2), which
// keep their digits next to the vertices too.  On the C-yoke 2.3 % of the
// waves' triangles do.  FP32: the near test (mesh32_near) keeps the points off
// the vertices.
template <class R, int N>
RH_FORM void mesh_tri_half_omega(const MeshVtxN<R, N>& a, const MeshVtxN<R, N>& b,
                                                    const MeshVtxN<R, N>& c, const R (&sab)[N], const R (&sbc)[N],
                                                    const R (&sca)[N], const double* __restrict__ rec, double top_c,
                                                    R (&om)[N])
{
    const MeshGeo<R> g = mesh_geo<R>(rec);
    R im[N], re[N];
    bool far = true;
#pragma unroll
    for (int i = 0; i < N; i++) {
        im[i] = dot(a.r[i], v3(g.n0, g.n1, g.n2));
        const R t = c.d[i] * g.l01 + b.d[i] * g.l02 + a.d[i] * g.l12;
        re[i] = (sab[i] * sbc[i]) * sca[i] - t;
        if constexpr (sizeof(R) == 8) far = far && fma(32.0, fabs(im[i]), t) < re[i];
    }
    if constexpr (sizeof(R) == 8) {
        if (rh_all(far)) {
            rh_atan32(im, re, top_c, om);
            return;
        }
        RH_KEEP_BRANCH();
#pragma unroll
        for (int i = 0; i < N; i++) re[i] = tri_re2(a.r[i], a.d[i], b.r[i], b.d[i], c.r[i], c.d[i]);
        rh_atan2_rest(im, re, om);
    } else {
        rh_atan2_wave(im, re, top_c, om);
    }
}

// FP64 half solid angle of a face of an FP32 sweep record, whose normal and
// areas are stored as floats: the fan triangles' triple products r0 . (r1 x r2)
// are taken as r0 . ((v1 - v0) x (v2 - v0)) from the FP64 vertices, signed by
// the stored normal (the same quantity as area * (r0 . n) of the FP64 sweep).
RH_HD double mesh_face_half_omega_near(const double* __restrict__ rec, const double p[3])
{
    const float* f = reinterpret_cast<const float*>(rec + 12);
    const V3<double> e1 = v3(rec[3] - rec[0], rec[4] - rec[1], rec[5] - rec[2]);
    const V3<double> e2 = v3(rec[6] - rec[0], rec[7] - rec[1], rec[8] - rec[2]);
    const V3<double> c1 = cross(e1, e2);
    const double sg = (c1.x * f[0] + c1.y * f[1] + c1.z * f[2] >= 0.0) ? 1.0 : -1.0;
    const V3<double> r0 = rel<double>(rec, p), r1 = rel<double>(rec + 3, p), r2 = rel<double>(rec + 6, p);
    const double R0 = rh_sqrt(dot(r0, r0)), R1 = rh_sqrt(dot(r1, r1)), R2 = rh_sqrt(dot(r2, r2));
    double im = sg * dot(r0, c1);
    double re = R0 * R1 * R2 + dot(r0, r1) * R2 + dot(r0, r2) * R1 + dot(r1, r2) * R0;
    if (rec[17] > 3.5) {
        const V3<double> r3 = rel<double>(rec + 9, p);
        const double R3 = rh_sqrt(dot(r3, r3));
        const V3<double> c2 = cross(e2, v3(rec[9] - rec[0], rec[10] - rec[1], rec[11] - rec[2]));
        const double im2 = sg * dot(r0, c2);
        const double re2 = R0 * R2 * R3 + dot(r0, r2) * R3 + dot(r0, r3) * R2 + dot(r2, r3) * R0;
        const double pr = re * re2 - im * im2;
        const double pi = re * im2 + im * re2;
        re = pr;
        im = pi;
    }
    return rh_atan2_wave(im, re);
}

// Near test of the FP32 mesh sweep: FP32 offsets carry eps32 of the distance,
// so a term's relative error grows like eps32 * size / distance.  A wave with
// a point within kNear32 entity sizes of a vertex (faces: the longest side;
// edges: the length) evaluates that entity in FP64.  thr: kNear32 sizes, as
// the record carries it (faces: slot 35, edges: slot 6, second float).
RH_HD bool mesh32_near(float dmin, float thr)
{
    return rh_any(dmin < thr);
}

// L_e of an FP32 sweep edge record in FP64 (vertices in slots 0-5, twice the
// FP64 length in slot 9).
RH_HD double mesh_edge_L_near(const double* __restrict__ rec, const double p[3])
{
    const MeshVtx<double> a = mesh_vtx<double>(rec, p), b = mesh_vtx<double>(rec + 3, p);
    return edge_L(a.r, a.d, b.r, b.d, 0.5 * rec[9]);
}

// A face of an FP32 sweep record in FP64 (triangle or quadrilateral): half its
// solid angle and the sum of L_e w_e over the sides it owns.
struct MeshFace64 {
    double om, h0, h1, h2;
};
RH_HD MeshFace64 mesh_face_near(const double* __restrict__ rec, int mask, const double p[3])
{
    const int nv = rec[17] > 3.5 ? 4 : 3;
    MeshFace64 t{mesh_face_half_omega_near(rec, p), 0.0, 0.0, 0.0};
    for (int k = 0; k < 3; k++) {
        if (!(mask & (1 << k))) continue;
        const double* e = rec + kMeshFaceEdges + 4 * k;
        const int k1 = (k + 1 == nv) ? 0 : k + 1;
        const MeshVtx<double> a = mesh_vtx<double>(rec + 3 * k, p), b = mesh_vtx<double>(rec + 3 * k1, p);
        const double L = edge_L(a.r, a.d, b.r, b.d, dot(a.r, b.r), 0.5 * e[0]);
        t.h0 += L * e[1];
        t.h1 += L * e[2];
        t.h2 += L * e[3];
    }
    return t;
}

// Half the signed solid angle of a quadrilateral record, likewise: the fans
// (v0,v1,v2) and (v0,v2,v3) multiplied as complex numbers.
template <class R, int N>
RH_FORM void mesh_quad_half_omega(const MeshVtxN<R, N>& a, const MeshVtxN<R, N>& b,
                                                     const MeshVtxN<R, N>& c, const MeshVtxN<R, N>& d,
                                                     const R (&sab)[N], const R (&sbc)[N], const R (&scd)[N],
                                                     const double* __restrict__ rec, double top_c, R (&om)[N])
{
    const MeshGeo<R> g = mesh_geo<R>(rec);
    R im[N], re[N];
    bool far = true;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const R h = dot(a.r[i], v3(g.n0, g.n1, g.n2));
        const R i1 = g.a1 * h, i2 = g.a2 * h;
        const R sac = a.d[i] + c.d[i], sad = a.d[i] + d.d[i];
        const R t1 = c.d[i] * g.l01 + b.d[i] * g.l02 + a.d[i] * g.l12;
        const R t2 = d.d[i] * g.l02 + c.d[i] * g.l03 + a.d[i] * g.l23;
        const R r1 = (sab[i] * sbc[i]) * sac - t1;
        const R r2 = (sac * scd[i]) * sad - t2;
        im[i] = r1 * i2 + i1 * r2;
        re[i] = r1 * r2 - i1 * i2;
        if constexpr (sizeof(R) == 8) far = far && fabs(im[i]) < 0.03125 * re[i] && t1 <= r1 && t2 <= r2;
    }
    if constexpr (sizeof(R) == 8) {
        if (rh_all(far)) {
            rh_atan32(im, re, top_c, om);
            return;
        }
        RH_KEEP_BRANCH();
#pragma unroll
        for (int i = 0; i < N; i++) {
            const R h = dot(a.r[i], v3(g.n0, g.n1, g.n2));
            const R i1 = g.a1 * h, i2 = g.a2 * h;
            const R r1 = tri_re2(a.r[i], a.d[i], b.r[i], b.d[i], c.r[i], c.d[i]);
            const R r2 = tri_re2(a.r[i], a.d[i], c.r[i], c.d[i], d.r[i], d.d[i]);
            im[i] = r1 * i2 + i1 * r2;
            re[i] = r1 * r2 - i1 * i2;
        }
        rh_atan2_rest(im, re, om);
    } else {
        rh_atan2_wave(im, re, top_c, om);
    }
}

// Charged record of an edge with net weight w from its geometry, and of a face
// with net charge s whose sides are the edges face_edge[k] (-1: not owned) of
// the geometry edge_geo and the charged records ch_edge; pack32: for the FP32
// sweep.
RH_HD void mesh_charge_edge(const double* __restrict__ g, const double w[3], bool pack32, double* __restrict__ o)
{
    for (int k = 0; k < kMeshEdgeGeo - 1; k++) o[k] = g[k];
    o[9] = 2.0 * g[9];
    o[10] = w[0];
    o[11] = w[1];
    o[12] = w[2];
    o[13] = 0.0;
    if (pack32) {
        // slot 6: 2 len and the near distance of the FP32 sweep (kNear32 lengths)
        float* f = reinterpret_cast<float*>(o + 6);
        const float len = float(g[9]);
        f[0] = 2.0f * len;
        f[1] = kNear32 * len;
    }
}
RH_HD void mesh_charge_face(const double* __restrict__ g, double s, const int64_t* __restrict__ face_edge,
                            const double* __restrict__ edge_geo, const double* __restrict__ ch_edge, bool pack32,
                            double* __restrict__ o)
{
    const double n0 = g[12], n1 = g[13], n2 = g[14];
    const bool tri = !(g[17] > 3.5);
    const double a1 = g[15], a2 = g[16];
    const double nk = tri ? 2.0 * a1 : 1.0;  // triangles: n scaled by four times the area
    for (int k = 0; k < 12; k++) o[k] = g[k];
    o[12] = nk * n0;
    o[13] = nk * n1;
    o[14] = nk * n2;
    o[15] = 2.0 * a1;
    o[16] = 2.0 * a2;
    o[17] = g[17];
    // squared distances of (v0,v1), (v1,v2), (v0,v2), (v2,v3), (v0,v3)
    const int pa[5] = {0, 1, 0, 2, 0}, pb[5] = {1, 2, 2, 3, 3};
    double l2[5];
    for (int k = 0; k < 5; k++) {
        const double* u = g + 3 * pa[k];
        const double* v = g + 3 * pb[k];
        l2[k] = (tri && k > 2) ? 0.0 : sq3(v[0] - u[0], v[1] - u[1], v[2] - u[2]);
        o[kMeshFaceLen2 + k] = l2[k];
    }
    o[kMeshFaceLen2 + 5] = 0.0;
    o[18] = -2.0 * (s * n0);
    o[19] = -2.0 * (s * n1);
    o[20] = -2.0 * (s * n2);
    o[21] = 0.0;
    // owned edges: twice the length and the net weight of the charged edge record
    for (int k = 0; k < 3; k++) {
        const int64_t e = face_edge[k];
        double* d = o + kMeshFaceEdges + 4 * k;
        if (e >= 0) {
            const double* ce = ch_edge + kMeshEdge * e;
            d[0] = 2.0 * edge_geo[kMeshEdgeGeo * e + 9];
            d[1] = ce[10];
            d[2] = ce[11];
            d[3] = ce[12];
        } else {
            d[0] = d[1] = d[2] = d[3] = 0.0;
        }
    }
    o[kMeshFaceEdges + 12] = 0.0;
    o[kMeshFaceEdges + 13] = 0.0;
    if (pack32) {
        // slot 35: the near distance of the FP32 sweep (kNear32 longest sides)
        const int nv = tri ? 3 : 4;
        double lmax = 0.0;
        for (int k = 0; k < nv; k++) {
            const double* a = g + 3 * k;
            const double* b = g + 3 * ((k + 1) % nv);
            const double d0 = b[0] - a[0], d1 = b[1] - a[1], d2 = b[2] - a[2];
            lmax = fmax(lmax, sqrt(d0 * d0 + d1 * d1 + d2 * d2));
        }
        reinterpret_cast<float*>(o + kMeshFaceEdges + 13)[0] = float(double(kNear32) * lmax);
    }
    if (pack32) {
        float* f = reinterpret_cast<float*>(o + 12);
        f[0] = float(nk * n0);
        f[1] = float(nk * n1);
        f[2] = float(nk * n2);
        f[3] = float(2.0 * a1);
        f[4] = float(2.0 * a2);
        f[5] = 0.0f;
        float* l = reinterpret_cast<float*>(o + kMeshFaceLen2);
        for (int k = 0; k < 5; k++) l[k] = float(l2[k]);
    }
}

// Plane test of one inside record.
RH_HD bool mesh_inside(const double* __restrict__ rec, const double p[3])
{
    const int np = int(rec[0]);
    bool in = true;
    for (int k = 0; k < kMeshPlanes; k++) {
        if (k < np) {
            const double* q = rec + 4 + 4 * k;
            in = in && (q[0] * p[0] + q[1] * p[1] + q[2] * p[2] < q[3]);
        }
    }
    return in;
}

}  // namespace rh
