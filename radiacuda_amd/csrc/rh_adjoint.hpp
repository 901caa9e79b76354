// rh_adjoint.hpp -- derivatives of the element fields for the adjoint kernels.
//
// dB/dM is the field block itself (B is linear in M).  For dB/d(vertex) the
// element's surface is taken as its faces fanned into triangles (v0, vk, vk+1),
// each CCW about the outward normal, and the field of the uniformly
// magnetized body is written per triangle t with unit normal n_t and surface
// charge sigma_t = n_t . M:
//
//     4 pi H(p) = sum_t sigma_t [ sum_{e in t} L_e (t_e x n_t) - Omega_t n_t ]
//
// L_e = ln((R_b + s_b)/(R_a + s_a)) over the triangle's edge a -> b and
// Omega_t the signed solid angle (Van Oosterom & Strackee).  For planar faces
// the internal fan edges cancel pairwise and this equals the face form used by
// the forward kernels; for displaced vertices it stays a closed triangulated
// surface, so its derivative is that of a well-defined field.  The device
// sweep (rh_adjoint.hip) has the derivatives in closed form; here they are
// forward-mode (dual numbers) with the three coordinates of one triangle
// corner seeded at a time, the independent form that the host build checks it
// with.
#pragma once

#include "rh_math.hpp"

namespace rh {

template <int K>
struct Dual {
    double v;
    double d[K];
    RH_HD Dual() : v(0.0)
    {
        for (int k = 0; k < K; k++) d[k] = 0.0;
    }
    RH_HD Dual(double x) : v(x)  // NOLINT: implicit constant
    {
        for (int k = 0; k < K; k++) d[k] = 0.0;
    }
};

template <int K>
RH_HD Dual<K> operator+(const Dual<K>& a, const Dual<K>& b)
{
    Dual<K> r;
    r.v = a.v + b.v;
    for (int k = 0; k < K; k++) r.d[k] = a.d[k] + b.d[k];
    return r;
}
template <int K>
RH_HD Dual<K> operator-(const Dual<K>& a, const Dual<K>& b)
{
    Dual<K> r;
    r.v = a.v - b.v;
    for (int k = 0; k < K; k++) r.d[k] = a.d[k] - b.d[k];
    return r;
}
template <int K>
RH_HD Dual<K> operator-(const Dual<K>& a)
{
    Dual<K> r;
    r.v = -a.v;
    for (int k = 0; k < K; k++) r.d[k] = -a.d[k];
    return r;
}
template <int K>
RH_HD Dual<K> operator*(const Dual<K>& a, const Dual<K>& b)
{
    Dual<K> r;
    r.v = a.v * b.v;
    for (int k = 0; k < K; k++) r.d[k] = a.d[k] * b.v + a.v * b.d[k];
    return r;
}
template <int K>
RH_HD Dual<K> operator/(const Dual<K>& a, const Dual<K>& b)
{
    Dual<K> r;
    const double ib = 1.0 / b.v;
    r.v = a.v * ib;
    for (int k = 0; k < K; k++) r.d[k] = (a.d[k] - r.v * b.d[k]) * ib;
    return r;
}
template <int K>
RH_HD bool operator<(const Dual<K>& a, const Dual<K>& b) { return a.v < b.v; }
template <int K>
RH_HD bool operator>(const Dual<K>& a, const Dual<K>& b) { return a.v > b.v; }
template <int K>
RH_HD bool operator>=(const Dual<K>& a, const Dual<K>& b) { return a.v >= b.v; }
template <int K>
RH_HD bool operator<=(const Dual<K>& a, const Dual<K>& b) { return a.v <= b.v; }

template <int K>
RH_HD Dual<K> rh_sqrt(const Dual<K>& a)
{
    Dual<K> r;
    r.v = sqrt(a.v);
    const double h = 0.5 / r.v;
    for (int k = 0; k < K; k++) r.d[k] = a.d[k] * h;
    return r;
}
template <int K>
RH_HD Dual<K> rh_log(const Dual<K>& a)
{
    Dual<K> r;
    r.v = log(a.v);
    const double ia = 1.0 / a.v;
    for (int k = 0; k < K; k++) r.d[k] = a.d[k] * ia;
    return r;
}
template <int K>
RH_HD Dual<K> rh_atan2(const Dual<K>& y, const Dual<K>& x)
{
    Dual<K> r;
    r.v = atan2(y.v, x.v);
    const double q = 1.0 / (x.v * x.v + y.v * y.v);
    for (int k = 0; k < K; k++) r.d[k] = (x.v * y.d[k] - y.v * x.d[k]) * q;
    return r;
}

template <class T>
RH_HD V3<T> vsub(const V3<T>& a, const V3<T>& b) { return V3<T>{a.x - b.x, a.y - b.y, a.z - b.z}; }
template <class T>
RH_HD V3<T> vscale(const V3<T>& a, const T& s) { return V3<T>{a.x * s, a.y * s, a.z * s}; }

// Adds 4 pi H of triangle (a, b, c) -- corners relative to the observation
// point, CCW about the outward normal -- for magnetization M.
template <class T>
RH_HD void tri_field(const V3<T>& a, const V3<T>& b, const V3<T>& c, const double M[3], V3<T>& H)
{
    const V3<T> nn = cross(vsub(b, a), vsub(c, a));
    const T an = rh_sqrt(dot(nn, nn));
    const T ian = T(1.0) / an;
    const V3<T> n = vscale(nn, ian);
    const T sigma = n.x * T(M[0]) + n.y * T(M[1]) + n.z * T(M[2]);
    const T Ra = rh_sqrt(dot(a, a)), Rb = rh_sqrt(dot(b, b)), Rc = rh_sqrt(dot(c, c));
    const V3<T>* P[3] = {&a, &b, &c};
    const T Rv[3] = {Ra, Rb, Rc};
    V3<T> s{T(0.0), T(0.0), T(0.0)};
    for (int e = 0; e < 3; e++) {
        const V3<T>& u = *P[e];
        const V3<T>& w = *P[(e + 1) % 3];
        const V3<T> d = vsub(w, u);
        const T len = rh_sqrt(dot(d, d));
        const V3<T> t = vscale(d, T(1.0) / len);
        T num, den;
        edge_ratio(u, Rv[e], w, Rv[(e + 1) % 3], t, num, den);
        const T L = rh_log(num / den);
        const V3<T> m = cross(t, n);
        s.x = s.x + L * m.x;
        s.y = s.y + L * m.y;
        s.z = s.z + L * m.z;
    }
    const T im = dot(a, cross(b, c));
    const T re = Ra * Rb * Rc + dot(a, b) * Rc + dot(a, c) * Rb + dot(b, c) * Ra;
    const T om = T(2.0) * rh_atan2(im, re);
    H.x = H.x + sigma * (s.x - om * n.x);
    H.y = H.y + sigma * (s.y - om * n.y);
    H.z = H.z + sigma * (s.z - om * n.z);
}

// Adjoint geometry record of one element: nv, ntri, vertices (3 nv, element
// frame, in the caller's vertex order), triangles (3 ntri vertex indices).
RH_HD int adj_nv(const double* rec) { return int(rec[0]); }
RH_HD int adj_ntri(const double* rec) { return int(rec[1]); }

// 4 pi H at p (value only) from the triangulated surface.
RH_HD void adj_field_value(const double* rec, const double p[3], const double M[3], double H[3])
{
    const int nv = adj_nv(rec), nt = adj_ntri(rec);
    const double* V = rec + 2;
    const double* T = V + 3 * nv;
    V3<double> h{0.0, 0.0, 0.0};
    for (int t = 0; t < nt; t++) {
        const int i0 = int(T[3 * t]), i1 = int(T[3 * t + 1]), i2 = int(T[3 * t + 2]);
        const V3<double> a = rel<double>(V + 3 * i0, p), b = rel<double>(V + 3 * i1, p),
                         c = rel<double>(V + 3 * i2, p);
        tri_field(a, b, c, M, h);
    }
    H[0] = h.x;
    H[1] = h.y;
    H[2] = h.z;
}

// Derivative of g . (4 pi H_t(p)) with respect to the three coordinates of
// corner k of triangle t; returns the triangle's indices' vertex in *vid.
RH_HD void adj_tri_corner_grad(const double* rec, int t, int k, const double p[3],
                               const double M[3], const double g[3], double out[3], int* vid)
{
    const int nv = adj_nv(rec);
    const double* V = rec + 2;
    const double* T = V + 3 * nv;
    const int id[3] = {int(T[3 * t]), int(T[3 * t + 1]), int(T[3 * t + 2])};
    V3<Dual<3>> r[3];
    for (int q = 0; q < 3; q++) {
        const double* v = V + 3 * id[q];
        r[q] = V3<Dual<3>>{Dual<3>(v[0] - p[0]), Dual<3>(v[1] - p[1]), Dual<3>(v[2] - p[2])};
    }
    r[k].x.d[0] = 1.0;
    r[k].y.d[1] = 1.0;
    r[k].z.d[2] = 1.0;
    V3<Dual<3>> h{Dual<3>(0.0), Dual<3>(0.0), Dual<3>(0.0)};
    tri_field(r[0], r[1], r[2], M, h);
    for (int c = 0; c < 3; c++) out[c] = g[0] * h.x.d[c] + g[1] * h.y.d[c] + g[2] * h.z.d[c];
    *vid = id[k];
}

// (1 - asinh(s)/s)/s^2 on s^2 <= 1/100 by powers of s^2: Chebyshev interpolant
// fitted at 60 digits, within 6e-17 relative
RH_TABLE d_asinh_p[6] = {0.16666666666666666, -0.0749999999999521,   0.04464285708693904,
                                    -0.030381920556719857, 0.02236754133836989, -0.016940234967509307};

// One triangle's part of dL/dvertex: geometry that does not depend on the
// observation point, and the sums over points.
struct TriLane {
    V3<double> v[3];  // corners, element frame
    V3<double> n, t[3];
    double len[3], il[3], ia, sigma;  // side lengths and reciprocals, 1/(2 area), n . M
    V3<double> M;
    V3<double> G[3];  // per corner: terms of L and of the solid angle
    V3<double> N;     // adjoint of the unit normal
    double al[3];     // per side: adjoint of its direction's own component
};

RH_FORM V3<double> axpy(double a, const V3<double>& x, const V3<double>& y)
{
    return V3<double>{fma(a, x.x, y.x), fma(a, x.y, y.y), fma(a, x.z, y.z)};
}

// Geometry of a triangle whose corners T.v are set, magnetization M, sums zero.
RH_FORM void tri_open(TriLane& T, const V3<double>& M)
{
    for (int k = 0; k < 3; k++) {
        T.G[k] = V3<double>{0.0, 0.0, 0.0};
        T.al[k] = 0.0;
    }
    T.N = V3<double>{0.0, 0.0, 0.0};
    T.M = M;
    const V3<double> nn = cross(vsub(T.v[1], T.v[0]), vsub(T.v[2], T.v[0]));
    T.ia = 1.0 / sqrt(dot(nn, nn));
    T.n = vscale(nn, T.ia);
    T.sigma = dot(T.n, T.M);
    for (int e = 0; e < 3; e++) {
        const V3<double> d = vsub(T.v[(e + 1) % 3], T.v[e]);
        T.len[e] = sqrt(dot(d, d));
        T.il[e] = 1.0 / T.len[e];
        T.t[e] = vscale(d, T.il[e]);
    }
}

// Derivatives of f = g . 4 pi H_t at one point, in closed form.  With
// m = sigma n x g, S = sum_e L_e t_e and u -> w the side e,
//     f = sigma (S . (n x g) - Omega n . g),
//     D = Ru Rw + u . w,  L = asinh(len (Ru + Rw)/D),
//     dL/dlen = (Ru + Rw)/D,  dL/dRu = dL/dRw = -len/D,
//     dOmega/dw = -(u x w)/(Rw D) per side (both ends alike, by 1/Ru, 1/Rw),
// the last because the solid angle changes by the area that a moved side
// sweeps, int s/r^3 = 1/(Rw D) along it.  No term needs a derivative of a
// logarithm's or an arctangent's argument.  Sums over points are taken of the
// differences between a corner's two sides, never of the sides' own terms,
// which are larger by distance over size.  gx: minus the sum of the corner
// derivatives (the normal's and the directions' parts cancel in it).
RH_FORM void tri_point(TriLane& T, const double x[3], const V3<double>& g, V3<double>& gx)
{
    V3<double> r[3];
    double R[3], iR[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        r[k] = V3<double>{T.v[k].x - x[0], T.v[k].y - x[1], T.v[k].z - x[2]};
        // R and 1/R from one seed y: with q = R^2 y and e = 1 - q y both are
        // the seed's value times 1 + e/2 + 3 e^2/8
        const double d = dot(r[k], r[k]);
        const double y = rh_rsq_seed(d);
        const double q = d * y, e = fma(-q, y, 1.0), c = e * fma(e, 0.375, 0.5);
        R[k] = fma(q, c, q);
        iR[k] = fma(y, c, y);
    }
    const V3<double> ng = cross(T.n, g);
    const double gn = dot(T.n, g), sgn = T.sigma * gn;
    V3<double> X[3], S{0.0, 0.0, 0.0};
    double uw[3], iD[3], sd[3], s2[3], w1[3], k1[3];
#pragma unroll
    for (int e = 0; e < 3; e++) {
        const int f = (e + 1) % 3;
        X[e] = cross(r[e], r[f]);
        uw[e] = dot(r[e], r[f]);
        const double RR = R[e] * R[f];
        double D = RR + uw[e];
        // beyond a right angle the sum cancels: |u x w|^2 = (RR - u.w) D
        if (uw[e] < 0.0) D = dot(X[e], X[e]) * rh_rcp(RR - uw[e]);
        iD[e] = rh_rcp(D);
        sd[e] = (R[e] + R[f]) * iD[e];
        const double s = T.len[e] * sd[e];
        s2[e] = s * s;
    }
    // w1 = sd - L/len and k1 = L/len: where every lane's sides are short
    // against their distance by the series, which loses no digits in w1
    if (rh_all(fmax(fmax(s2[0], s2[1]), s2[2]) <= 0.01)) {
#pragma unroll
        for (int e = 0; e < 3; e++) {
            double p = d_asinh_p[5];
#pragma unroll
            for (int i = 4; i >= 0; i--) p = fma(p, s2[e], d_asinh_p[i]);
            w1[e] = sd[e] * s2[e] * p;
            k1[e] = sd[e] - w1[e];
        }
    } else {
        RH_KEEP_BRANCH();
        const CoefPtr c = rh_coef_rare(d_log_p);
#pragma unroll
        for (int e = 0; e < 3; e++) {
            // len s = sinh L: e^L = (Ru + Rw + len)^2 / (2 D)
            const double q = R[e] + R[(e + 1) % 3] + T.len[e];
            k1[e] = rh_log_ratio_c(q * (0.5 * q) * iD[e], 1.0, c) * T.il[e];
            w1[e] = sd[e] - k1[e];
        }
    }
    const double re = R[0] * R[1] * R[2] + uw[0] * R[2] + uw[2] * R[1] + uw[1] * R[0];
    const double om = 2.0 * rh_atan2_wave(dot(r[0], X[1]), re);
    double kk[3], cc[3];
#pragma unroll
    for (int e = 0; e < 3; e++) {
        S = axpy(k1[e] * T.len[e], T.t[e], S);
        const double tm = T.sigma * dot(T.t[e], ng);
        T.al[e] = fma(tm, w1[e], T.al[e]);
        kk[e] = tm * T.len[e] * iD[e];
        cc[e] = -sgn * iD[e];
    }
    // the normal: f = phi sigma, d sigma = dn . M
    const double phi = dot(S, ng) - om * gn;
    const V3<double> gS = cross(g, S);
    T.N = axpy(phi, T.M, axpy(T.sigma, V3<double>{fma(-om, g.x, gS.x), fma(-om, g.y, gS.y), fma(-om, g.z, gS.z)}, T.N));
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int in = (k + 2) % 3;  // side ending in corner k; side k starts there
        const double kr = kk[in] + kk[k];
        const V3<double> h{iR[k] * fma(kr, r[k].x, fma(cc[in], X[in].x, cc[k] * X[k].x)),
                           iR[k] * fma(kr, r[k].y, fma(cc[in], X[in].y, cc[k] * X[k].y)),
                           iR[k] * fma(kr, r[k].z, fma(cc[in], X[in].z, cc[k] * X[k].z))};
        const double dk = T.sigma * (k1[in] - k1[k]);
        T.G[k] = V3<double>{T.G[k].x + fma(dk, ng.x, -h.x), T.G[k].y + fma(dk, ng.y, -h.y),
                            T.G[k].z + fma(dk, ng.z, -h.z)};
        gx.x += h.x;
        gx.y += h.y;
        gx.z += h.z;
    }
}

// Corner gradients from the sums.  Side directions: dt = (dd - t (t . dd))/len
// moved both ends by -+ dd; the length's part is along t; the unit normal:
// n = (v1 - v0) x (v2 - v0)/|.|
RH_FORM void tri_close(const TriLane& T, V3<double> (&G)[3])
{
    const V3<double> e1 = vsub(T.v[1], T.v[0]), e2 = vsub(T.v[2], T.v[0]);
    const V3<double> q = vscale(axpy(-dot(T.n, T.N), T.n, T.N), T.ia);
    const V3<double> g1 = cross(e2, q), g2 = cross(q, e1);
    G[0] = vsub(T.G[0], V3<double>{g1.x + g2.x, g1.y + g2.y, g1.z + g2.z});
    G[1] = V3<double>{T.G[1].x + g1.x, T.G[1].y + g1.y, T.G[1].z + g1.z};
    G[2] = V3<double>{T.G[2].x + g2.x, T.G[2].y + g2.y, T.G[2].z + g2.z};
    for (int k = 0; k < 3; k++) G[k] = axpy(T.al[(k + 2) % 3], T.t[(k + 2) % 3], axpy(-T.al[k], T.t[k], G[k]));
}

}  // namespace rh
