// FP64 setup kernels: radiation / receiving patterns, near-field Galerkin
// blocks, plane-wave excitation and far-field (RCS) sums.
#include "cplx.hpp"
#include "geo.hpp"
#include "setup.hpp"

#include <stdexcept>
#include <type_traits>

namespace mlfma {

namespace {
constexpr double kPiD = 3.14159265358979323846;
constexpr double kEps0D = 2.2204e-16;   // Code/PhyConstant.h:13

struct R3 {
    double x, y, z;
};
__device__ __forceinline__ R3 mk(const double* p) { return {p[0], p[1], p[2]}; }
__device__ __forceinline__ R3 sub3(R3 a, R3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ R3 add3(R3 a, R3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ R3 scl3(R3 a, double s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ double dot3(R3 a, R3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ R3 crs3(R3 a, R3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ double nrm3(R3 a) { return sqrt(dot3(a, a)); }
__device__ __forceinline__ R3 gpt(const GaussRule& g, int q, const double* t) {
    return {g.l1[q] * t[0] + g.l2[q] * t[3] + g.l3[q] * t[6], g.l1[q] * t[1] + g.l2[q] * t[4] + g.l3[q] * t[7],
            g.l1[q] * t[2] + g.l2[q] * t[5] + g.l3[q] * t[8]};
}
// exp(-j k R) for complex k = kr + j ki
__device__ __forceinline__ double2 expmjk(double2 k, double R) {
    double s, c;
    sincos(k.x * R, &s, &c);
    const double m = (k.y != 0.0) ? exp(k.y * R) : 1.0;
    return make_double2(m * c, -m * s);
}

// Analytic integrals over a flat source triangle of 1/R and 1/R^3 (vector and
// scalar parts) for one observation point on that triangle (the identical-face
// terms); Code/Operator.h:72-305 and :585-674.  The point's height D above the
// triangle's plane is exactly 0: the reference computes D = n.(r - v) in floating
// point, and that rounding noise (~1e-16 |r|) picks between the two branches of the
// 1/R^3 scalar integral, one of which divides an O(1) angle difference by the noise;
// D = 0 gives the reference's value wherever its noise stays below 10 eps0.
struct SingFrame {
    R3 rho[3], l[3], u[3], n;
};
struct SingPt {
    R3 Iv, Iv3, rho;
    double Is, Is3;
};

__device__ void sing_frame(const double* t, const double* nn, SingFrame& f) {
    f.n = mk(nn);
    for (int v = 0; v < 3; ++v) {
        R3 p = mk(t + 3 * v);
        f.rho[v] = sub3(p, scl3(f.n, dot3(f.n, p)));
    }
    for (int e = 0; e < 3; ++e) {
        R3 d = sub3(f.rho[(e + 1) % 3], f.rho[e]);
        double L = nrm3(d);
        f.l[e] = {d.x / L, d.y / L, d.z / L};
        f.u[e] = crs3(f.l[e], f.n);
    }
}

__device__ void sing_point(R3 r, const double* t, const SingFrame& f, bool want3, SingPt& o) {
    const double th = 50.0 * kEps0D;
    const R3 rho = sub3(r, scl3(f.n, dot3(f.n, r)));
    o.rho = rho;
    o.Iv = {0, 0, 0};
    o.Iv3 = {0, 0, 0};
    o.Is = 0;
    o.Is3 = 0;
    for (int e = 0; e < 3; ++e) {
        // edge e runs from vertex e ("minus" end) to vertex e+1 ("plus" end)
        const R3 dp = sub3(f.rho[(e + 1) % 3], rho), dm = sub3(f.rho[e], rho);
        const double Lp = dot3(dp, f.l[e]), Lm = dot3(dm, f.l[e]);
        const double P0 = fabs(dot3(dp, f.u[e]));
        const double Pp = nrm3(dp), Pm = nrm3(dm);
        R3 P0v = {0, 0, 0};
        if (!(P0 < th)) {
            const R3 pm = sub3(dp, scl3(f.l[e], Lp));
            P0v = {pm.x / P0, pm.y / P0, pm.z / P0};
        }
        const double D = 0.0;
        const double R0 = sqrt(P0 * P0 + D * D), Rp = sqrt(Pp * Pp + D * D), Rm = sqrt(Pm * Pm + D * D);
        const double LOGp = (Rp + Lp < th) ? 0.0 : log(Rp + Lp);
        const double LOGm = (Rm + Lm < th) ? 0.0 : log(Rm + Lm);
        const double c1 = 0.5 * (R0 * R0 * (LOGp - LOGm) + Rp * Lp - Rm * Lm);
        o.Iv = add3(o.Iv, scl3(f.u[e], c1));
        const double ad = fabs(D);
        const double denp = R0 * R0 + ad * Rp, denm = R0 * R0 + ad * Rm;
        const double atp = (denp < th) ? 0.0 : atan((P0 * Lp) / denp);
        const double atm = (denm < th) ? 0.0 : atan((P0 * Lm) / denm);
        const double pu = dot3(P0v, f.u[e]);
        o.Is = o.Is + pu * (P0 * (LOGp - LOGm) - ad * (atp - atm));
        if (want3) {
            o.Iv3 = sub3(o.Iv3, scl3(f.u[e], LOGp - LOGm));
            const double t10 = 10.0 * kEps0D;
            if (ad >= t10) {
                const double ap = atan((P0 * Lp) / (R0 * R0 + ad * Rp));
                const double am = atan((P0 * Lm) / (R0 * R0 + ad * Rm));
                o.Is3 = o.Is3 + pu * ((1.0 / ad) * (ap - am));
            } else if (P0 >= t10) {
                o.Is3 = o.Is3 - pu * (Lp / (P0 * Rp) - Lm / (P0 * Rm));
            } else {
                o.Is3 = 0.0;   // the reference resets the accumulator (Code/Operator.h:671-673)
            }
        }
    }
}

// Galerkin integrals between one half of field RWG F and one half of source RWG
// S on the same face (identical-face singular extraction), free vertices vF, vS:
//   L(k):  Code/Operator.h:709-881     (EFIE = eta * L, Code/EFIE.cpp:6-194)
//   K(k):  Code/Operator.h:883-1046
//   M(k):  MFIE, Code/MFIE.cpp:6-212
// without the factor len_F len_S / (4 pi) and the halves' signs.
template <int NK, bool WL, bool WK, bool WM>
__device__ void same_face_ops(const FaceGeo& F, R3 vF, const FaceGeo& S, R3 vS, const GaussRule& g, const double2* ks,
                              double2* aL, double2* aK, double2* aM) {
    const R3 nF = mk(F.nrm);
    const double AF = F.area, recAf = 1.0 / (2.0 * AF), AS = S.area, recAs = 1.0 / (2.0 * AS);
    *aM = make_double2(0, 0);
    for (int q = 0; q < NK; ++q) aL[q] = aK[q] = make_double2(0, 0);
    for (int a = 0; a < g.n; ++a) {
        const R3 rf = gpt(g, a, F.tri);
        const R3 pf = sub3(rf, vF);
        for (int b = 0; b < g.n; ++b) {
            const R3 rs = gpt(g, b, S.tri);
            const R3 ps = sub3(rs, vS);
            const R3 Rv = sub3(rf, rs);
            const double R = nrm3(Rv);
            const double w = g.w[a] * g.w[b];
            const double dL = WL ? dot3(pf, ps) : 0.0;
            const double dK = WK ? dot3(pf, crs3(Rv, ps)) : 0.0;
            const double dM = WM ? dot3(crs3(sub3(rf, vS), ps), crs3(pf, nF)) : 0.0;
#pragma unroll
            for (int q = 0; q < NK; ++q) {
                const double2 k = ks[q];
                const double2 jk = make_double2(-k.y, k.x);
                double2 G, G3;
                if (R < kEps0D) {
                    G = make_double2(k.y, -k.x);   // -j k
                    G3 = make_double2(0, 0);
                } else {
                    const double2 e = expmjk(k, R);
                    G = make_double2(e.x / R - 1.0 / R, e.y / R);
                    G3 = cscale(cmul(e, make_double2(1.0 - k.y * R, k.x * R)), 1.0 / (R * R * R));
                    const double2 k2 = cmul(k, k);
                    G3.x -= 1.0 / (R * R * R) + 0.5 * k2.x / R;
                    G3.y -= 0.5 * k2.y / R;
                }
                if (WL) {
                    // jk w (G pf.ps - 4 G / k^2)
                    const double2 c4 = cdiv(make_double2(4.0, 0.0), cmul(k, k));
                    cfma(aL[q], cscale(jk, w), csub(cscale(G, dL), cmul(G, c4)));
                }
                if (WK) cfma(aK[q], make_double2(w, 0.0), cscale(G3, dK));
                if (WM && q == 0) cfma(*aM, make_double2(w, 0.0), cscale(G3, dM));
            }
        }
    }
    SingFrame fr;
    sing_frame(S.tri, S.nrm, fr);
    const R3 rho0N = sub3(vS, scl3(fr.n, dot3(fr.n, vS)));
    for (int a = 0; a < g.n; ++a) {
        const R3 rf = gpt(g, a, F.tri);
        const double wF = g.w[a];
        SingPt sp;
        sing_point(rf, S.tri, fr, WK || WM, sp);
        const R3 RWGf = scl3(sub3(rf, vF), recAf);
        const R3 pv1 = sub3(sp.rho, rho0N);
        const R3 Ri = sub3(rf, vS);
        if (WM) {   // identity term, Code/MFIE.cpp:175-192
            const R3 RWGs = scl3(Ri, recAs);
            aM->x += 4.0 * kPiD * wF * AF * dot3(RWGf, RWGs);
        }
#pragma unroll
        for (int q = 0; q < NK; ++q) {
            const double2 k = ks[q];
            const double2 jk = make_double2(-k.y, k.x);
            const double2 k2 = cmul(k, k);
            if (WL) {
                const R3 Ikon = scl3(add3(sp.Iv, scl3(pv1, sp.Is)), recAs);
                const double2 t = csub(make_double2(dot3(RWGf, Ikon), 0.0),
                                       cscale(cdiv(make_double2(1.0, 0.0), k2), sp.Is / (AF * AS)));
                cfma(aL[q], cscale(jk, wF * 2.0 * AF), t);
            }
            if (WK || (WM && q == 0)) {
                // Ikon = (k^2/2)(Iv + pv1 Is)/(2As) + (Iv3 + pv1 Is3)/(2As)
                const double2 h = cscale(k2, 0.5);
                const R3 a1 = add3(sp.Iv, scl3(pv1, sp.Is));
                const R3 a3 = add3(sp.Iv3, scl3(pv1, sp.Is3));
                const double2 I0 = make_double2(h.x * a1.x * recAs + a3.x * recAs, h.y * a1.x * recAs);
                const double2 I1 = make_double2(h.x * a1.y * recAs + a3.y * recAs, h.y * a1.y * recAs);
                const double2 I2 = make_double2(h.x * a1.z * recAs + a3.z * recAs, h.y * a1.z * recAs);
                // Ri x Ikon
                const double2 X0 = csub(cscale(I2, Ri.y), cscale(I1, Ri.z));
                const double2 X1 = csub(cscale(I0, Ri.z), cscale(I2, Ri.x));
                const double2 X2 = csub(cscale(I1, Ri.x), cscale(I0, Ri.y));
                if (WK) {
                    double2 d = cadd(cadd(cscale(X0, RWGf.x), cscale(X1, RWGf.y)), cscale(X2, RWGf.z));
                    aK[q] = cadd(aK[q], cscale(d, wF * 2.0 * AF));
                }
                if (WM && q == 0) {
                    const R3 c2 = crs3(RWGf, nF);
                    double2 d = cadd(cadd(cscale(X0, c2.x), cscale(X1, c2.y)), cscale(X2, c2.z));
                    *aM = cadd(*aM, cscale(d, wF * 2.0 * AF));
                }
            }
        }
    }
}

// complex 3-vectors of the face-pair sums
struct C3 {
    double2 x, y, z;
};
__device__ __forceinline__ void acc3(C3& s, double2 g, R3 p) {
    s.x.x = fma(g.x, p.x, s.x.x), s.x.y = fma(g.y, p.x, s.x.y);
    s.y.x = fma(g.x, p.y, s.y.x), s.y.y = fma(g.y, p.y, s.y.y);
    s.z.x = fma(g.x, p.z, s.z.x), s.z.y = fma(g.y, p.z, s.z.y);
}
__device__ __forceinline__ double2 dotc(R3 p, const C3& s) {
    return make_double2(fma(p.z, s.z.x, fma(p.y, s.y.x, p.x * s.x.x)), fma(p.z, s.z.y, fma(p.y, s.y.y, p.x * s.x.y)));
}
__device__ __forceinline__ C3 crossc(R3 p, const C3& s) {
    C3 o;
    o.x = make_double2(p.y * s.z.x - p.z * s.y.x, p.y * s.z.y - p.z * s.y.y);
    o.y = make_double2(p.z * s.x.x - p.x * s.z.x, p.z * s.x.y - p.x * s.z.y);
    o.z = make_double2(p.x * s.y.x - p.y * s.x.x, p.x * s.y.y - p.y * s.x.y);
    return o;
}

}  // namespace

// ---------------------------------------------------------------- near field
// Code/Zmartix.h:188-278 (EFIE), :372-465 (CFIE), :541-643 (PMCHWT).  An entry
// is the signed sum over the two halves of each RWG, and every (face, free
// vertex) pair is a half of one RWG only, so a pair of faces with its 49
// kernel evaluations (sincos, 1/R; exp in a lossy medium) serves 9 entries'
// halves: evaluating per entry repeated it up to nine times.  9,720 PMCHWT RWG
// in 40 leaves: 113 ms per entry, 11 ms by face pairs; 151,230 RWG: 1.4 and
// 0.2 s; 300,000 RWG CFIE: 1.2 and 0.14 s; 48,000 RWG in leaves of up to 18
// (faces shared least): 50 and 8 ms.  k_face_pairs takes one pair of faces per thread and leaves
// the integrals for the 3 x 3 free-vertex pairs in a bounded scratch array,
// k_face_same those of identical faces (singular extraction), and
// k_near_assemble sums each entry's four in a fixed order.
//
// The sums over the source points need the kernels only against 1 and r' - v_0:
// with T_n = sum G (r' - v_n), L wants (r - v_m).T_n, and since
// (r - r') x (r' - v_n) = (r - v_n) x (r' - v_n), K and the MFIE want
// (r - v_n) x T_n of the gradient kernel.
template <int MODE>
__global__ __launch_bounds__(64) void k_face_pairs(NearFill nf, const int2* __restrict__ items, GaussRule g,
                                                   NearConsts c, size_t cap, double2* __restrict__ scr) {
    constexpr int PL = MODE == 2 ? 3 : 1;
    const int2 it = items[blockIdx.x];
    const FillBlock& B = nf.blocks[it.x];
    const int f0 = nf.face_ptr[B.gt], nF = nf.face_ptr[B.gt + 1] - f0;
    const int s0 = nf.face_ptr[B.gs], nS = nf.face_ptr[B.gs + 1] - s0;
    const int e = it.y * 64 + threadIdx.x;
    if (e >= nF * nS) return;
    const int sl = e / nF, fl = e - sl * nF;
    const FaceGeo& F = nf.faces[nf.face_idx[f0 + fl]];
    const FaceGeo& S = nf.faces[nf.face_idx[s0 + sl]];
    if (F.id == S.id) return;   // k_face_same
    double tS[9], tF[9];
    for (int v = 0; v < 9; ++v) tS[v] = S.tri[v], tF[v] = F.tri[v];
    const R3 vS0 = mk(tS);
    double2 D1[3][3], D2[3][3], DK[3][3];   // [field vertex][source vertex]
    for (int m = 0; m < 3; ++m)
        for (int n = 0; n < 3; ++n) D1[m][n] = D2[m][n] = DK[m][n] = make_double2(0, 0);
    double2 E1 = {0, 0}, E2 = {0, 0};
    const R3 nrm = mk(F.nrm);
    for (int a = 0; a < g.n; ++a) {
        const R3 rf = gpt(g, a, tF);
        const double wF = g.w[a];
        double2 g1 = {0, 0}, g2 = {0, 0}, h = {0, 0};
        C3 G1 = {{0, 0}, {0, 0}, {0, 0}}, G2 = G1, H = G1;
        for (int b = 0; b < g.n; ++b) {
            const R3 rs = gpt(g, b, tS);
            const R3 ps = sub3(rs, vS0);
            const double R2 = dot3(sub3(rf, rs), sub3(rf, rs));
            const double R = sqrt(R2), ri = 1.0 / R;
            const double w = g.w[b];
            const double wi = w * ri, wi3 = wi * (ri * ri);
            const double2 e1 = expmjk(c.k1, R);
            const double2 u1 = cscale(e1, wi);
            g1 = cadd(g1, u1);
            acc3(G1, u1, ps);
            if (MODE >= 1) {   // gradient kernel e (1 + j k R) / R^3, both media of PMCHWT together
                double2 q = cmul(e1, make_double2(1.0 - c.k1.y * R, c.k1.x * R));
                if (MODE == 2) {
                    const double2 e2 = expmjk(c.k2, R);
                    const double2 u2 = cscale(e2, wi);
                    g2 = cadd(g2, u2);
                    acc3(G2, u2, ps);
                    q = cadd(q, cmul(e2, make_double2(1.0 - c.k2.y * R, c.k2.x * R)));
                }
                q = cscale(q, wi3);
                h = cadd(h, q);
                acc3(H, q, ps);
            }
        }
        E1 = cadd(E1, cscale(g1, wF));
        if (MODE == 2) E2 = cadd(E2, cscale(g2, wF));
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const R3 vn = mk(tS + 3 * n), d = sub3(vS0, vn);
            C3 T1 = G1, T2 = G2, TH = H;
            acc3(T1, g1, d);
            if (MODE == 2) acc3(T2, g2, d);
            if (MODE >= 1) {
                acc3(TH, h, d);
                TH = crossc(sub3(rf, vn), TH);
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                const R3 pf = scl3(sub3(rf, mk(tF + 3 * m)), wF);
                D1[m][n] = cadd(D1[m][n], dotc(pf, T1));
                if (MODE == 2) D2[m][n] = cadd(D2[m][n], dotc(pf, T2));
                if (MODE == 2) DK[m][n] = cadd(DK[m][n], dotc(pf, TH));
                if (MODE == 1) DK[m][n] = cadd(DK[m][n], dotc(crs3(pf, nrm), TH));
            }
        }
    }
    // L = jk (sum G pf.ps - 4 / k^2 sum G)
    const double2 four = make_double2(4.0, 0.0);
    const double2 jk1 = make_double2(-c.k1.y, c.k1.x), jk2 = make_double2(-c.k2.y, c.k2.x);
    E1 = cmul(E1, cdiv(four, cmul(c.k1, c.k1)));
    if (MODE == 2) E2 = cmul(E2, cdiv(four, cmul(c.k2, c.k2)));
    double2* o = scr + B.slot0 + e;
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            double2* q = o + (size_t)(m * 3 + n) * PL * cap;
            const double2 L1 = cmul(jk1, csub(D1[m][n], E1));
            if (MODE == 2) {
                const double2 L2 = cmul(jk2, csub(D2[m][n], E2));
                q[0] = cadd(L1, cmul(c.etai, L2));
                q[cap] = DK[m][n];
                q[2 * cap] = cadd(L1, cmul(c.inv_etai, L2));
            } else if (MODE == 0) {
                q[0] = cmul(c.eta1, L1);
            } else {   // alpha E + (1 - alpha) eta M, E = eta L  (Code/Zmartix.h:432)
                q[0] = cadd(cscale(cmul(c.eta1, L1), c.alpha), cscale(cmul(c.eta1, DK[m][n]), 1.0 - c.alpha));
            }
        }
}

// Identical faces: one thread per (listed pair, free-vertex pair).
template <int MODE>
__global__ __launch_bounds__(64) void k_face_same(NearFill nf, int count, const int2* __restrict__ same, GaussRule g,
                                                  NearConsts c, size_t cap, double2* __restrict__ scr) {
    constexpr int PL = MODE == 2 ? 3 : 1;
    const int idx = blockIdx.x * 64 + threadIdx.x;
    if (idx >= count * 9) return;
    const int p = idx / 9, m = (idx - p * 9) / 3, n = idx - p * 9 - m * 3;
    const FillBlock& B = nf.blocks[same[p].x];
    const int e = same[p].y;
    const int f0 = nf.face_ptr[B.gt], nF = nf.face_ptr[B.gt + 1] - f0, s0 = nf.face_ptr[B.gs];
    const int sl = e / nF, fl = e - sl * nF;
    const FaceGeo& F = nf.faces[nf.face_idx[f0 + fl]];
    const FaceGeo& S = nf.faces[nf.face_idx[s0 + sl]];
    const R3 vF = mk(F.tri + 3 * m), vS = mk(S.tri + 3 * n);
    double2* q = scr + (size_t)(m * 3 + n) * PL * cap + B.slot0 + e;
    double2 L[2], K[2], M;
    if (MODE == 2) {
        const double2 ks[2] = {c.k1, c.k2};
        same_face_ops<2, true, true, false>(F, vF, S, vS, g, ks, L, K, &M);
        q[0] = cadd(L[0], cmul(c.etai, L[1]));
        q[cap] = cadd(K[0], K[1]);
        q[2 * cap] = cadd(L[0], cmul(c.inv_etai, L[1]));
    } else if (MODE == 0) {
        same_face_ops<1, true, false, false>(F, vF, S, vS, g, &c.k1, L, K, &M);
        q[0] = cmul(c.eta1, L[0]);
    } else {
        same_face_ops<1, true, false, true>(F, vF, S, vS, g, &c.k1, L, K, &M);
        q[0] = cadd(cscale(cmul(c.eta1, L[0]), c.alpha), cscale(cmul(c.eta1, M), 1.0 - c.alpha));
    }
}

// Entries of the blocks: rows of the target group x columns of the source
// group, 256 per workgroup, rows fastest (layout of NearDev, geo.hpp).
template <int PL>
__global__ __launch_bounds__(256) void k_near_assemble(NearFill nf, const int2* __restrict__ items, size_t cap,
                                                       const double2* __restrict__ scr, double2* __restrict__ Z) {
    const int2 it = items[blockIdx.x];
    const FillBlock& B = nf.blocks[it.x];
    const int i0 = nf.row_ptr[B.gt], nr = nf.row_ptr[B.gt + 1] - i0;
    const int j0 = nf.row_ptr[B.gs], nc = nf.row_ptr[B.gs + 1] - j0;
    const int e = it.y * 256 + threadIdx.x;
    if (e >= nr * nc) return;
    const int col = e / nr, row = e - col * nr;
    const int nF = nf.face_ptr[B.gt + 1] - nf.face_ptr[B.gt];
    const int2 sf = nf.side[i0 + row], ss = nf.side[j0 + col];   // face * 4 + free vertex of the - and + halves
    const double sc = nf.len[i0 + row] * nf.len[j0 + col] / (4.0 * kPiD);
    double2 z[PL];
    for (int p = 0; p < PL; ++p) z[p] = make_double2(0, 0);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int f = a == 0 ? sf.x : sf.y, s = b == 0 ? ss.x : ss.y;
            const double2* v = scr + (size_t)((f & 3) * 3 + (s & 3)) * PL * cap + B.slot0 + (s >> 2) * nF + (f >> 2);
            const double w = a == b ? sc : -sc;
#pragma unroll
            for (int p = 0; p < PL; ++p) z[p] = cadd(z[p], cscale(v[(size_t)p * cap], w));
        }
    double2* o = Z + B.out + (size_t)col * B.ld + row;
#pragma unroll
    for (int p = 0; p < PL; ++p) o[(size_t)p * B.plane] = z[p];
}

void launch_near_fill(hipStream_t st, int mode, const NearFill& nf, const int2* pair_items, int npair,
                      const int2* same, int nsame, const int2* entry_items, int nentry, const GaussRule& g,
                      const NearConsts& c, size_t cap, double2* scr, double2* Z) {
    const unsigned sb = (unsigned)(((long long)nsame * 9 + 63) / 64);
#define FILL(M)                                                                        \
    k_face_pairs<M><<<npair, 64, 0, st>>>(nf, pair_items, g, c, cap, scr);             \
    if (nsame > 0) k_face_same<M><<<sb, 64, 0, st>>>(nf, nsame, same, g, c, cap, scr); \
    k_near_assemble<M == 2 ? 3 : 1><<<nentry, 256, 0, st>>>(nf, entry_items, cap, scr, Z)
    if (npair == 0) return;
    if (mode == 2) {
        FILL(2);
    } else if (mode == 1) {
        FILL(1);
    } else {
        FILL(0);
    }
#undef FILL
}

// ---------------------------------------------------------------- patterns
// Code/ProcessFMM.h:17-180: per RWG (internal order) and k-space sample,
//   Vs = sum_q w l e^{+jk khat.(r-c)} (r - v_free)                (KernelVsmi_Efie)
//   Vf = sum_q w l e^{-jk khat.(r-c)} (-khat x (khat x (r - v)))   (KernelVfmj_Efie)
//   or alpha * that + (1-alpha) khat x (n x (r - v))               (KernelVfmj_Cfie)
// positive face minus negative face.
template <bool CFIE>
__global__ __launch_bounds__(256) void k_patterns(int K, const RwgGeo* __restrict__ geo, const int* __restrict__ leaf_of,
                                                  const double* __restrict__ centre, const double* __restrict__ kp,
                                                  double2 k, GaussRule g, double alpha, double2* __restrict__ Vs,
                                                  double2* __restrict__ Vf) {
    const int i = blockIdx.x;
    const int q = blockIdx.y * blockDim.x + threadIdx.x;
    if (q >= K) return;
    const RwgGeo& G = geo[i];
    const int lf = leaf_of[i];
    const R3 c = {centre[3 * lf], centre[3 * lf + 1], centre[3 * lf + 2]};
    const R3 kh = {kp[q], kp[K + q], kp[2 * K + q]};
    double2 s0 = {0, 0}, s1 = {0, 0}, s2 = {0, 0}, f0 = {0, 0}, f1 = {0, 0}, f2 = {0, 0};
    for (int a = 0; a < g.n; ++a) {
        const double w = g.w[a] * G.len;
        for (int side = 1; side >= 0; --side) {
            const double sg = side == 1 ? 1.0 : -1.0;
            const R3 r = gpt(g, a, G.tri[side]);
            const R3 pf = sub3(r, mk(G.vf[side]));
            const double ph = dot3(sub3(r, c), kh);
            double sn, cs;
            sincos(k.x * ph, &sn, &cs);
            const double mf = (k.y != 0.0) ? exp(k.y * ph) : 1.0;    // |e^{-jk ph}|
            const double ms = (k.y != 0.0) ? exp(-k.y * ph) : 1.0;   // |e^{+jk ph}|
            const double2 es = make_double2(sg * w * ms * cs, sg * w * ms * sn);
            const double2 ef = make_double2(sg * w * mf * cs, -sg * w * mf * sn);
            s0 = cadd(s0, cscale(es, pf.x));
            s1 = cadd(s1, cscale(es, pf.y));
            s2 = cadd(s2, cscale(es, pf.z));
            const R3 t1 = crs3(kh, pf);
            const R3 t2 = crs3(kh, t1);
            R3 v = {-t2.x, -t2.y, -t2.z};
            if (CFIE) {
                const R3 m = crs3(kh, crs3(mk(G.nrm[side]), pf));
                v = add3(scl3(v, alpha), scl3(m, 1.0 - alpha));
            }
            f0 = cadd(f0, cscale(ef, v.x));
            f1 = cadd(f1, cscale(ef, v.y));
            f2 = cadd(f2, cscale(ef, v.z));
        }
    }
    double2* o = Vs + (size_t)i * 3 * K + q;
    o[0] = s0, o[K] = s1, o[2 * K] = s2;
    o = Vf + (size_t)i * 3 * K + q;
    o[0] = f0, o[K] = f1, o[2 * K] = f2;
}

void launch_patterns(hipStream_t st, bool cfie, int N, int K, const RwgGeo* geo, const int* leaf_of,
                     const double* centre, const double* kp, double2 k, const GaussRule& g, double alpha, double2* Vs,
                     double2* Vf) {
    dim3 grid(N, (K + 255) / 256);   // gridDim.y is limited to 65535
    if (cfie) k_patterns<true><<<grid, 256, 0, st>>>(K, geo, leaf_of, centre, kp, k, g, alpha, Vs, Vf);
    else k_patterns<false><<<grid, 256, 0, st>>>(K, geo, leaf_of, centre, kp, k, g, alpha, Vs, Vf);
}

// ---------------------------------------------------------------- excitation
// Code/Vm.h:10-203: E-testing <f, E e^{-jk kinc.r}>, H-testing with (n x H).rho
// (CFIE) or H.rho (PMCHWT); one thread per RWG, written at the reference index.
// Up to NI incidences per thread, so that the RWG's record and quadrature points
// are read once for all of them.  With one incidence per launch 8 of them at
// 75,000 RWG took 176 us, together 84.
template <int NI>
__global__ __launch_bounds__(256) void k_excitation(int N, int mode, const RwgGeo* __restrict__ geo,
                                                    const int* __restrict__ perm, GaussRule g, ExcitationBatch b,
                                                    size_t ld, double2* __restrict__ v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const RwgGeo& G = geo[i];
    double2 vE[NI], vH[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) vE[j] = vH[j] = make_double2(0, 0);
    for (int q = 0; q < g.n; ++q) {
        for (int side = 1; side >= 0; --side) {
            const R3 r = gpt(g, q, G.tri[side]);
            // rho = r - v+ on the positive face, v- - r on the negative face
            const R3 rho = side == 1 ? sub3(r, mk(G.vf[1])) : sub3(mk(G.vf[0]), r);
            const double wl = G.len * g.w[q];
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                if (j >= b.n) break;   // uniform
                const ExcitationArgs& a = b.a[j];
                const R3 kin = {a.kinc[0], a.kinc[1], a.kinc[2]};
                const R3 E = {a.einc[0], a.einc[1], a.einc[2]};
                const R3 H = {a.hinc[0], a.hinc[1], a.hinc[2]};
                const double2 e = expmjk(a.k, dot3(kin, r));
                vE[j] = cadd(vE[j], cscale(e, wl * dot3(E, rho)));
                if (mode == 1) vH[j] = cadd(vH[j], cscale(e, wl * dot3(crs3(mk(G.nrm[side]), H), rho)));
                if (mode == 2) vH[j] = cadd(vH[j], cscale(e, wl * dot3(H, rho)));
            }
        }
    }
    const int r = perm[i];
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        if (j >= b.n) break;
        double2* o = v + (size_t)j * ld;
        if (mode == 0) o[r] = vE[j];
        else if (mode == 1) o[r] = cadd(cscale(vE[j], b.a[j].alpha), cscale(vH[j], 1.0 - b.a[j].alpha));
        else {
            o[r] = vE[j];
            o[N + r] = vH[j];
        }
    }
}

void launch_excitation(hipStream_t st, int N, int mode, const RwgGeo* geo, const int* perm, const GaussRule& g,
                       const ExcitationBatch& b, size_t ld, double2* v) {
    if (b.n < 1 || b.n > kExcitationBatch) throw std::invalid_argument("excitation: 1..8 incidences per launch");
    if (b.n == 1) k_excitation<1><<<(N + 255) / 256, 256, 0, st>>>(N, mode, geo, perm, g, b, ld, v);
    else k_excitation<kExcitationBatch><<<(N + 255) / 256, 256, 0, st>>>(N, mode, geo, perm, g, b, ld, v);
}

// ---------------------------------------------------------------- far field
// Code/RCS.h:54-192: per observation direction, block partial sums of
//   PEC:    jk eta sum_n I_n F_n,  F_n = l sum_q w (I - rr).rho e^{+jk r.p}
//   PMCHWT: jk1 sum_n (F_n I_J - (r x rho part) I_M)
// A thread takes its RWG's quadrature points once for NA directions and sums
// V = l sum_q w rho e^{+jk r.p} first; the projections (I - rr).V and r x V
// follow once per direction instead of once per point.  Bound by the FP64 sine
// and cosine of every (point, direction).  181 directions of 75,000 RWG: 879 us
// with one direction per thread and projected points, now 636.
// One direction per thread is for launches too small to fill the chip with four,
// and a single chain of latency: it takes its record into registers at once (138
// of them; with four directions there is no room) and hides the phase's origin
// from the compiler, which otherwise computes the sine's reduction of huge
// arguments for every point instead of branching round it.  Without the two, 361
// directions of 2,430 RWG took 91 us and 37 of 12,000 took 48, now 54 and 30;
// four directions are faster without them (189 us, 203 with the hidden phase:
// 361 of 12,000).
template <int NA>
__global__ __launch_bounds__(256) void k_farfield(int N, int pmchwt, const RwgGeo* __restrict__ geo,
                                                  const int* __restrict__ perm, GaussRule g, double2 k, int nang,
                                                  const double* __restrict__ dirs, const double2* __restrict__ I,
                                                  size_t istride, double2* __restrict__ partial) {
    __shared__ double2 red[NA][3][4];
    const int a0 = blockIdx.y * NA;
    R3 rd[NA];
    int ang[NA];   // past the last direction: repeated, not stored
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        ang[a] = min(a0 + a, nang - 1);
        rd[a] = {dirs[3 * ang[a]], dirs[3 * ang[a] + 1], dirs[3 * ang[a] + 2]};
    }
    double2 V[NA][3];
#pragma unroll
    for (int a = 0; a < NA; ++a) V[a][0] = V[a][1] = V[a][2] = make_double2(0, 0);
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) {
        std::conditional_t<NA == 1, const RwgGeo, const RwgGeo&> G = geo[i];
        for (int q = 0; q < g.n; ++q) {
            const double wl = G.len * g.w[q];
            for (int side = 1; side >= 0; --side) {
                const R3 r = gpt(g, q, G.tri[side]);
                const R3 rho = scl3(side == 1 ? sub3(r, mk(G.vf[1])) : sub3(mk(G.vf[0]), r), wl);
#pragma unroll
                for (int a = 0; a < NA; ++a) {
                    double rp = dot3(r, rd[a]);
                    if (NA == 1) asm("" : "+v"(rp));
                    const double2 e = expmjk(make_double2(-k.x, -k.y), rp);   // e^{+jk r.p}
                    V[a][0] = cadd(V[a][0], cscale(e, rho.x));
                    V[a][1] = cadd(V[a][1], cscale(e, rho.y));
                    V[a][2] = cadd(V[a][2], cscale(e, rho.z));
                }
            }
        }
        const int r = perm[i];
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const double2* Ia = I + (size_t)ang[a] * istride;   // monostatic: every angle has its own current vector
            const double2 IJ = Ia[r];
            const R3 d = rd[a];
            const double2 v0 = V[a][0], v1 = V[a][1], v2 = V[a][2];
            const double2 dv = cadd(cadd(cscale(v0, d.x), cscale(v1, d.y)), cscale(v2, d.z));
            V[a][0] = cmul(csub(v0, cscale(dv, d.x)), IJ);
            V[a][1] = cmul(csub(v1, cscale(dv, d.y)), IJ);
            V[a][2] = cmul(csub(v2, cscale(dv, d.z)), IJ);
            if (pmchwt) {
                const double2 IM = Ia[N + r];
                V[a][0] = csub(V[a][0], cmul(csub(cscale(v2, d.y), cscale(v1, d.z)), IM));
                V[a][1] = csub(V[a][1], cmul(csub(cscale(v0, d.z), cscale(v2, d.x)), IM));
                V[a][2] = csub(V[a][2], cmul(csub(cscale(v1, d.x), cscale(v0, d.y)), IM));
            }
        }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double2 s = wave_sum(V[a][c]);
            if (lane == 0) red[a][c][wave] = s;
        }
    __syncthreads();
    if ((int)threadIdx.x < 3 * NA) {
        const int a = threadIdx.x / 3, c = threadIdx.x - 3 * a;
        const double2 s = cadd(cadd(red[a][c][0], red[a][c][1]), cadd(red[a][c][2], red[a][c][3]));
        if (a0 + a < nang) partial[((size_t)(a0 + a) * gridDim.x + blockIdx.x) * 3 + c] = s;
    }
}

void launch_farfield(hipStream_t st, int N, int pmchwt, const RwgGeo* geo, const int* perm, const GaussRule& g,
                     double2 k, int nang, const double* dirs, const double2* I, size_t istride, double2* partial,
                     int nblocks) {
    // four directions per thread from 16 workgroups per CU of one each, so that a
    // quarter of them still fills the chip.  Near the line the two are alike
    // (12,000 RWG: 84 directions one by one 57.6 us, 88 and 100 by fours 61.8 and
    // 62.6); below it one by one wins (60: 45.3), above it fours do (361: 189).
    if ((long long)nblocks * nang >= 4096)
        k_farfield<4><<<dim3(nblocks, (nang + 3) / 4), 256, 0, st>>>(N, pmchwt, geo, perm, g, k, nang, dirs, I, istride,
                                                                     partial);
    else
        k_farfield<1><<<dim3(nblocks, nang), 256, 0, st>>>(N, pmchwt, geo, perm, g, k, nang, dirs, I, istride, partial);
}

}  // namespace mlfma
