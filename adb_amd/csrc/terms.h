// terms.h - the barrier Hessian of one contact in a small orthonormal frame.
//
// Every squared distance of a contact is the minimum over the closest-point
// parameters beta of |g(beta, x)|^2 with g = sum_k gamma_k(beta) x_k, so with
// g = delta n at the minimum (n unit, gamma the weights there, E_i = dg/dbeta_i
// the edge vectors of the line or plane, n normal to them) the envelope
// theorem gives, for point displacements x_k = t_k + s_k n (t_k normal to n),
//     grad d = 2 delta gamma (x) n
//     Hess d = 2 [ |G|^2 - |P_E G + delta N*|^2 ],   G = sum_k gamma_k x_k,
// P_E the projection on span(E_i) and N* = sum_i E_i* (n . dE_i) with E_i* the
// dual basis.  With T the part of G in span(E), V the rest of its tangential
// part and sigma = gamma . s this is
//     Hess d = 2 [ sigma^2 + V^2 - 2 delta T . N* - delta^2 |N*|^2 ],
// so H = B1 Hess d + B2 grad d grad d^T acts on five coordinates only: the
// tangential ones tau_1, tau_2 (gamma / |gamma| (x) f_1, f_2) and the normal
// ones y in R^3 (Helmert basis of the point weights (x) n):
//     H = (2 B1 + 4 B2 delta^2) sigma^2 - 4 B1 delta (T_1 m_1 . s + T_2 m_2 . s)
//         - 2 B1 delta^2 ((m_1 . s)^2 + (m_2 . s)^2) + 2 B1 V^2
// with N* = (m_1 . s) f_1 + (m_2 . s) f_2.  Point-point: both tangents belong
// to V, m = 0.  Point-line: f_1 along the line, f_2 belongs to V, m_2 = 0.
// Point-plane and line-line: both tangents in span(E), V = 0.  The eigenvalues
// of the 12 x 12 Hessian are those of this 5 x 5 matrix (and zeros): its PSD
// projection costs a twelfth of that of the 9 x 9 matrix in the space of point
// differences.
#pragma once
#include "dmath.h"

namespace adb {

// two doubles loaded or stored by one 16-byte access at an address that is
// only known to be a double's (callers' arrays may start anywhere)
typedef double dd8 __attribute__((ext_vector_type(2), aligned(8)));

// Helmert basis of the complement of (1, 1, 1, 1) / 2 in R^4
#define HS2 0.70710678118654752440
#define HS6 0.40824829046386301637
#define HS12 0.28867513459481288225
__constant__ double kHel[3][4] = {{HS2, -HS2, 0.0, 0.0}, {HS6, HS6, -2.0 * HS6, 0.0}, {HS12, HS12, HS12, -3.0 * HS12}};

constexpr int MAX_SWEEPS = 15;
// Jacobi stops when the squared off-diagonal Frobenius norm is below this
// fraction of the total (off-diagonal entries ~1e-12 relative: rounding-level
// for the projected Hessian, and reachable in a few sweeps, unlike 1e-30,
// which sits at the FP64 noise floor of the rotations themselves)
constexpr double JACOBI_TOL = 1e-24;
// rotations of off-diagonal entries below JACOBI_SKIP * |A|_F are skipped: 36
// such entries add at most 36e-28 |A|_F^2 to the off-diagonal sum, far below
// the stop test, and late sweeps then cost little
constexpr double JACOBI_SKIP = 1e-14;
// Reciprocal square root from the hardware approximation, refined by two
// Newton steps (each doubles the correct bits).  The Jacobi rotation parameters
// need no correct rounding, and this chain is several times shorter than IEEE
// division and square root.
__device__ __forceinline__ double rsq_r(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    double e = fma(-h * y, y, 0.5); y = fma(y, e, y);
    e = fma(-h * y, y, 0.5); return fma(y, e, y);
}
// The same with one Newton step: where only the rotation angle depends on
// the value, an error there leaves a residual of that relative size in the
// annihilated entry (removed by the next sweep), not a non-orthogonal rotation.
__device__ __forceinline__ double rcp_r1(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    return fma(y, fma(-x, y, 1.0), y);
}
__device__ __forceinline__ double rsq_r1(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    return fma(y, fma(-(0.5 * x) * y, y, 0.5), y);
}
// Jacobi rotation annihilating a_pq (Golub and Van Loan, Algorithm 8.5.1):
// tau = (a_qq - a_pp) / (2 a_pq), t = sign(tau) / (|tau| + sqrt(1 + tau^2)),
// c = 1 / sqrt(1 + t^2), s = t c; after it a_pp' = a_pp - t a_pq, a_qq' = a_qq + t a_pq.
// t sets only the angle (one Newton step each); c keeps two, so that
// c^2 + s^2 = 1 to rounding and the accumulated rotations stay orthogonal.
__device__ __forceinline__ void jacobi_cs(double app, double aqq, double apq, double& c, double& s, double& t) {
    const double tau = (aqq - app) * (0.5 * rcp_r1(apq));
    if (fabs(tau) > 1e150) {
        t = 0.5 * rcp_r1(tau);
    } else {
        const double x = fma(tau, tau, 1.0);
        t = (tau >= 0 ? 1.0 : -1.0) * rcp_r1(fma(x, rsq_r1(x), fabs(tau)));      // x rsq(x) = sqrt(x)
    }
    c = rsq_r(fma(t, t, 1.0));
    s = t * c;
}

// packed upper-triangle index of an N x N symmetric matrix
template <int N> __host__ __device__ constexpr int PK_(int p, int q) {
    return p <= q ? p * N - p * (p - 1) / 2 + (q - p) : q * N - q * (q - 1) / 2 + (p - q);
}
// Cyclic Jacobi on a packed symmetric matrix A (registers, static indices)
// with the eigenvectors V (row-major N x N, registers); rotations of entries
// below JACOBI_SKIP |A|_F are skipped, and a scheduling barrier after each
// rotation bounds the live ranges.  Returns with the eigenvalues on A's diagonal.
template <int N>
__device__ __forceinline__ void jacobi_packed(double (&A)[N * (N + 1) / 2], double (&V)[N * N]) {
#pragma unroll
    for (int e = 0; e < N * N; e++) V[e] = (e % (N + 1) == 0) ? 1.0 : 0.0;
    for (int sweep = 0; sweep < MAX_SWEEPS; sweep++) {
        double off = 0.0, tot = 0.0;
#pragma unroll
        for (int p = 0; p < N; p++)
#pragma unroll
            for (int q = p; q < N; q++) {
                const double x = A[PK_<N>(p, q)] * A[PK_<N>(p, q)];
                if (p == q) tot += x; else { off += 2.0 * x; tot += 2.0 * x; }
            }
        if (off <= JACOBI_TOL * tot || off == 0.0) break;
        const double thr = JACOBI_SKIP * sqrt(tot);
#pragma unroll
        for (int p = 0; p < N - 1; p++)
#pragma unroll
            for (int q = p + 1; q < N; q++) {
                const double apq = A[PK_<N>(p, q)];
                if (fabs(apq) > thr) {
                    const double app = A[PK_<N>(p, p)], aqq = A[PK_<N>(q, q)];
                    double c, s, t;
                    jacobi_cs(app, aqq, apq, c, s, t);
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        if (k == p || k == q) continue;
                        const double akp = A[PK_<N>(k, p)], akq = A[PK_<N>(k, q)];
                        A[PK_<N>(k, p)] = fma(c, akp, -s * akq);
                        A[PK_<N>(k, q)] = fma(s, akp, c * akq);
                    }
                    A[PK_<N>(p, p)] = fma(-t, apq, app);
                    A[PK_<N>(q, q)] = fma(t, apq, aqq);
                    A[PK_<N>(p, q)] = 0.0;
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const double vkp = V[N * k + p], vkq = V[N * k + q];
                        V[N * k + p] = fma(c, vkp, -s * vkq);
                        V[N * k + q] = fma(s, vkp, c * vkq);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
    }
}

// Feature pair of a distance type as point slots: PP (a, b), PL (point a,
// line b c), PLANE (all four).  Slots are 0..3; two bits each.
__device__ __forceinline__ void feature_slots(int is_ee, int type, int& kind, int& a, int& b, int& c) {
    // entries a | b << 2 | c << 4 for the types below the PLANE one
    constexpr unsigned long long PT = 0x04ull | 0x08ull << 6 | 0x0cull << 12 | 0x24ull << 18 | 0x38ull << 24 | 0x1cull << 30;
    constexpr unsigned long long EE = 0x08ull | 0x0cull << 6 | 0x09ull << 12 | 0x0dull << 18 | 0x12ull << 24 | 0x13ull << 30 |
                                      0x38ull << 36 | 0x39ull << 42;
    const unsigned npp = is_ee ? 4 : 3, npl = is_ee ? 8 : 6, t = (unsigned)type;    // any other value: PLANE
    kind = t < npp ? K_PP : (t < npl ? K_PL : K_PLANE);
    const unsigned v = (unsigned)((is_ee ? EE : PT) >> (6 * min(t, 7u))) & 63u;
    a = v & 3; b = (v >> 2) & 3; c = (v >> 4) & 3;
}
__device__ __forceinline__ d3 pick(d3 p0, d3 p1, d3 p2, d3 p3, int k) {
    return k == 0 ? p0 : (k == 1 ? p1 : (k == 2 ? p2 : p3));
}
__device__ __forceinline__ d3 unit(d3 a) { double l = sqrt(sqn(a)); return mk(a.x / l, a.y / l, a.z / l); }

// The frame of a contact: separation sum_k gam_k x_k = delta n, tangents f1,
// f2, and the weights of the two normal functionals m1, m2 (see above).  f1 is
// the edge (PL), the first edge (PLANE) or any tangent (PP).  (Friction has its
// own basis, of the reference's signs: friction_frame.)
struct Frame {
    int kind;
    unsigned in;                 // bit k: point k takes part
    d3 n, f1, f2;
    double gam[4], m1[4], m2[4];
    double delta, gn;            // gn = |gam|
};
__device__ __forceinline__ void contact_frame(int is_ee, int type, d3 P0, d3 P1, d3 P2, d3 P3, Frame& F) {
    int kind, a, b, c;
    feature_slots(is_ee, type, kind, a, b, c);
    F.kind = kind;
    if (kind == K_PLANE) {
        const d3 e1 = is_ee ? P1 - P0 : P2 - P1, e2 = is_ee ? P3 - P2 : P3 - P1;
        const d3 w = is_ee ? P0 - P2 : P0 - P1;
        const d3 nv = cross(e1, e2);
        const double G = sqn(nv), l1 = sqrt(sqn(e1)), gl = sqrt(G);
        const double iG = 1.0 / G, ig = 1.0 / gl, i1 = 1.0 / l1;
        F.n = ig * nv;
        F.f1 = i1 * e1;
        F.f2 = cross(F.n, F.f1);
        F.delta = dot(w, F.n);
        const double x = dot(w, cross(e2, nv)) * iG, y = dot(w, cross(e1, nv)) * iG;
        // N* = e1* N1 + e2* N2: e1* = (1, -a / b) / l1, e2* = (0, 1 / b) in (f1, f2), e2 = (a, b)
        const double ib = l1 * ig;                       // b = |e1 x e2| / |e1|
        const double ab = dot(e2, F.f1) * i1 * ib;       // a / (l1 b)
        if (is_ee) {
            const double l0 = -x, l2 = -y;               // closest-point parameters on the edges
            F.gam[0] = 1.0 - l0; F.gam[1] = l0; F.gam[2] = -(1.0 - l2); F.gam[3] = -l2;
            F.m1[0] = -i1; F.m1[1] = i1; F.m1[2] = 0.0; F.m1[3] = 0.0;
            F.m2[0] = ab; F.m2[1] = -ab; F.m2[2] = -ib; F.m2[3] = ib;
        } else {
            F.gam[0] = 1.0; F.gam[1] = x - y - 1.0; F.gam[2] = -x; F.gam[3] = y;
            F.m1[0] = 0.0; F.m1[1] = -i1; F.m1[2] = i1; F.m1[3] = 0.0;
            F.m2[0] = 0.0; F.m2[1] = ab - ib; F.m2[2] = -ab; F.m2[3] = ib;
        }
        F.in = 15u;
    } else {
        const d3 A = pick(P0, P1, P2, P3, a), Bp = pick(P0, P1, P2, P3, b), C = pick(P0, P1, P2, P3, c);
        d3 w = A - Bp;
        double t = 0.0, il = 0.0;
        if (kind == K_PL) {
            // the perpendicular part of w, subtracted twice: orthogonal to the
            // edge to rounding also when delta is far below the edge length
            const d3 e = C - Bp;
            const double ie = 1.0 / sqn(e);
            t = dot(w, e) * ie;
            w = w - t * e;
            const double t2 = dot(w, e) * ie;
            w = w - t2 * e;
            t += t2;
            il = sqrt(ie);
            F.f1 = il * e;
        }
        const double dd = sqn(w);
        F.delta = sqrt(dd);
        if (dd > 0.0) {
            F.n = (1.0 / F.delta) * w;
        } else if (kind == K_PL) {      // touching: any normal of the edge
            const d3 ax = fabs(F.f1.x) < 0.5 ? mk(1, 0, 0) : mk(0, 1, 0);
            F.n = unit(cross(F.f1, ax));
        } else {
            F.n = mk(1, 0, 0);
        }
        if (kind == K_PL) {
            F.f2 = cross(F.f1, F.n);
        } else {
            // the larger of x x n and y x n
            const d3 cx = mk(0.0, -F.n.z, F.n.y), cy = mk(F.n.z, 0.0, -F.n.x);
            F.f1 = unit(sqn(cx) > sqn(cy) ? cx : cy);
            F.f2 = cross(F.n, F.f1);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const bool ka = k == a, kb = k == b, kc = kind == K_PL && k == c;
            F.gam[k] = ka ? 1.0 : (kb ? t - 1.0 : (kc ? -t : 0.0));
            F.m1[k] = kb ? -il : (kc ? il : 0.0);
            F.m2[k] = 0.0;
        }
        F.in = (1u << a) | (1u << b) | (kind == K_PL ? 1u << c : 0u);
    }
    F.gn = sqrt(((F.gam[0] * F.gam[0] + F.gam[1] * F.gam[1]) + F.gam[2] * F.gam[2]) + F.gam[3] * F.gam[3]);
}
// the three Helmert components of a weight vector over the four points
__device__ __forceinline__ void helmert(const double v[4], double o[3]) {
    o[0] = HS2 * (v[0] - v[1]);
    o[1] = HS6 * ((v[0] + v[1]) - 2.0 * v[2]);
    o[2] = HS12 * (((v[0] + v[1]) + v[2]) - 3.0 * v[3]);
}
// the weights of Helmert components y
__device__ __forceinline__ void unhelmert(const double y[3], unsigned in, double v[4]) {
    const double a = HS2 * y[0], b = HS6 * y[1], c = HS12 * y[2];
    v[0] = (a + b) + c; v[1] = (b + c) - a; v[2] = c - 2.0 * b; v[3] = -3.0 * c;
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = (in >> k) & 1u ? v[k] : 0.0;
}
// H in the frame's five coordinates (tau1, tau2, y), packed
__device__ __forceinline__ void frame_matrix(const Frame& F, double B1, double B2, double (&M)[15]) {
    double g[3], m1[3], m2[3];
    helmert(F.gam, g); helmert(F.m1, m1); helmert(F.m2, m2);
    const double dd = F.delta * F.delta, A = 2.0 * B1 + 4.0 * B2 * dd;
    const double kc = -2.0 * B1 * F.delta * F.gn, kn = -2.0 * B1 * dd, kt = 2.0 * B1 * F.gn * F.gn;
    M[PK_<5>(0, 0)] = F.kind == K_PP ? kt : 0.0;
    M[PK_<5>(0, 1)] = 0.0;
    M[PK_<5>(1, 1)] = F.kind != K_PLANE ? kt : 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        M[PK_<5>(0, 2 + i)] = kc * m1[i];
        M[PK_<5>(1, 2 + i)] = kc * m2[i];
#pragma unroll
        for (int j = i; j < 3; j++) M[PK_<5>(2 + i, 2 + j)] = A * g[i] * g[j] + kn * (m1[i] * m1[j] + m2[i] * m2[j]);
    }
}

// V diag(w) V^T of the eigenpairs left by jacobi_packed, negative eigenvalues dropped
template <int N>
__device__ __forceinline__ void project_packed(double (&A)[N * (N + 1) / 2], const double (&V)[N * N]) {
    double w[N];
#pragma unroll
    for (int k = 0; k < N; k++) w[k] = fmax(A[PK_<N>(k, k)], 0.0);
#pragma unroll
    for (int p = 0; p < N; p++)
#pragma unroll
        for (int q = p; q < N; q++) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < N; k++) s += V[N * p + k] * w[k] * V[N * q + k];
            A[PK_<N>(p, q)] = s;
        }
}

// Mollified edge-edge contact, energy m(x) B(d): its Hessian in the space of
// point differences, index 3 a + i (Helmert row a, component i), packed.
// x = |u x w|^2 with u = P1 - P0, w = P3 - P2; m' and m'' the derivatives.
struct Mollifier { double m, m1, m2; CrossNorm cn; };
__device__ __forceinline__ bool mollifier(double eps_x, d3 P0, d3 P1, d3 P2, d3 P3, Mollifier& q) {
    const double eps = eps_x * sqn(P0 - P1) * sqn(P2 - P3);
    q.cn.init(P1 - P0, P3 - P2);
    const double x = q.cn.value();
    q.m = 1.0; q.m1 = 0.0; q.m2 = 0.0;
    if (!(x < eps)) return false;
    q.m = (-x / eps + 2) * x / eps;
    q.m1 = 2.0 / eps - 2.0 * x / (eps * eps);
    q.m2 = -2.0 / (eps * eps);
    return true;
}
__device__ __forceinline__ void mollified_matrix(const Frame& F, const Mollifier& q, double B0, double B1, double B2,
                                                 double (&K)[45]) {
    double M[15];
    frame_matrix(F, B1, B2, M);
    double gt[3], gh[3];
    helmert(F.gam, gt);
    const double ign = 1.0 / F.gn;
#pragma unroll
    for (int a = 0; a < 3; a++) gh[a] = gt[a] * ign;          // unit tangential weights
    // Helmert rows of u and w
    const double Cu[3] = {-2.0 * HS2, 0.0, 0.0}, Cw[3] = {0.0, 2.0 * HS6, -4.0 * HS12};
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int b = a; b < 3; b++)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    if (3 * a + i > 3 * b + j) continue;
                    const double ni = cmp(F.n, i), nj = cmp(F.n, j);
                    const double f1i = cmp(F.f1, i), f1j = cmp(F.f1, j), f2i = cmp(F.f2, i), f2j = cmp(F.f2, j);
                    const double tt = M[PK_<5>(0, 0)] * f1i * f1j + M[PK_<5>(1, 1)] * f2i * f2j;
                    const double hb = M[PK_<5>(0, 2 + b)] * f1i + M[PK_<5>(1, 2 + b)] * f2i;
                    const double ha = M[PK_<5>(0, 2 + a)] * f1j + M[PK_<5>(1, 2 + a)] * f2j;
                    const double hd = gh[a] * gh[b] * tt + gh[a] * hb * nj + gh[b] * ni * ha + M[PK_<5>(2 + a, 2 + b)] * ni * nj;
                    const double gxi = Cu[a] * q.cn.grad(0, i) + Cw[a] * q.cn.grad(1, i);
                    const double gxj = Cu[b] * q.cn.grad(0, j) + Cw[b] * q.cn.grad(1, j);
                    const double hx = Cu[a] * (Cu[b] * q.cn.hess(0, i, 0, j) + Cw[b] * q.cn.hess(0, i, 1, j)) +
                                      Cw[a] * (Cu[b] * q.cn.hess(1, i, 0, j) + Cw[b] * q.cn.hess(1, i, 1, j));
                    const double gdi = 2.0 * F.delta * gt[a] * ni, gdj = 2.0 * F.delta * gt[b] * nj;
                    K[PK_<9>(3 * a + i, 3 * b + j)] = q.m * hd + B1 * q.m1 * (gxi * gdj + gdi * gxj) +
                                                      B0 * (q.m2 * gxi * gxj + q.m1 * hx);
                }
}

} // namespace adb
