// contact.hip - PT / EE / VG contact terms on gfx950.
//
// Replaces IPC::ipc_hess_pt_12x12 / ipc_hess_ee_12x12 (model/core_ipc.cpp:21-83),
// project_to_psd (model/psd.h:9-33), pt_uktk / ee_uktk (model/pt_ipc.cpp:22-107,
// model/ee_ipc.cpp:21-118), friction (model/friction.cpp:15-47), the J^T H J body
// mapping (model/pt_ipc.cpp:153-169, model/ee_ipc.cpp:175-192) and the VG term
// (model/vg_ipc.cpp:12-30, model/abd.cpp:380-401).
//
// World path (contact_terms): k_contact_classify computes each contact's
// distance type, squared distance and class, the dimension D = 3 n of the
// translation-free space of the n + 1 points it involves, and appends it to
// that class's list; then one thread per contact:
//   class 1 (two points, D = 3): closed-form projection (k_contact_small<1>);
//   class 2 (three points, D = 6): record fields (k_contact_scalars2) and the
//     projection, 3 x 3 in the contact's frame (k_contact_pk2, side stream);
//   class 3 (point-plane, edge-edge interior, D = 9): the whole record, 5 x 5
//     in the contact's frame (k_contact_plane, side stream);
//   class 4 (mollified edge pairs, D = 9): the 9 x 9 matrix into the record,
//     then cyclic Jacobi in registers (k_contact_c3r, nine threads per contact
//     building the matrix and a tenth the other record fields, then
//     k_contact_psd9, one thread per contact, on a side stream).
// Each contact writes a compact body-space record (world.h) that the
// assembly expands into its four 12 x 12 blocks; the class 1 and class 2
// record kernels stage it per wavefront in LDS and store it cooperatively
// (Stage, stage_flush).
//
// PSD projection: every barrier and mollifier term depends on the points only
// through differences, so the Hessian annihilates rigid translations.  With
// Q = h (x) I3, h the Helmert basis of the complement of (1, ..., 1) over the
// contact's points, H = Q^T (Q H Q^T) Q and the projection onto the PSD cone
// is Q^T P(Q H Q^T) Q: a D x D symmetric eigenproblem.  Both paths always
// rebuild V diag(max(w, 0)) V^T; where the reference returns a Hessian whose
// eigenvalues are all >= 0 unchanged (its test sees the rounding-level
// eigenvalues of the translations) that equals it within the Jacobi tolerance.
//
// Kernel-level API (the abdtk functions): k_hess_api, one thread per contact
// in the five-coordinate frame of terms.h; mollified edge pairs in
// k_hess_moll.  Against the 16-lane groups with a 9 x 9 Jacobi in LDS that
// they replaced (a barrier per round of rotations): 1021 PT contacts 114 ->
// 22 us a call, 2e5 EE contacts (a tenth mollified) 4458 -> 200 us.
#include <cstdio>
#include <algorithm>
#include <cstring>
#include "dmath.h"
#include "staging.h"
#include "terms.h"
#include "world.h"

namespace adb {

struct KParams {
    double d_hat, kappa, eps_x;
    int psd;
    double mu, eps_v, max_uk;
    int pt_fric, ee_fric;
};

// ---------------------------------------------------------------- barrier Hessian column
// Geometry and barrier scalars of a mollified edge pair (no private arrays
// indexed by lane-dependent values).
struct Geo {
    d3 p0, p1, p2, p3;
    int type;
    double d, B0, B1, B2;
    double m, m1, m2;       // EE mollifier m(x) and dm/dx, d2m/dx2
    RedMap map;
    RedDist rd;
    CrossNorm mc;           // x = |(a1 - a0) x (b1 - b0)|^2
};

__device__ __forceinline__ void geo_init(Geo& G, const KParams& kp) {
    const double dh = kp.d_hat, ka = kp.kappa;
    G.B1 = barrier_d1(G.d, dh, ka);
    G.B2 = barrier_d2(G.d, dh, ka);
    G.B0 = barrier(G.d, dh, ka);
    G.map = ee_map(G.type);
    d3 r0 = mk(0, 0, 0), r1 = mk(0, 0, 0), r2 = mk(0, 0, 0);
    const d3 p0 = G.p0, p1 = G.p1, p2 = G.p2, p3 = G.p3;
    switch (G.type) {
    case EA0_EB0: r0 = p0 - p2; break;
    case EA0_EB1: r0 = p0 - p3; break;
    case EA1_EB0: r0 = p1 - p2; break;
    case EA1_EB1: r0 = p1 - p3; break;
    case EA_EB0:  r0 = p0 - p2; r1 = p1 - p2; break;
    case EA_EB1:  r0 = p0 - p3; r1 = p1 - p3; break;
    case EA0_EB:  r0 = p2 - p0; r1 = p3 - p0; break;
    case EA1_EB:  r0 = p2 - p1; r1 = p3 - p1; break;
    default:      r0 = p2 - p0; r1 = p1 - p0; r2 = p3 - p2; break;
    }
    G.rd.init(G.map.kind, r0, r1, r2);
    G.m = 1.0; G.m1 = 0.0; G.m2 = 0.0;
    const double eps = kp.eps_x * sqn(p0 - p1) * sqn(p2 - p3);
    G.mc.init(p1 - p0, p3 - p2);
    const double x = G.mc.value();
    if (x < eps) {
        G.m = (-x / eps + 2) * x / eps;
        G.m1 = 2.0 / eps - 2.0 * x / (eps * eps);
        G.m2 = -2.0 / (eps * eps);
    }
}
// point-space gradient entry (k, i) of d, and of the mollifier
__device__ __forceinline__ double grad_d(const Geo& G, int k, int i) {
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < 3; m++)
        if (m < G.map.nr) s += red_sign(G.map, m, k) * cmp(G.rd.g[m], i);
    return s;
}
__device__ __forceinline__ double grad_m(const Geo& G, int k, int i) {
    if (G.m2 == 0.0) return 0.0;
    // x depends on y = p1 - p0 (points 1, 0) and z = p3 - p2 (points 3, 2)
    const double sy = (k == 1 ? 1.0 : 0.0) - (k == 0 ? 1.0 : 0.0);
    const double sz = (k == 3 ? 1.0 : 0.0) - (k == 2 ? 1.0 : 0.0);
    return G.m1 * (sy * G.mc.grad(0, i) + sz * G.mc.grad(1, i));
}
// vertex-space gradient entry j = (point, component) < 12 (model/core_ipc.cpp:36-43,70-80)
__device__ __forceinline__ double barrier_grad(const Geo& G, int j) {
    const int l = j / 3, c = j % 3;
    const double gdj = grad_d(G, l, c);
    return G.m * gdj * G.B1 + grad_m(G, l, c) * G.B0;
}

// ---------------------------------------------------------------- friction setup
__device__ __forceinline__ void basis_pp(d3 p0, d3 p1, d3& c0, d3& c1) {
    d3 d = p1 - p0;
    d3 cx = cross(mk(1, 0, 0), d), cy = cross(mk(0, 1, 0), d);
    if (sqn(cx) > sqn(cy)) { c0 = unit(cx); c1 = unit(cross(d, cx)); }
    else { c0 = unit(cy); c1 = unit(cross(d, cy)); }
}
__device__ __forceinline__ void basis_pe(d3 p, d3 e0, d3 e1, d3& c0, d3& c1) { d3 e = e1 - e0; c0 = unit(e); c1 = unit(cross(e, p - e0)); }
__device__ __forceinline__ double pe_closest(d3 p, d3 e0, d3 e1) { d3 e = e1 - e0; return dot(p - e0, e) / sqn(e); }
__device__ __forceinline__ void solve2(double m00, double m01, double m11, double r0, double r1, double& x, double& y) {
    double det = m00 * m11 - m01 * m01;
    x = (r0 * m11 - m01 * r1) / det;
    y = (m00 * r1 - m01 * r0) / det;
}
// coefficients g0..g3 of the relative tangential displacement sum_k g_k x_k
// and the tangent basis (c0, c1) (model/pt_ipc.cpp:31-103, model/ee_ipc.cpp:38-110)
__device__ __forceinline__ void friction_frame(int is_ee, int type, d3 P0, d3 P1, d3 P2, d3 P3,
                                               double& g0, double& g1, double& g2, double& g3, d3& c0, d3& c1) {
    if (!is_ee) {
        double t0, t1, t2;
        switch (type) {
        case P_T0: basis_pp(P0, P1, c0, c1); t0 = 1; t1 = 0; t2 = 0; break;
        case P_T1: basis_pp(P0, P2, c0, c1); t0 = 0; t1 = 1; t2 = 0; break;
        case P_T2: basis_pp(P0, P3, c0, c1); t0 = 0; t1 = 0; t2 = 1; break;
        case P_E0: { double l = pe_closest(P0, P1, P2); t0 = 1 - l; t1 = l; t2 = 0; basis_pe(P0, P1, P2, c0, c1); } break;
        case P_E1: { double l = pe_closest(P0, P2, P3); t0 = 0; t1 = 1 - l; t2 = l; basis_pe(P0, P2, P3, c0, c1); } break;
        case P_E2: { double l = pe_closest(P0, P3, P1); t0 = l; t1 = 0; t2 = 1 - l; basis_pe(P0, P3, P1, c0, c1); } break;
        default: {
            d3 b0 = P2 - P1, b1 = P3 - P1, r = P0 - P1;
            double x, y; solve2(dot(b0, b0), dot(b0, b1), dot(b1, b1), dot(b0, r), dot(b1, r), x, y);
            t0 = 1 - x - y; t1 = x; t2 = y;
            d3 n = cross(b0, b1);
            c0 = unit(b0); c1 = unit(cross(n, b0));
        }
        }
        g0 = -1.0; g1 = t0; g2 = t1; g3 = t2;
    } else {
        double l0, l1;
        switch (type) {
        case EA0_EB0: basis_pp(P0, P2, c0, c1); l0 = 0; l1 = 0; break;
        case EA0_EB1: basis_pp(P0, P3, c0, c1); l0 = 0; l1 = 1; break;
        case EA1_EB0: basis_pp(P1, P2, c0, c1); l0 = 1; l1 = 0; break;
        case EA1_EB1: basis_pp(P1, P3, c0, c1); l0 = 1; l1 = 1; break;
        case EA_EB0: l0 = pe_closest(P2, P0, P1); l1 = 0; basis_pe(P2, P0, P1, c0, c1); break;
        case EA_EB1: l0 = pe_closest(P3, P0, P1); l1 = 1; basis_pe(P3, P0, P1, c0, c1); break;
        case EA0_EB: l0 = 0; l1 = pe_closest(P0, P2, P3); basis_pe(P0, P2, P3, c0, c1); break;
        case EA1_EB: l0 = 1; l1 = pe_closest(P1, P2, P3); basis_pe(P1, P2, P3, c0, c1); break;
        default: {
            d3 w = P0 - P2, ea = P1 - P0, eb = P3 - P2;
            solve2(sqn(ea), -dot(eb, ea), sqn(eb), -dot(w, ea), dot(w, eb), l0, l1);
            d3 n = cross(ea, eb);
            c0 = unit(ea); c1 = unit(cross(n, ea));
        }
        }
        l0 = fmax(fmin(1.0, l0), 0.0);
        l1 = fmax(fmin(1.0, l1), 0.0);
        g0 = -(1 - l0); g1 = -l0; g2 = 1 - l1; g3 = l1;
    }
}

// 2x2 symmetric PSD projection (closed-form eigenpairs)
__device__ __forceinline__ void psd2(double a, double b, double c, double& o0, double& o1, double& o2) {
    double h = 0.5 * (a + c), dlt = 0.5 * (a - c);
    double r = sqrt(dlt * dlt + b * b);
    double lmin = h - r, lmax = h + r;
    if (lmin >= 0.0) { o0 = a; o1 = b; o2 = c; return; }
    if (lmax <= 0.0) { o0 = 0; o1 = 0; o2 = 0; return; }
    double vx, vy;
    if (dlt >= 0) { vx = lmax - c; vy = b; } else { vx = b; vy = lmax - a; }
    double n = sqrt(vx * vx + vy * vy);
    if (n == 0.0) { vx = 1; vy = 0; } else { vx /= n; vy /= n; }
    o0 = lmax * vx * vx; o1 = lmax * vx * vy; o2 = lmax * vy * vy;
}
// friction 2x2 middle matrix M (model/friction.cpp:53-74) and force scale
__device__ __forceinline__ void friction_M(double u0, double u1, double lam, const KParams& kp, double& fs, double M[3]) {
    double u = sqrt(u0 * u0 + u1 * u1);
    double f1 = f1_over_x(u, kp.eps_v);
    fs = kp.mu * lam * f1;
    if (u >= kp.eps_v) {
        double k = kp.mu * lam * f1 / (u * u);
        double t0 = -u1, t1 = u0;
        M[0] = k * t0 * t0; M[1] = k * t0 * t1; M[2] = k * t1 * t1;
    } else if (u <= kp.max_uk) {
        double k = kp.mu * lam * f1;
        M[0] = k; M[1] = 0; M[2] = k;
    } else {
        double k = (-1.0 / (kp.eps_v * kp.eps_v)) / u;
        double m0 = (k * u0 * u0 + f1) * kp.mu * lam, m1 = (k * u1 * u0) * kp.mu * lam, m2 = (k * u1 * u1 + f1) * kp.mu * lam;
        psd2(m0, m1, m2, M[0], M[1], M[2]);
    }
}

// ---------------------------------------------------------------- kernel-level API
// H and g of IPC::ipc_hess_{pt,ee}_12x12 for n independent inputs, one thread
// each: the Hessian in the contact's five-coordinate frame (terms.h),
// projected there by a 5 x 5 Jacobi in registers, and expanded to the 12 x 12
// blocks as it is stored (column by column, 16-byte stores: a lane's column
// is 96 consecutive bytes).  Bound by the 1.3 KB stored per contact for large
// n, by the Jacobi's dependent chain for small n (64-lane workgroups, so that
// a few contacts spread over the CUs).  Mollified edge pairs are left to
// k_hess_moll.
__device__ __forceinline__ void load_points(const double* __restrict__ x, int e, d3& P0, d3& P1, d3& P2, d3& P3) {
    const dd8* p = reinterpret_cast<const dd8*>(x + 12 * (size_t)e);
    dd8 v[6];
#pragma unroll
    for (int k = 0; k < 6; k++) v[k] = p[k];
    P0 = mk(v[0].x, v[0].y, v[1].x); P1 = mk(v[1].y, v[2].x, v[2].y);
    P2 = mk(v[3].x, v[3].y, v[4].x); P3 = mk(v[4].y, v[5].x, v[5].y);
}
template <int IS_EE>
__global__ __launch_bounds__(64) void k_hess_api(KParams kp, int n, const double* __restrict__ x, const int* __restrict__ type,
                                                 const double* __restrict__ dist, double* __restrict__ H, double* __restrict__ g,
                                                 double* __restrict__ moll) {
    const int e = blockIdx.x * 64 + threadIdx.x;
    if (e >= n) return;
    d3 P0, P1, P2, P3;
    load_points(x, e, P0, P1, P2, P3);
    if (IS_EE) {
        Mollifier q;
        if (mollifier(kp.eps_x, P0, P1, P2, P3, q)) return;
        if (moll) moll[e] = 1.0;
    }
    const double d = dist[e];
    const double B1 = barrier_d1(d, kp.d_hat, kp.kappa), B2 = barrier_d2(d, kp.d_hat, kp.kappa);
    Frame F;
    contact_frame(IS_EE, type[e], P0, P1, P2, P3, F);
    double M[15];
    frame_matrix(F, B1, B2, M);
    if (kp.psd) {
        double V[25];
        jacobi_packed<5>(M, V);
        project_packed<5>(M, V);
    }
    const double gs = 2.0 * B1 * F.delta;
    double* ge = g + 12 * (size_t)e;
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int i = 0; i < 3; i++) ge[3 * k + i] = gs * F.gam[k] * cmp(F.n, i);
    // entry ((k, i), (l, j)) = gh_k gh_l T_ij + gh_k h_l,i n_j + n_i gh_l h_k,j + N_kl n_i n_j:
    // T the tangential 3 x 3 matrix, h_l = sum_t M(t, y) (Q_l) f_t, N = Q M(y, y) Q^T
    double gh[4], N[4][4], T[6];
    d3 h[4];
    const double ign = 1.0 / F.gn;
    double c1[4], c2[4];
    {
        const double y1[3] = {M[PK_<5>(0, 2)], M[PK_<5>(0, 3)], M[PK_<5>(0, 4)]};
        const double y2[3] = {M[PK_<5>(1, 2)], M[PK_<5>(1, 3)], M[PK_<5>(1, 4)]};
        unhelmert(y1, F.in, c1);
        unhelmert(y2, F.in, c2);
        double R[3][4];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const double ya[3] = {M[PK_<5>(2 + a, 2)], M[PK_<5>(2 + a, 3)], M[PK_<5>(2 + a, 4)]};
            unhelmert(ya, F.in, R[a]);
        }
#pragma unroll
        for (int l = 0; l < 4; l++) {
            const double col[3] = {R[0][l], R[1][l], R[2][l]};
            unhelmert(col, F.in, N[l]);
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        gh[k] = F.gam[k] * ign;
        h[k] = c1[k] * F.f1 + c2[k] * F.f2;
    }
    {
        const double a = M[PK_<5>(0, 0)], b = M[PK_<5>(0, 1)], c = M[PK_<5>(1, 1)];
        int u = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = i; j < 3; j++) {
                const double f1i = cmp(F.f1, i), f1j = cmp(F.f1, j), f2i = cmp(F.f2, i), f2j = cmp(F.f2, j);
                T[u++] = a * f1i * f1j + b * (f1i * f2j + f2i * f1j) + c * f2i * f2j;
            }
    }
    dd8* He = reinterpret_cast<dd8*>(H + 144 * (size_t)e);
#pragma unroll
    for (int l = 0; l < 4; l++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const double nj = cmp(F.n, j);
            double col[12];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const double hkj = cmp(h[k], j);
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const double Tij = T[PK_<3>(i, j)];
                    col[3 * k + i] = gh[k] * fma(gh[l], Tij, cmp(h[l], i) * nj) + cmp(F.n, i) * fma(gh[l], hkj, N[k][l] * nj);
                }
            }
#pragma unroll
            for (int r = 0; r < 6; r++) He[6 * (3 * l + j) + r] = dd8{col[2 * r], col[2 * r + 1]};
        }
}

// The mollified edge pairs of the same call: each 64-lane workgroup scans
// `per` contacts, gathers the mollified ones in LDS, then one thread each
// builds and projects the 9 x 9 matrix in the space of point differences (a
// 9 x 9 Jacobi in registers; one wavefront per SIMD).  A kernel of its own:
// with its registers in k_hess_api every contact would run at a quarter of
// the occupancy, and a wavefront with one mollified lane would wait for it.
constexpr int HM_PER = 1024;
__global__ __launch_bounds__(64) void k_hess_moll(KParams kp, int n, int per, const double* __restrict__ x,
                                                  const int* __restrict__ type, const double* __restrict__ dist,
                                                  double* __restrict__ H, double* __restrict__ g, double* __restrict__ moll) {
    __shared__ int list[HM_PER];
    const int lane = threadIdx.x, e0 = blockIdx.x * per, e1 = min(n, e0 + per);
    int cnt = 0;
    for (int b = e0; b < e1; b += 64) {
        bool on = false;
        if (b + lane < e1) {
            d3 P0, P1, P2, P3;
            load_points(x, b + lane, P0, P1, P2, P3);
            Mollifier q;
            on = mollifier(kp.eps_x, P0, P1, P2, P3, q);
        }
        const unsigned long long m = __ballot(on);
        if (on) list[cnt + __popcll(m & ((1ull << lane) - 1ull))] = b + lane;
        cnt += __popcll(m);
    }
    __syncthreads();
    for (int i = lane; i < cnt; i += 64) {
        const int e = list[i];
        d3 P0, P1, P2, P3;
        load_points(x, e, P0, P1, P2, P3);
        Mollifier q;
        mollifier(kp.eps_x, P0, P1, P2, P3, q);
        const double d = dist[e];
        const double B0 = barrier(d, kp.d_hat, kp.kappa), B1 = barrier_d1(d, kp.d_hat, kp.kappa), B2 = barrier_d2(d, kp.d_hat, kp.kappa);
        double K[45];
        {
            Frame F;
            contact_frame(1, type[e], P0, P1, P2, P3, F);
            mollified_matrix(F, q, B0, B1, B2, K);
            const double gs = 2.0 * B1 * q.m * F.delta, gm = B0 * q.m1;
            double* ge = g + 12 * (size_t)e;
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const double gx = k < 2 ? q.cn.grad(0, c) : q.cn.grad(1, c);
                    ge[3 * k + c] = gs * F.gam[k] * cmp(F.n, c) + (k == 1 || k == 3 ? gm : -gm) * gx;
                }
            if (moll) moll[e] = q.m;
        }
        if (kp.psd) {
            double V[81];
            jacobi_packed<9>(K, V);
            project_packed<9>(K, V);
        }
        dd8* He = reinterpret_cast<dd8*>(H + 144 * (size_t)e);
        // entry ((k, i), (l, j)) = sum_ab Hel[a][k] K(3 a + i, 3 b + j) Hel[b][l]
#pragma unroll
        for (int l = 0; l < 4; l++)
#pragma unroll
            for (int j = 0; j < 3; j++) {
                double col[12];
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    double t[3], v[4];
#pragma unroll
                    for (int a = 0; a < 3; a++) {
                        const double r[3] = {K[PK_<9>(3 * a + i, j)], K[PK_<9>(3 * a + i, 3 + j)], K[PK_<9>(3 * a + i, 6 + j)]};
                        double o[4];
                        unhelmert(r, 15u, o);
                        t[a] = o[l];
                    }
                    unhelmert(t, 15u, v);
#pragma unroll
                    for (int k = 0; k < 4; k++) col[3 * k + i] = v[k];
                }
#pragma unroll
                for (int r = 0; r < 6; r++) He[6 * (3 * l + j) + r] = dd8{col[2 * r], col[2 * r + 1]};
            }
    }
}

// ---------------------------------------------------------------- world contact terms
// Contact ids: the four world vertex ids of contact `cid` (PT: point, face
// vertices; EE: edge a, edge b).  Points 0..nside0-1 belong to body I.
struct WorldArgs {
    KParams kp;
    int n_pt, n_ee;
    const int4* pt; const int4* ee;
    const int* voff; const int* foff; const int* eoff; const int* face; const int* edge;
    const double* X; const double* Xs; const double* xbar; const double* mass;
    int* ctype; double* cdist; int* ccls; int* list; int* list3; int* counts;
    double* rec; double* tk; double* lam;
};

// R[R_D] = D + 100 (dynamic(I) + 2 dynamic(J)): the assembly drops the
// blocks of static bodies (mass < 0, model/assemble_matrices.cpp:43-58)
__device__ __forceinline__ double rec_code(const WorldArgs& a, int cid, int D) {
    const int4 c = cid < a.n_pt ? a.pt[cid] : a.ee[cid - a.n_pt];
    const int di = a.mass[c.x] > 0.0 ? 1 : 0, dj = a.mass[c.z] > 0.0 ? 1 : 0;
    return (double)(D + 100 * (di + 2 * dj));
}
__device__ __forceinline__ bool contact_ids(const WorldArgs& a, int cid, int& id0, int& id1, int& id2, int& id3) {
    if (cid < a.n_pt) {
        const int4 c = a.pt[cid];
        const int f = a.foff[c.z] + c.w;
        id0 = a.voff[c.x] + c.y; id1 = a.face[3 * f]; id2 = a.face[3 * f + 1]; id3 = a.face[3 * f + 2];
        return false;
    }
    const int4 c = a.ee[cid - a.n_pt];
    const int ea = a.eoff[c.x] + c.y, eb = a.eoff[c.z] + c.w;
    id0 = a.edge[2 * ea]; id1 = a.edge[2 * ea + 1]; id2 = a.edge[2 * eb]; id3 = a.edge[2 * eb + 1];
    return true;
}

// Class of an active contact by the points its barrier depends on:
// 1 = two points (D = 3), 2 = three points (D = 6), 3 = four points (D = 9),
// 4 = every mollified edge-edge contact (D = 9).  Inactive contacts (d >= d_hat)
// get an empty record here.
__device__ __forceinline__ int classify_one(const WorldArgs& a, int cid) {
    int id0, id1, id2, id3;
    const bool is_ee = contact_ids(a, cid, id0, id1, id2, id3);
    const d3 p0 = ld3(a.X + 3 * (size_t)id0), p1 = ld3(a.X + 3 * (size_t)id1);
    const d3 p2 = ld3(a.X + 3 * (size_t)id2), p3 = ld3(a.X + 3 * (size_t)id3);
    int type; double d;
    if (!is_ee) { type = pt_type(p0, p1, p2, p3); d = pt_dist(p0, p1, p2, p3, type); }
    else { type = ee_type(p0, p1, p2, p3); d = ee_dist(p0, p1, p2, p3, type); }
    a.ctype[cid] = type; a.cdist[cid] = d;
    int cls = 0;
    if (d < a.kp.d_hat) {
        const int kind = is_ee ? ee_map(type).kind : pt_map(type).kind;
        cls = kind == K_PP ? 1 : (kind == K_PL ? 2 : 3);
        if (is_ee) {
            // mollifier active: x = |(p1 - p0) x (p3 - p2)|^2 < eps_x |p0 - p1|^2 |p2 - p3|^2
            const double eps = a.kp.eps_x * sqn(p0 - p1) * sqn(p2 - p3);
            const d3 c = cross(p1 - p0, p3 - p2);
            if (dot(c, c) < eps) cls = 4;
        }
    } else {
        a.rec[REC * (size_t)cid + R_D] = 0.0;
        double* tk = a.tk + TKN * (size_t)cid;
        for (int i = 0; i < TKN; i++) tk[i] = 0.0;
        a.lam[cid] = 0.0;
    }
    a.ccls[cid] = min(cls, 3);      // Helmert rows of the record
    return cls;
}

// Classification and the per-class lists (class 1 from the front of `list`,
// class 2 from its back, class 3 from the front of `list3`, class 4 from its
// back).  Device-scope atomics on one
// address serialize (~11 ns each on gfx950), so the slots are claimed per
// workgroup: each workgroup classifies a tile of rpt x CL_THREADS contacts,
// counts its classes with LDS atomics (one per wavefront and class), takes
// one global range per class, and then writes the list entries.
constexpr int CL_THREADS = 1024;
constexpr int CL_RPT_MAX = 8;
__global__ __launch_bounds__(CL_THREADS) void k_contact_classify(WorldArgs a, int rpt) {
    __shared__ int lcnt[4], lbase[4];
    const int total = a.n_pt + a.n_ee;
    const int lane = __lane_id();
    if (threadIdx.x < 4) lcnt[threadIdx.x] = 0;
    __syncthreads();
    int cls_r[CL_RPT_MAX], pos_r[CL_RPT_MAX];
    const int base = blockIdx.x * CL_THREADS * rpt;
#pragma unroll
    for (int r = 0; r < CL_RPT_MAX; r++) {
        cls_r[r] = 0; pos_r[r] = 0;
        if (r < rpt) {
            const int cid = base + r * CL_THREADS + threadIdx.x;
            const int cls = cid < total ? classify_one(a, cid) : 0;
            cls_r[r] = cls;
#pragma unroll
            for (int k = 1; k <= 4; k++) {
                const unsigned long long m = __ballot(cls == k);
                if (m == 0ull) continue;
                const int leader = __ffsll((long long)m) - 1;
                int b = 0;
                if (lane == leader) b = atomicAdd(&lcnt[k - 1], __popcll(m));
                b = __shfl(b, leader);
                if (cls == k) pos_r[r] = b + __popcll(m & ((1ull << lane) - 1ull));
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < 4) lbase[threadIdx.x] = lcnt[threadIdx.x] ? atomicAdd(&a.counts[threadIdx.x], lcnt[threadIdx.x]) : 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < CL_RPT_MAX; r++) {
        if (r >= rpt) break;
        const int cid = base + r * CL_THREADS + threadIdx.x;
        const int cls = cls_r[r];
        if (cls == 1) a.list[lbase[0] + pos_r[r]] = cid;
        else if (cls == 2) a.list[total - 1 - (lbase[1] + pos_r[r])] = cid;
        else if (cls == 3) a.list3[lbase[2] + pos_r[r]] = cid;
        else if (cls == 4) a.list3[total - 1 - (lbase[3] + pos_r[r])] = cid;
    }
}

// Friction of one contact (model/friction.cpp:15-47) with the tangential
// displacement measured from the step start.
struct Fric {
    double gm0, gm1, gm2, gm3;
    d3 c0, c1;
    double u0, u1, lam, fs, M[3];
    bool on;
};
__device__ __forceinline__ void friction_eval(const WorldArgs& a, int is_ee, int type, double d, double B1,
                                              d3 P0, d3 P1, d3 P2, d3 P3, int id0, int id1, int id2, int id3, Fric& f) {
    friction_frame(is_ee, type, P0, P1, P2, P3, f.gm0, f.gm1, f.gm2, f.gm3, f.c0, f.c1);
    const d3 d0 = P0 - ld3(a.Xs + 3 * (size_t)id0), d1 = P1 - ld3(a.Xs + 3 * (size_t)id1);
    const d3 d2 = P2 - ld3(a.Xs + 3 * (size_t)id2), d3v = P3 - ld3(a.Xs + 3 * (size_t)id3);
    f.u0 = f.gm0 * dot(f.c0, d0) + f.gm1 * dot(f.c0, d1) + f.gm2 * dot(f.c0, d2) + f.gm3 * dot(f.c0, d3v);
    f.u1 = f.gm0 * dot(f.c1, d0) + f.gm1 * dot(f.c1, d1) + f.gm2 * dot(f.c1, d2) + f.gm3 * dot(f.c1, d3v);
    f.lam = -B1 * 2 * sqrt(d);
    f.on = is_ee ? a.kp.ee_fric : a.kp.pt_fric;
    f.fs = 0.0; f.M[0] = 0.0; f.M[1] = 0.0; f.M[2] = 0.0;
    if (f.on) friction_M(f.u0, f.u1, f.lam, a.kp, f.fs, f.M);
}
// F[i][j] = sum_{r, q} M_rq c_r[i] c_q[j]
__device__ __forceinline__ double fric_F(const Fric& f, int i, int j) {
    const double c0i = cmp(f.c0, i), c1i = cmp(f.c1, i), c0j = cmp(f.c0, j), c1j = cmp(f.c1, j);
    return f.M[0] * c0i * c0j + f.M[1] * (c0i * c1j + c1i * c0j) + f.M[2] * c1i * c1j;
}

// Record fields shared by the per-thread and per-group paths, emitted as
// put(field, value).  Friction part: F and G of the record; the lagged basis
// (gm_k, c0, c1: TKN doubles); lambda is stored by the caller.
template <class Put>
__device__ __forceinline__ void fric_fields(const Fric& f, int nside0, const double w[4][4], Put put) {
    const double gmv[4] = {f.gm0, f.gm1, f.gm2, f.gm3};
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) put(R_F + 3 * i + j, fric_F(f, i, j));
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int al = 0; al < 4; al++) {
            double g = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if ((k < nside0) == (s == 0)) g += gmv[k] * w[k][al];
            put(R_G + 4 * s + al, g);
        }
}
template <class Put>
__device__ __forceinline__ void tk_fields(const Fric& f, Put put) {
    const double gmv[4] = {f.gm0, f.gm1, f.gm2, f.gm3};
#pragma unroll
    for (int k = 0; k < 4; k++) put(k, gmv[k]);
#pragma unroll
    for (int r = 0; r < 3; r++) { put(4 + r, cmp(f.c0, r)); put(7 + r, cmp(f.c1, r)); }
}
// Body-space gradient from per-point vertex gradients gv_k (friction included).
template <class Put>
__device__ __forceinline__ void grad_fields(int nside0, const double w[4][4], const d3 gv[4], Put put) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int al = 0; al < 4; al++)
#pragma unroll
            for (int r = 0; r < 3; r++) {
                double g = 0.0;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if ((k < nside0) == (s == 0)) g += w[k][al] * cmp(gv[k], r);
                put(R_GRAD + 12 * s + 3 * al + r, g);
            }
}
__device__ __forceinline__ void write_fric(const WorldArgs& a, int cid, int nside0, const Fric& f, const double w[4][4]) {
    double* R = a.rec + REC * (size_t)cid;
    fric_fields(f, nside0, w, [&](int k, double v) { R[k] = v; });
    double* tk = a.tk + TKN * (size_t)cid;
    tk_fields(f, [&](int k, double v) { tk[k] = v; });
    a.lam[cid] = f.lam;
}
__device__ __forceinline__ void write_grad(const WorldArgs& a, int cid, int nside0, const double w[4][4], const d3 gv[4]) {
    double* R = a.rec + REC * (size_t)cid;
    grad_fields(nside0, w, gv, [&](int k, double v) { R[k] = v; });
}

// Record sections staged per wavefront.  A contact kernel with one thread per
// record would store each field with 64 lanes on 64 different cache lines;
// instead lane l puts field k of a section into S[k][l] (element-major, row
// padded to 65 doubles), and stage_flush stores the section's NF consecutive
// doubles of each of the wavefront's records with consecutive lanes on
// consecutive (record, field) pairs: a store instruction then covers a few
// lines.  Lanes past the end of the contact list compute a duplicate of the
// last contact (nothing of theirs is stored), so every flush runs with the
// whole wavefront active.
constexpr int SNF = 24, SLD = 65;
struct Stage {
    double (*S)[SLD];
    int lane, cid, nvalid;
};
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// base[stride * cid_r + off + k] = S[k][r] for records r < nvalid, fields k < NF,
// as 16-byte stores of field pairs (the texture address unit's work grows with
// the number of store instructions, not with the cache lines they cover; off,
// stride and record bases are even in doubles, so every pair is aligned)
template <int NF>
__device__ __forceinline__ void stage_flush(const Stage& st, double* base, int stride, int off) {
    static_assert(NF <= SNF && NF % 2 == 0, "sections of an even number of fields within the staging rows");
    constexpr int NP = NF / 2;
    wave_lds_sync();
#pragma unroll 1
    for (int it = 0; it < NP; it++) {
        const int t = it * 64 + st.lane;      // < 64 NP, so r < 64
        const int r = t / NP, jp = t - r * NP;
        const int c = __shfl(st.cid, r);
        if (r < st.nvalid) {
            double2 v;
            v.x = st.S[2 * jp][r];
            v.y = st.S[2 * jp + 1][r];
            *reinterpret_cast<double2*>(base + (size_t)stride * c + off + 2 * jp) = v;
        }
    }
    wave_lds_sync();
}
__device__ __forceinline__ void load_w(const double* xbar, int id0, int id1, int id2, int id3, double w[4][4]) {
    const d3 x0 = ld3(xbar + 3 * (size_t)id0), x1 = ld3(xbar + 3 * (size_t)id1);
    const d3 x2 = ld3(xbar + 3 * (size_t)id2), x3 = ld3(xbar + 3 * (size_t)id3);
    const d3 xs[4] = {x0, x1, x2, x3};
#pragma unroll
    for (int k = 0; k < 4; k++) { w[k][0] = 1.0; w[k][1] = xs[k].x; w[k][2] = xs[k].y; w[k][3] = xs[k].z; }
}

// Class 1 contacts, one thread each: d = |r|^2, r = x_a - x_b.  In the
// Helmert coordinate y = (x_a - x_b) / sqrt(2) the Hessian is
// K = 4 B1 I + 8 B2 r r^T with eigenvalues 4 B1 (twice, normal to r) and
// 4 B1 + 8 B2 d (along r).
__device__ __forceinline__ void contact_small(const WorldArgs& a, const Stage& st, bool valid) {
    const int cid = st.cid, l = st.lane;
    double (*S)[SLD] = st.S;
    int id0, id1, id2, id3;
    const int is_ee = contact_ids(a, cid, id0, id1, id2, id3);
    const d3 P0 = ld3(a.X + 3 * (size_t)id0), P1 = ld3(a.X + 3 * (size_t)id1);
    const d3 P2 = ld3(a.X + 3 * (size_t)id2), P3 = ld3(a.X + 3 * (size_t)id3);
    const int type = a.ctype[cid];
    const double d = a.cdist[cid];
    const RedMap mp = is_ee ? ee_map(type) : pt_map(type);
    const int nside0 = is_ee ? 2 : 1;
    const double B1 = barrier_d1(d, a.kp.d_hat, a.kp.kappa);
    const double B2 = barrier_d2(d, a.kp.d_hat, a.kp.kappa);
    const d3 z = mk(0, 0, 0);
    double w[4][4];
    load_w(a.xbar, id0, id1, id2, id3, w);
    // friction first: D, F, G (fields 0..17), the lagged basis and lambda
    // stored now; kept: gm_k and ft = fs (u0 c0 + u1 c1), the friction
    // gradient of point k being gm_k ft
    double gmv[4];
    d3 ft = z;
    {
        Fric f;
        friction_eval(a, is_ee, type, d, B1, P0, P1, P2, P3, id0, id1, id2, id3, f);
        S[R_D][l] = rec_code(a, cid, 3);
        fric_fields(f, nside0, w, [&](int k, double v) { S[k][l] = v; });
        stage_flush<R_Z>(st, a.rec, REC, 0);
        tk_fields(f, [&](int k, double v) { S[k][l] = v; });
        stage_flush<TKN>(st, a.tk, TKN, 0);
        if (valid) a.lam[cid] = f.lam;
        gmv[0] = f.gm0; gmv[1] = f.gm1; gmv[2] = f.gm2; gmv[3] = f.gm3;
        if (f.on) {
            const double t0 = f.fs * f.u0, t1 = f.fs * f.u1;
            ft = mk(t0 * f.c0.x + t1 * f.c1.x, t0 * f.c0.y + t1 * f.c1.y, t0 * f.c0.z + t1 * f.c1.z);
        }
    }
    d3 gv[4];
    double hz[4];         // Helmert weight of point slot k (zero off the contact's slots)
    {
        const int ka = mp.plus[0], kb = mp.minus[0];
        const d3 r = pick(P0, P1, P2, P3, ka) - pick(P0, P1, P2, P3, kb);
        const double lp = 4.0 * B1, ll = 4.0 * B1 + 8.0 * B2 * d;
        if (a.kp.psd) {
            const double cp = fmax(lp, 0.0), cl = fmax(ll, 0.0);
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    const double rr = cmp(r, i) * cmp(r, j) / d;
                    S[3 * i + j][l] = cl * rr + cp * ((i == j ? 1.0 : 0.0) - rr);
                }
        } else {
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int j = 0; j < 3; j++) S[3 * i + j][l] = (i == j ? lp : 0.0) + 8.0 * B2 * cmp(r, i) * cmp(r, j);
        }
        S[9][l] = 0.0;      // pad to a field pair: R_PK + 9 is past a 2-point record
        stage_flush<10>(st, a.rec, REC, R_PK);
#pragma unroll
        for (int k = 0; k < 4; k++) hz[k] = k == ka ? HS2 : (k == kb ? -HS2 : 0.0);
        const d3 g = mk(2 * r.x * B1, 2 * r.y * B1, 2 * r.z * B1);
#pragma unroll
        for (int k = 0; k < 4; k++) gv[k] = k == ka ? g : (k == kb ? mk(-g.x, -g.y, -g.z) : z);
    }
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int al = 0; al < 4; al++) {
            double zz = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if ((k < nside0) == (s == 0)) zz += hz[k] * w[k][al];
            S[4 * s + al][l] = zz;
        }
    stage_flush<8>(st, a.rec, REC, R_Z);
#pragma unroll
    for (int k = 0; k < 4; k++)
        gv[k] = mk(gv[k].x + gmv[k] * ft.x, gv[k].y + gmv[k] * ft.y, gv[k].z + gmv[k] * ft.z);
    grad_fields(nside0, w, gv, [&](int k, double v) { S[k - R_GRAD][l] = v; });
    stage_flush<24>(st, a.rec, REC, R_GRAD);
}
// Class 4 contacts (mollified edge pairs) in two launches.
// k_contact_c3r: ten threads per contact.  Thread role r < 9 builds the entries
// of the 9x9 Helmert-coordinate matrix K = (C (x) I3) Mred (C^T (x) I3) +
// mollifier terms (C = h4 S^T, Cm the same for y = p1 - p0, z = p3 - p2) of
// one component pair (i, j) = (r / 3, r % 3) and stores them with their
// mirror images (K exactly symmetric) in the record's PK field; role 9
// writes the record's other fields (Z, friction, gradient, class code).
// k_contact_psd9: one thread per contact projects K in place, cyclic Jacobi
// on the packed upper triangle in registers with the eigenvectors beside it
// (a scheduling barrier after each rotation keeps the live ranges to one
// rotation).  Split this way the geometry's registers stay out of the Jacobi
// kernel, and the matrix of a contact is built by nine threads at once.
constexpr int C3_ROLES = 10;
struct C3Ctx {
    Geo G;
    int id0, id1, id2, id3;
    double* R;
};
__device__ __forceinline__ void c3_setup(const WorldArgs& a, int cid, C3Ctx& x) {
    x.R = a.rec + REC * (size_t)cid;
    Geo& G = x.G;
    contact_ids(a, cid, x.id0, x.id1, x.id2, x.id3);
    G.p0 = ld3(a.X + 3 * (size_t)x.id0); G.p1 = ld3(a.X + 3 * (size_t)x.id1);
    G.p2 = ld3(a.X + 3 * (size_t)x.id2); G.p3 = ld3(a.X + 3 * (size_t)x.id3);
    G.type = a.ctype[cid]; G.d = a.cdist[cid];
    geo_init(G, a.kp);
}
// the entries of K for component pair role = (i, j), into the PK field
__device__ __forceinline__ void c3_kbuild(const C3Ctx& x, int role) {
    const Geo& G = x.G;
    double* R = x.R;
    double C[3][3], Cm[3][2];
#pragma unroll
    for (int q = 0; q < 3; q++) {
#pragma unroll
        for (int m = 0; m < 3; m++) {
            double c = 0.0;
#pragma unroll
            for (int k = 0; k < 4; k++) c += kHel[q][k] * red_sign(G.map, m, k);
            C[q][m] = m < G.map.nr ? c : 0.0;
        }
        Cm[q][0] = kHel[q][1] - kHel[q][0];
        Cm[q][1] = kHel[q][3] - kHel[q][2];
    }
    {
        const int i = role / 3, j = role % 3;
        double K[3][3];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int b = 0; b < 3; b++) K[q][b] = 0.0;
#pragma unroll
        for (int m = 0; m < 3; m++)
#pragma unroll
            for (int n = 0; n < 3; n++) {
                if (m < G.map.nr && n < G.map.nr) {
                    const double Mv = G.B1 * G.rd.hess(m, i, n, j) + G.B2 * cmp(G.rd.g[m], i) * cmp(G.rd.g[n], j);
#pragma unroll
                    for (int q = 0; q < 3; q++)
#pragma unroll
                        for (int b = 0; b < 3; b++) K[q][b] += C[q][m] * C[b][n] * Mv;
                }
            }
        {
            double gdi[3], gdj[3], gxi[3], gxj[3];
#pragma unroll
            for (int q = 0; q < 3; q++) {
                double si = 0.0, sj = 0.0;
#pragma unroll
                for (int m = 0; m < 3; m++)
                    if (m < G.map.nr) { si += C[q][m] * cmp(G.rd.g[m], i); sj += C[q][m] * cmp(G.rd.g[m], j); }
                gdi[q] = si; gdj[q] = sj;
                gxi[q] = G.m2 != 0.0 ? Cm[q][0] * G.mc.grad(0, i) + Cm[q][1] * G.mc.grad(1, i) : 0.0;
                gxj[q] = G.m2 != 0.0 ? Cm[q][0] * G.mc.grad(0, j) + Cm[q][1] * G.mc.grad(1, j) : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 3; q++)
#pragma unroll
                for (int b = 0; b < 3; b++) {
                    double hxk = 0.0;
                    if (G.m2 != 0.0) {
#pragma unroll
                        for (int u = 0; u < 2; u++)
#pragma unroll
                            for (int v = 0; v < 2; v++) hxk += Cm[q][u] * Cm[b][v] * G.mc.hess(u, i, v, j);
                    }
                    const double gmi = G.m1 * gxi[q], gmj = G.m1 * gxj[b];
                    K[q][b] = G.m * K[q][b] + G.B1 * (gmi * gdj[b] + gdi[q] * gmj) + G.B0 * (G.m2 * gxi[q] * gxj[b] + G.m1 * hxk);
                }
        }
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int b = 0; b < 3; b++)
                if (3 * q + i <= 3 * b + j) {
                    // entry (3q + i, 3b + j) of the upper triangle and its mirror; the
                    // lower-triangle entries of this pair are upper ones of pair (j, i)
                    R[R_PK + 9 * (3 * q + i) + 3 * b + j] = K[q][b];
                    R[R_PK + 9 * (3 * b + j) + 3 * q + i] = K[q][b];
                }
    }
}
// everything but PK: Z, friction (F, G, Tk, lambda), the gradient, the class code
__device__ __forceinline__ void c3_fields(const WorldArgs& a, int cid, const C3Ctx& x) {
    const Geo& G = x.G;
    double* R = x.R;
    const int id0 = x.id0, id1 = x.id1, id2 = x.id2, id3 = x.id3;
    const int nside0 = 2;
    double w[4][4];
    load_w(a.xbar, id0, id1, id2, id3, w);
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int al = 0; al < 4; al++) {
                double zz = 0.0;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if ((k < nside0) == (s == 0)) zz += kHel[q][k] * w[k][al];
                R[R_Z + 8 * q + 4 * s + al] = zz;
            }
    Fric f;
    friction_eval(a, 1, G.type, G.d, G.B1, G.p0, G.p1, G.p2, G.p3, id0, id1, id2, id3, f);
    write_fric(a, cid, nside0, f, w);
    const double gmv[4] = {f.gm0, f.gm1, f.gm2, f.gm3};
    d3 gv[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        double g3[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double g = barrier_grad(G, 3 * k + c);
            if (f.on) g += f.fs * (gmv[k] * cmp(f.c0, c) * f.u0 + gmv[k] * cmp(f.c1, c) * f.u1);
            g3[c] = g;
        }
        gv[k] = mk(g3[0], g3[1], g3[2]);
    }
    write_grad(a, cid, nside0, w, gv);
    R[R_D] = rec_code(a, cid, 9);
}
__device__ __forceinline__ void psd9(const WorldArgs& a, int cid) {
    double* R = a.rec + REC * (size_t)cid;
    double A[45], V[81];
#pragma unroll
    for (int p = 0; p < 9; p++)
#pragma unroll
        for (int q = p; q < 9; q++) A[PK_<9>(p, q)] = R[R_PK + 9 * p + q];
    jacobi_packed<9>(A, V);
    project_packed<9>(A, V);
#pragma unroll
    for (int p = 0; p < 9; p++)
#pragma unroll
        for (int q = p; q < 9; q++) {
            R[R_PK + 9 * p + q] = A[PK_<9>(p, q)];
            R[R_PK + 9 * q + p] = A[PK_<9>(p, q)];
        }
}
// The roles and the Jacobi are separate kernels, so the role threads get the
// registers of their own code (two wavefronts per SIMD) while the Jacobi
// holds ~280 (one).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_contact_c3r(WorldArgs a) {
    const int n4 = a.counts[3], last = a.n_pt + a.n_ee - 1;
    const long long n = (long long)C3_ROLES * n4;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x) {
        const int cid = a.list3[last - (int)(t / C3_ROLES)], role = (int)(t % C3_ROLES);
        C3Ctx x;
        c3_setup(a, cid, x);
        if (role < 9) c3_kbuild(x, role);
        else c3_fields(a, cid, x);
    }
}
__global__ __launch_bounds__(64) void k_contact_psd9(WorldArgs a) {
    const int n4 = a.counts[3], last = a.n_pt + a.n_ee - 1;
    for (int p = blockIdx.x * 64 + threadIdx.x; p < n4; p += gridDim.x * 64) psd9(a, a.list3[last - p]);
}

// record fields other than PK of a 3-point contact: D, friction, gradient, Z
__device__ __forceinline__ void scalars_c2(const WorldArgs& a, const Stage& st, bool valid) {
    const int cid = st.cid, l = st.lane;
    double (*S)[SLD] = st.S;
    int id0, id1, id2, id3;
    const int is_ee = contact_ids(a, cid, id0, id1, id2, id3);
    const d3 P0 = ld3(a.X + 3 * (size_t)id0), P1 = ld3(a.X + 3 * (size_t)id1);
    const d3 P2 = ld3(a.X + 3 * (size_t)id2), P3 = ld3(a.X + 3 * (size_t)id3);
    const int type = a.ctype[cid];
    const double d = a.cdist[cid];
    const RedMap mp = is_ee ? ee_map(type) : pt_map(type);
    const int nside0 = is_ee ? 2 : 1;
    const double B1 = barrier_d1(d, a.kp.d_hat, a.kp.kappa);
    const d3 z = mk(0, 0, 0);
    Fric f;
    friction_eval(a, is_ee, type, d, B1, P0, P1, P2, P3, id0, id1, id2, id3, f);
    double w[4][4];
    load_w(a.xbar, id0, id1, id2, id3, w);
    S[R_D][l] = rec_code(a, cid, 6);
    fric_fields(f, nside0, w, [&](int k, double v) { S[k][l] = v; });
    stage_flush<R_Z>(st, a.rec, REC, 0);
    tk_fields(f, [&](int k, double v) { S[k][l] = v; });
    stage_flush<TKN>(st, a.tk, TKN, 0);
    if (valid) a.lam[cid] = f.lam;
    const int ka = mp.plus[0], kb = mp.plus[1], km = mp.minus[0];
    const d3 pm = pick(P0, P1, P2, P3, km);
    RedDist rd;
    rd.init(K_PL, pick(P0, P1, P2, P3, ka) - pm, pick(P0, P1, P2, P3, kb) - pm, z);
    const d3 g0 = mk(B1 * rd.g[0].x, B1 * rd.g[0].y, B1 * rd.g[0].z);
    const d3 g1 = mk(B1 * rd.g[1].x, B1 * rd.g[1].y, B1 * rd.g[1].z);
    const d3 gm = mk(-(g0.x + g1.x), -(g0.y + g1.y), -(g0.z + g1.z));
    const double gmv[4] = {f.gm0, f.gm1, f.gm2, f.gm3};
    d3 ft = z;
    if (f.on) {
        const double t0 = f.fs * f.u0, t1 = f.fs * f.u1;
        ft = mk(t0 * f.c0.x + t1 * f.c1.x, t0 * f.c0.y + t1 * f.c1.y, t0 * f.c0.z + t1 * f.c1.z);
    }
    d3 gv[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const d3 gb = k == ka ? g0 : (k == kb ? g1 : (k == km ? gm : z));
        gv[k] = mk(gb.x + gmv[k] * ft.x, gb.y + gmv[k] * ft.y, gb.z + gmv[k] * ft.z);
    }
    grad_fields(nside0, w, gv, [&](int k, double v) { S[k - R_GRAD][l] = v; });
    stage_flush<24>(st, a.rec, REC, R_GRAD);
    // Helmert rows over the slots (m, a, b): (1, -1, 0) / sqrt 2, (1, 1, -2) / sqrt 6
#pragma unroll
    for (int aa = 0; aa < 2; aa++)
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int al = 0; al < 4; al++) {
                double zz = 0.0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const double h = aa == 0 ? (k == km ? HS2 : (k == ka ? -HS2 : 0.0))
                                             : (k == km ? HS6 : (k == ka ? HS6 : (k == kb ? -2.0 * HS6 : 0.0)));
                    if ((k < nside0) == (s == 0)) zz += h * w[k][al];
                }
                S[8 * aa + 4 * s + al][l] = zz;
            }
    stage_flush<16>(st, a.rec, REC, R_Z);
}

// PK of a 3-point contact (point-line distance) in the frame of terms.h: f2
// decouples (eigenvalue 2 B1 |gamma|^2), so what is left is 3 x 3, in f1 and
// the two Helmert components of the normal displacement over the slots
// (m, a, b).  Against the 6 x 6 Jacobi on the matrix of the point differences
// 276 -> 138 us (2000 crowded bodies, 1.05e6 contacts), 99 -> 40 us (2000 spheres,
// 3.9e5).
__device__ __forceinline__ void pk_c2(const WorldArgs& a, int cid) {
    int id0, id1, id2, id3;
    const int is_ee = contact_ids(a, cid, id0, id1, id2, id3);
    const d3 P0 = ld3(a.X + 3 * (size_t)id0), P1 = ld3(a.X + 3 * (size_t)id1);
    const d3 P2 = ld3(a.X + 3 * (size_t)id2), P3 = ld3(a.X + 3 * (size_t)id3);
    const int type = a.ctype[cid];
    const double d = a.cdist[cid];
    const RedMap mp = is_ee ? ee_map(type) : pt_map(type);
    const double B1 = barrier_d1(d, a.kp.d_hat, a.kp.kappa);
    const double B2 = barrier_d2(d, a.kp.d_hat, a.kp.kappa);
    Frame F;
    contact_frame(is_ee, type, P0, P1, P2, P3, F);
    double gh[2], mh[2];
    {
        auto at = [](const double v[4], int k) { return k == 0 ? v[0] : (k == 1 ? v[1] : (k == 2 ? v[2] : v[3])); };
        const int km = mp.minus[0], ka = mp.plus[0], kb = mp.plus[1];
        const double g0 = at(F.gam, km), g1 = at(F.gam, ka), g2 = at(F.gam, kb);
        const double m0 = at(F.m1, km), m1 = at(F.m1, ka), m2 = at(F.m1, kb);
        gh[0] = HS2 * (g0 - g1); gh[1] = HS6 * ((g0 + g1) - 2.0 * g2);
        mh[0] = HS2 * (m0 - m1); mh[1] = HS6 * ((m0 + m1) - 2.0 * m2);
    }
    double A[6], kt = 2.0 * B1 * F.gn * F.gn;
    {
        const double dd = F.delta * F.delta, As = 2.0 * B1 + 4.0 * B2 * dd, kc = -2.0 * B1 * F.delta * F.gn, kn = -2.0 * B1 * dd;
        A[PK_<3>(0, 0)] = 0.0;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            A[PK_<3>(0, 1 + i)] = kc * mh[i];
#pragma unroll
            for (int j = i; j < 2; j++) A[PK_<3>(1 + i, 1 + j)] = As * gh[i] * gh[j] + kn * mh[i] * mh[j];
        }
    }
    if (a.kp.psd) {
        double V[9];
        jacobi_packed<3>(A, V);
        project_packed<3>(A, V);
        kt = fmax(kt, 0.0);
    }
    double* R = a.rec + REC * (size_t)cid + R_PK;
    const double ign = 1.0 / F.gn;
    const double e[2] = {gh[0] * ign, gh[1] * ign};
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    const double ni = cmp(F.n, i), nj = cmp(F.n, j), fi = cmp(F.f1, i), fj = cmp(F.f1, j);
                    const double tt = A[PK_<3>(0, 0)] * (fi * fj) + kt * (cmp(F.f2, i) * cmp(F.f2, j));
                    R[6 * (3 * q + i) + 3 * b + j] = e[q] * e[b] * tt + (e[q] * A[PK_<3>(0, 1 + b)] * (fi * nj) + e[b] * A[PK_<3>(0, 1 + q)] * (ni * fj)) +
                                                     A[PK_<3>(1 + q, 1 + b)] * (ni * nj);
                }
}

// Class 3 contacts (point-plane, edge-edge interior), one thread each: the
// whole record from the frame of terms.h, the projection a 5 x 5 Jacobi in
// registers.  Bound by the scattered points and the 1.2 KB record.  Ten
// threads per contact building the 9 x 9 matrix in memory and a second kernel
// projecting it there took 751 + 147 us for all class 3 and 4 contacts of 2000
// crowded bodies; this takes 342 us, and 149 + 130 us are left for the
// mollified ones.
__device__ __forceinline__ void contact_plane(const WorldArgs& a, const Stage& st, bool valid) {
    const int cid = st.cid, l = st.lane;
    double (*S)[SLD] = st.S;
    int id0, id1, id2, id3;
    const int is_ee = contact_ids(a, cid, id0, id1, id2, id3);
    const d3 P0 = ld3(a.X + 3 * (size_t)id0), P1 = ld3(a.X + 3 * (size_t)id1);
    const d3 P2 = ld3(a.X + 3 * (size_t)id2), P3 = ld3(a.X + 3 * (size_t)id3);
    const int type = a.ctype[cid];
    const double d = a.cdist[cid];
    const int nside0 = is_ee ? 2 : 1;
    const double B1 = barrier_d1(d, a.kp.d_hat, a.kp.kappa);
    const double B2 = barrier_d2(d, a.kp.d_hat, a.kp.kappa);
    Frame F;
    contact_frame(is_ee, type, P0, P1, P2, P3, F);
    double M[15];
    frame_matrix(F, B1, B2, M);
    if (a.kp.psd) {
        double V[25];
        jacobi_packed<5>(M, V);
        project_packed<5>(M, V);
    }
    {
        double g[3];
        helmert(F.gam, g);
        const double ign = 1.0 / F.gn;
#pragma unroll
        for (int q = 0; q < 3; q++) g[q] *= ign;
        // rows (q, i) of the 9 x 9 matrix, two rows a section
#pragma unroll
        for (int r0 = 0; r0 < 10; r0 += 2) {
#pragma unroll
            for (int r = r0; r < r0 + 2 && r < 9; r++) {
                const int q = r / 3, i = r % 3;
                const double ni = cmp(F.n, i), f1 = cmp(F.f1, i), f2 = cmp(F.f2, i);
                // the row's weights of f1, f2 and n at column component j, Helmert row b
                const double u1 = M[PK_<5>(0, 0)] * f1 + M[PK_<5>(0, 1)] * f2, u2 = M[PK_<5>(0, 1)] * f1 + M[PK_<5>(1, 1)] * f2;
                const double c1 = g[q] * u1 + M[PK_<5>(0, 2 + q)] * ni, c2 = g[q] * u2 + M[PK_<5>(1, 2 + q)] * ni;
#pragma unroll
                for (int b = 0; b < 3; b++) {
                    const double cn = g[q] * (M[PK_<5>(0, 2 + b)] * f1 + M[PK_<5>(1, 2 + b)] * f2) + M[PK_<5>(2 + q, 2 + b)] * ni;
#pragma unroll
                    for (int j = 0; j < 3; j++)
                        S[9 * (r - r0) + 3 * b + j][l] = g[b] * (c1 * cmp(F.f1, j) + c2 * cmp(F.f2, j)) + cn * cmp(F.n, j);
                }
            }
            if (r0 < 8) stage_flush<18>(st, a.rec, REC, R_PK + 9 * r0);
            else { S[9][l] = 0.0; stage_flush<10>(st, a.rec, REC, R_PK + 72); }      // 9 entries and a pad
        }
    }
    double w[4][4];
    load_w(a.xbar, id0, id1, id2, id3, w);
    double gmv[4];
    d3 ft = mk(0, 0, 0);
    {
        Fric f;
        friction_eval(a, is_ee, type, d, B1, P0, P1, P2, P3, id0, id1, id2, id3, f);
        S[R_D][l] = rec_code(a, cid, 9);
        fric_fields(f, nside0, w, [&](int k, double v) { S[k][l] = v; });
        stage_flush<R_Z>(st, a.rec, REC, 0);
        tk_fields(f, [&](int k, double v) { S[k][l] = v; });
        stage_flush<TKN>(st, a.tk, TKN, 0);
        if (valid) a.lam[cid] = f.lam;
        gmv[0] = f.gm0; gmv[1] = f.gm1; gmv[2] = f.gm2; gmv[3] = f.gm3;
        if (f.on) {
            const double t0 = f.fs * f.u0, t1 = f.fs * f.u1;
            ft = mk(t0 * f.c0.x + t1 * f.c1.x, t0 * f.c0.y + t1 * f.c1.y, t0 * f.c0.z + t1 * f.c1.z);
        }
    }
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int al = 0; al < 4; al++) {
                double zz = 0.0;
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if ((k < nside0) == (s == 0)) zz += kHel[q][k] * w[k][al];
                S[8 * q + 4 * s + al][l] = zz;
            }
    stage_flush<24>(st, a.rec, REC, R_Z);
    const double gs = 2.0 * B1 * F.delta;
    d3 gv[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const double g = gs * F.gam[k];
        gv[k] = mk(g * F.n.x + gmv[k] * ft.x, g * F.n.y + gmv[k] * ft.y, g * F.n.z + gmv[k] * ft.z);
    }
    grad_fields(nside0, w, gv, [&](int k, double v) { S[k - R_GRAD][l] = v; });
    stage_flush<24>(st, a.rec, REC, R_GRAD);
}

// record fields other than PK of 3-point contacts, one thread each
// one 64-contact slice of the class list per wavefront and pass (block of
// 256 lanes, four staging areas: 49.9 KB, three blocks per CU as the
// registers allow); class 1 at list[0, n1), class 2 at list[total - n2, total)
// (stored from the back)
template <int CLS>
__device__ __forceinline__ void contact_slices(const WorldArgs& a) {
    __shared__ double S[4][SNF][SLD];
    const int total = a.n_pt + a.n_ee;
    const int cnt = a.counts[CLS - 1];
    const int wv = threadIdx.x >> 6;
    Stage st;
    st.S = S[wv];
    st.lane = threadIdx.x & 63;
    for (int p0 = (blockIdx.x * 4 + wv) * 64; p0 < cnt; p0 += gridDim.x * 256) {
        const int p = min(p0 + st.lane, cnt - 1);
        st.nvalid = min(64, cnt - p0);
        st.cid = CLS == 3 ? a.list3[p] : a.list[CLS == 1 ? p : total - 1 - p];
        if (CLS == 1) contact_small(a, st, p0 + st.lane < cnt);
        else if (CLS == 3) contact_plane(a, st, p0 + st.lane < cnt);
        else scalars_c2(a, st, p0 + st.lane < cnt);
    }
}
__global__ __launch_bounds__(256) void k_contact_scalars2(WorldArgs a) { contact_slices<2>(a); }
__global__ __launch_bounds__(256, 2) void k_contact_plane(WorldArgs a) { contact_slices<3>(a); }
__global__ __launch_bounds__(64) void k_contact_pk2(WorldArgs a) {
    const int total = a.n_pt + a.n_ee;
    const int cnt = a.counts[1];
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < cnt; p += gridDim.x * blockDim.x)
        pk_c2(a, a.list[total - 1 - p]);
}

template <int CLS>
__global__ __launch_bounds__(256) void k_contact_small(WorldArgs a) {
    static_assert(CLS == 1, "3-point contacts: k_contact_scalars2 / k_contact_pk2");
    contact_slices<1>(a);
}

// VG contact: compact body-space form.  The VG block of body I is
// (w w^T) (x) K with w = (1, xbar) and K = B''(d^2) (2d)^2 e_y e_y^T + friction,
// gradient w (x) gx (model/vg_ipc.cpp:12-30, model/barrier.cpp:31-69).
struct VgArgs {
    KParams kp; int n; double ground_y; int vg_fric;
    const int2* vg; const int* voff; const double* X; const double* Xs;
    double* K; double* lam;
};
__global__ void k_vg_world(VgArgs a) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.n) return;
    int2 c = a.vg[k];
    int v = a.voff[c.x] + c.y;
    d3 p = ld3(a.X + 3 * (size_t)v), p0 = ld3(a.Xs + 3 * (size_t)v);
    double dd = p.y - a.ground_y, d = dd * dd;
    double* K = a.K + 12 * (size_t)k;
    if (!(d < a.kp.d_hat)) {
        for (int i = 0; i < 12; i++) K[i] = 0.0;
        a.lam[k] = 0.0;
        return;
    }
    double B1 = barrier_d1(d, a.kp.d_hat, a.kp.kappa);
    double lam = -B1 * 2 * dd;
    a.lam[k] = lam;
    double gy = 1.0 * barrier_d1(dd * dd, a.kp.d_hat, a.kp.kappa) * 2 * dd;
    double B2 = barrier_d2(dd * dd, a.kp.d_hat, a.kp.kappa);
    double s = dd * 2;
    double Kyy = B2 * s * s;
    double gx = 0.0, gz = 0.0, Kxx = 0.0, Kxz = 0.0, Kzz = 0.0;
    if (a.vg_fric) {
        double u0 = p.x - p0.x, u1 = p.z - p0.z;
        double fs, M[3];
        friction_M(u0, u1, lam, a.kp, fs, M);
        gx = fs * u0; gz = fs * u1;
        Kxx = M[0]; Kxz = M[1]; Kzz = M[2];
    }
    // K column-major 3x3 (x, y, z), then gx
    K[0] = Kxx; K[1] = 0.0; K[2] = Kxz;
    K[3] = 0.0; K[4] = Kyy; K[5] = 0.0;
    K[6] = Kxz; K[7] = 0.0; K[8] = Kzz;
    K[9] = gx; K[10] = gy; K[11] = gz;
}

static KParams make_kp(const adb_params& P) {
    KParams kp;
    kp.d_hat = P.d_hat; kp.kappa = P.kappa; kp.eps_x = P.eps_x; kp.psd = P.psd;
    kp.mu = P.mu; kp.eps_v = P.dt * P.evh; kp.max_uk = P.max_uk;
    kp.pt_fric = P.pt_fric; kp.ee_fric = P.ee_fric;
    return kp;
}

void contact_terms(World& w) {
    const int n = w.cs.n_pt + w.cs.n_ee;
    const size_t nn = (size_t)std::max(n, 1);
    w.crec.reserve(REC * nn);
    w.ctype.reserve(nn); w.cdist.reserve(nn); w.ccls.reserve(nn); w.clist.reserve(nn); w.clist3.reserve(nn);
    w.ccount.reserve(5);
    w.ctk.reserve(TKN * nn);
    w.clam.reserve(nn);
    // the contact set is final here: the assembly's pair structure, which
    // needs nothing else, forks from this point onto its own stream (queued
    // below, after the contact kernels)
    if (!w.ev_asm_fork) ADB_HIP(hipEventCreateWithFlags(&w.ev_asm_fork, hipEventDisableTiming));
    ADB_HIP(hipEventRecord(w.ev_asm_fork, w.stream));
    // class counts [0, 4) (entry 4, the chunk count, belongs to the assembly)
    ADB_HIP(hipMemsetAsync(w.ccount.p, 0, 4 * sizeof(int), w.stream));
    if (n > 0) {
        WorldArgs a;
        a.kp = make_kp(w.P);
        a.n_pt = w.cs.n_pt; a.n_ee = w.cs.n_ee;
        a.pt = w.cs.pt.p; a.ee = w.cs.ee.p;
        a.voff = w.voff.p; a.foff = w.foff.p; a.eoff = w.eoff.p; a.face = w.face.p; a.edge = w.edge.p;
        a.X = w.X.p; a.Xs = w.Xs.p; a.xbar = w.xbar.p; a.mass = w.mass.p;
        a.ctype = w.ctype.p; a.cdist = w.cdist.p; a.ccls = w.ccls.p; a.list = w.clist.p; a.list3 = w.clist3.p; a.counts = w.ccount.p;
        a.rec = w.crec.p; a.tk = w.ctk.p; a.lam = w.clam.p;
        {
            // ids and 4 points in; type, distance and list slot out
            ProfScope ps(w, PK_CONTACT_CLASSIFY, (double)n * 152.0);
            const int rpt = std::min(CL_RPT_MAX, std::max(1, (n + CL_THREADS * 512 - 1) / (CL_THREADS * 512)));
            hipLaunchKernelGGL(k_contact_classify, dim3((n + CL_THREADS * rpt - 1) / (CL_THREADS * rpt)), dim3(CL_THREADS), 0,
                               w.stream, a, rpt);
            ADB_HIP(hipGetLastError());
        }
        const int* snap = prof_snapshot(w, w.ccount.p);
        {
            // mollified edge pairs on the side stream (four 64-lane workgroups per CU,
            // one wave per SIMD, FP64-VALU-bound): they overlap the 2- and 3-point
            // kernels and the assembly's sort; the assembly waits for them
            // before its reduction
            if (!w.stream2) {
                ADB_HIP(hipStreamCreate(&w.stream2));
                ADB_HIP(hipStreamCreate(&w.stream3));
                for (hipEvent_t& e : w.ev_side) ADB_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
                ADB_HIP(hipEventCreateWithFlags(&w.ev_pk, hipEventDisableTiming));
            }
            ADB_HIP(hipEventRecord(w.ev_side[0], w.stream));
            ADB_HIP(hipStreamWaitEvent(w.stream2, w.ev_side[0], 0));
            {
                ProfScope ps(w, PK_CONTACT_GROUP, 0.0, w.stream2);
                ps.counts(snap, 0.0, 0.0, 0.0, 1608.0);
                // the class count is on the device: grids sized for the worst case, grid-stride loops
                hipLaunchKernelGGL(k_contact_c3r, dim3(std::min((C3_ROLES * n + 255) / 256, 16 * w.num_cu)), dim3(256), 0,
                                   w.stream2, a);
                ADB_HIP(hipGetLastError());
                if (a.kp.psd)
                    hipLaunchKernelGGL(k_contact_psd9, dim3(std::min((n + 63) / 64, 4 * w.num_cu)), dim3(64), 0, w.stream2, a);
                ADB_HIP(hipGetLastError());
            }
            ADB_HIP(hipEventRecord(w.ev_side[1], w.stream2));
            // the 3x3 projections of the 3-point contacts and the 4-point records on
            // a third stream, beside the 2- and 3-point record kernels (bound by
            // their scattered loads and stores); they write disjoint record fields
            ADB_HIP(hipStreamWaitEvent(w.stream3, w.ev_side[0], 0));
            {
                // per 3-point contact: ids, 4 points, type and distance in; PK (36 doubles)
                // out; per 4-point contact the whole record (147 doubles) and its inputs
                ProfScope ps(w, PK_CONTACT_PK, 0.0, w.stream3);
                ps.counts(snap, 0.0, 440.0, 1608.0, 0.0);
                hipLaunchKernelGGL(k_contact_pk2, dim3(std::min((n + 63) / 64, 16 * w.num_cu)), dim3(64), 0, w.stream3, a);
                ADB_HIP(hipGetLastError());
                hipLaunchKernelGGL(k_contact_plane, dim3(std::min((n + 255) / 256, 4 * w.num_cu)), dim3(256), 0, w.stream3, a);
                ADB_HIP(hipGetLastError());
            }
            ADB_HIP(hipEventRecord(w.ev_pk, w.stream3));
            w.side_pending = true;
        }
        {
            // per contact: list, ids, type, distance, X / Xs / xbar of 4 points in;
            // record (D = 3: 59 doubles; D = 6: 58 here, PK on the third stream),
            // lagged basis (10) and lambda out
            ProfScope ps(w, PK_CONTACT, 0.0);
            ps.counts(snap, 904.0, 896.0, 0.0, 0.0);
            const int grid = std::min((n + 255) / 256, 8 * w.num_cu);
            hipLaunchKernelGGL(k_contact_small<1>, dim3(grid), dim3(256), 0, w.stream, a);
            ADB_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_contact_scalars2, dim3(grid), dim3(256), 0, w.stream, a);
            ADB_HIP(hipGetLastError());
        }
    }
    const int nv = w.cs.n_vg;
    // at least V / 8 entries: the count grows step by step while a pile
    // settles, and each regrowth frees a buffer (a device-wide wait)
    const size_t nvc = std::max<size_t>(std::max(nv, 1), (size_t)w.V / 8);
    w.vgK.reserve(12 * nvc);
    w.vglam.reserve(nvc);
    if (nv > 0) {
        VgArgs v;
        v.kp = make_kp(w.P); v.n = nv; v.ground_y = w.P.ground_y; v.vg_fric = w.P.vg_fric;
        v.vg = w.cs.vg.p; v.voff = w.voff.p; v.X = w.X.p; v.Xs = w.Xs.p;
        v.K = w.vgK.p; v.lam = w.vglam.p;
        ProfScope ps(w, PK_VG_CONTACT, (double)nv * (8.0 + 48.0 + 96.0 + 8.0));
        hipLaunchKernelGGL(k_vg_world, dim3((nv + 255) / 256), dim3(256), 0, w.stream, v);
        ADB_HIP(hipGetLastError());
    }
    assemble_structure(w, true);
}

} // namespace adb

// ============================================================================ C ABI
using namespace adb;

extern "C" void adb_kernel_config_default(adb_kernel_config* c) {
    // abdtk build: barrier::d_hat = 1e-4, barrier::kappa = 1e-3 (model/barrier.cpp:7-8),
    // globals.eps_x = 1e-3 and globals.psd = true (model/settings.h:16,39)
    c->d_hat = 1e-4; c->kappa = 1e-3; c->eps_x = 1e-3; c->psd = 1;
}

static KParams api_kp(const adb_kernel_config* c) {
    KParams kp;
    adb_kernel_config d;
    if (!c) { adb_kernel_config_default(&d); c = &d; }
    kp.d_hat = c->d_hat; kp.kappa = c->kappa; kp.eps_x = c->eps_x; kp.psd = c->psd;
    kp.mu = 0; kp.eps_v = 1; kp.max_uk = 0; kp.pt_fric = 0; kp.ee_fric = 0;
    return kp;
}

extern "C" int adb_ipc_hess_pt_12x12_batched(const adb_kernel_config* cfg, int n, const double* pt, const int* type,
                                             const double* dist, double* H, double* g, void* stream) {
    if (n < 0) return ADB_E_ARG;
    if (n == 0) return ADB_OK;
    hipLaunchKernelGGL(k_hess_api<0>, dim3((n + 63) / 64), dim3(64), 0, (hipStream_t)stream,
                       api_kp(cfg), n, pt, type, dist, H, g, (double*)nullptr);
    return hipGetLastError() == hipSuccess ? ADB_OK : ADB_E_HIP;
}
extern "C" int adb_ipc_hess_ee_12x12_batched(const adb_kernel_config* cfg, int n, const double* ee, const int* type,
                                             const double* dist, double* H, double* g, double* moll, void* stream) {
    if (n < 0) return ADB_E_ARG;
    if (n == 0) return ADB_OK;
    const KParams kp = api_kp(cfg);
    hipLaunchKernelGGL(k_hess_api<1>, dim3((n + 63) / 64), dim3(64), 0, (hipStream_t)stream, kp, n, ee, type, dist, H, g, moll);
    // about one workgroup per SIMD, at most HM_PER contacts each
    const int per = std::min(HM_PER, std::max(64, (n / 1024 + 63) / 64 * 64));
    hipLaunchKernelGGL(k_hess_moll, dim3((n + per - 1) / per), dim3(64), 0, (hipStream_t)stream, kp, n, per, ee, type, dist, H, g, moll);
    return hipGetLastError() == hipSuccess ? ADB_OK : ADB_E_HIP;
}

template <int IS_EE>
static int single_hess(const adb_kernel_config* cfg, const double x[12], int type, double dist, double H[144], double g[12], double* moll) {
    double* m = host_staging().get();
    if (!m) return ADB_E_HIP;
    // x (12), dist, type | H (144), g (12), moll
    double *mH = m + 16, *mg = mH + 144, *mm = mg + 12;
    static_assert(16 + 144 + 12 + 1 <= HostStaging::N, "single contact in the staging page");
    std::memcpy(m, x, 12 * sizeof(double));
    m[12] = dist;
    int* mt = reinterpret_cast<int*>(m + 13);
    *mt = type;
    int rc;
    if (IS_EE) rc = adb_ipc_hess_ee_12x12_batched(cfg, 1, m, mt, m + 12, mH, mg, mm, nullptr);
    else rc = adb_ipc_hess_pt_12x12_batched(cfg, 1, m, mt, m + 12, mH, mg, nullptr);
    if (rc == ADB_OK && hipStreamSynchronize(nullptr) != hipSuccess) rc = ADB_E_HIP;
    if (rc != ADB_OK) return rc;
    std::memcpy(H, mH, 144 * sizeof(double));
    std::memcpy(g, mg, 12 * sizeof(double));
    if (IS_EE && moll) *moll = *mm;
    return ADB_OK;
}
extern "C" int adb_ipc_hess_pt_12x12(const adb_kernel_config* cfg, const double pt[12], int type, double dist, double H[144], double g[12]) {
    return single_hess<0>(cfg, pt, type, dist, H, g, nullptr);
}
extern "C" int adb_ipc_hess_ee_12x12(const adb_kernel_config* cfg, const double ee[12], int type, double dist, double H[144], double g[12], double* moll) {
    return single_hess<1>(cfg, ee, type, dist, H, g, moll);
}
