// pcg.hip - block-Jacobi preconditioned conjugate gradients on the BSR
// Hessian, FP64 throughout.  Replaces the direct PardisoLLT / SimplicialLLT
// solve of ABD::solve (model/abd.cpp:263-291): dq = -H^{-1} g.
//
// Two launches per iteration, no atomics and no host round trip:
//   spmv(k)  : every workgroup first sums the update partials of iteration
//              k - 1 (r.z, r.r per update workgroup) in a fixed order; from
//              them the stop test (r.r <= rtol^2 b.b) and beta = rz_k /
//              rz_{k-1}; then p = z + beta p_old (on the fly for every column
//              block, written for the workgroup's own rows into the other p
//              buffer), y = H p, and one p.y partial per workgroup
//   update(k): every workgroup sums the p.y partials in a fixed order, alpha =
//              rz / pAp, x += alpha p, r -= alpha y, z = M^-1 r (explicit
//              inverse of the diagonal block, 12 lanes per body), and one
//              (r.z, r.r) partial per workgroup
// At most SPMV_WGS and UPD_WGS workgroups, which loop over their rows or
// groups: every workgroup reads every partial of the other kernel, so one
// partial per 4 rows or per group, read by each wave, made an iteration
// quadratic in the bodies.  27 000 bodies in 256 scenes: 305 + 97 -> 13 + 24 us
// an iteration; 10 000 cards: 23 + 20 -> 13 + 18 us.  Small worlds are bound by
// the chain of dependent loads, which the kernels issue in three rounds
// ahead of the scalars: a chain of 64 tori 5.3 + 6.1 -> 4.2 + 4.9 us, of which
// an empty launch is 1.9 us each.
// Every workgroup evaluates the same scalars from the same partials in the
// same order, so they agree bit for bit; once the stop test holds every kernel
// returns at once, and the host queues iterations in batches, checking the
// flag of the previous batch while the current one runs.
#include <cmath>
#include <functional>
#include <type_traits>
#include "dmath.h"
#include "world.h"

namespace adb {

// scalars
// (S_KBASE: iterations of the batches before this one; S_BRUN: batched worlds,
// 1 while some scene is above its tolerance; S_RR: the last r.r; S_BB0, S_RR0:
// b.b and the final r.r of the part solved before, see pcg_solve)
enum { S_STOP = 0, S_ITERS, S_BB, S_RZ0, S_RZ1, S_KBASE, S_BRUN, S_RR, S_BB0, S_RR0, S_COUNT };
// stop flag values
enum { RUN = 0, CONVERGED = 1, BREAKDOWN = 2, NONFINITE = 3 };

constexpr int SP_ROWS = 4;       // block rows per spmv workgroup (one 64-lane team each)
// workgroups of an spmv or update launch: all that are resident at once or
// two rounds of them, and no more partials than one round of loads of the
// other kernel's workgroup takes (8 per thread)
constexpr int SPMV_WGS = 1024, UPD_WGS = 2048;
// iterations queued between host checks: w.tune.pcg_batch (even)

// The value of lane i ^ m (m = 32, 16, 8) or, where the lanes of a 16-lane row
// already repeat with period 2 m, of lane i ^ m for m = 4, 2, 1: lane swaps
// and row rotations, which stay in the vector unit.
template <int M> __device__ __forceinline__ double add_lane_xor(double v) {
    int2 a = *reinterpret_cast<int2*>(&v), b;
    if constexpr (M >= 16) {
        // both results of the swap: the lanes' own halves and the others'
        auto lo = M == 32 ? __builtin_amdgcn_permlane32_swap(a.x, a.x, false, false) : __builtin_amdgcn_permlane16_swap(a.x, a.x, false, false);
        auto hi = M == 32 ? __builtin_amdgcn_permlane32_swap(a.y, a.y, false, false) : __builtin_amdgcn_permlane16_swap(a.y, a.y, false, false);
        a = make_int2(lo[0], hi[0]);
        b = make_int2(lo[1], hi[1]);
    } else {
        b.x = __builtin_amdgcn_update_dpp(0, a.x, 0x120 + M, 0xf, 0xf, false);
        b.y = __builtin_amdgcn_update_dpp(0, a.y, 0x120 + M, 0xf, 0xf, false);
    }
    return *reinterpret_cast<double*>(&a) + *reinterpret_cast<double*>(&b);
}
// fixed-order wave sum, in every lane
__device__ __forceinline__ double wave_sum(double v) {
    v = add_lane_xor<32>(v);
    v = add_lane_xor<16>(v);
    v = add_lane_xor<8>(v);
    v = add_lane_xor<4>(v);
    v = add_lane_xor<2>(v);
    return add_lane_xor<1>(v);
}
// Value i of a wavefront's copy of an array (lane k holds value k).
__device__ __forceinline__ double lane_value(double v, int i) {
    const int2 a = *reinterpret_cast<int2*>(&v);
    const int2 b = make_int2(__builtin_amdgcn_readlane(a.x, i), __builtin_amdgcn_readlane(a.y, i));
    double r;
    __builtin_memcpy(&r, &b, 8);
    return r;
}
// Fixed-order sums of n values, the same in every thread of a workgroup of T,
// in two parts: load issues the loads, so the caller can place them among its
// own, done adds.  Each wave sums all the values itself (lane l adds l,
// l + 64, ... in order, then the wave sum); beyond 512 values they are split
// over the workgroup's waves, whose sums are added in wave order behind one
// barrier (SPLIT).  U values per lane, n <= 64 U or T U.
template <int T, int U, bool SPLIT> struct PartSum {
    static constexpr int NT = SPLIT ? T : 64;
    double x[U];
    __device__ __forceinline__ void load(const double* __restrict__ v, int n) {
        const int t = SPLIT ? threadIdx.x : threadIdx.x % 64;
#pragma unroll
        for (int u = 0; u < U; u++) x[u] = v[min(t + NT * u, n - 1)];
    }
    __device__ __forceinline__ double wave(int n) const {
        const int t = SPLIT ? threadIdx.x : threadIdx.x % 64;
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (t + NT * u < n) s += x[u];
        return wave_sum(s);
    }
};
// the waves' sums (SPLIT) added in wave order; one barrier, sh is not reused
template <int T, int NV> __device__ __forceinline__ void add_waves(double (*sh)[NV], double (&v)[NV]) {
    if (threadIdx.x % 64 == 0)
        for (int k = 0; k < NV; k++) sh[threadIdx.x / 64][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
        v[k] = 0.0;
#pragma unroll
        for (int w = 0; w < T / 64; w++) v[k] += sh[w][k];
    }
}
// orders a wave's LDS accesses among its own lanes
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// fixed-order workgroup sum (one value per wave combined in wave order)
__device__ double wg_sum(double v, double* sh) {
    v = wave_sum(v);
    const int w = threadIdx.x / 64, nw = (blockDim.x + 63) / 64;
    __syncthreads();
    if (threadIdx.x % 64 == 0) sh[w] = v;
    __syncthreads();
    double r = 0.0;
    for (int i = 0; i < nw; i++) r += sh[i];
    __syncthreads();
    return r;
}

// Preconditioner of the body groups: z = M_g^-1 r on group g's rows (n = 12
// bodies <= GN); group tables hold B entries, those past *count are unused.
constexpr int GN = 96;
struct Groups {
    const int* off; const int* body; const long long* moff; const double* Minv; const int* count;
    const int* tree; const int* tab;      // trees: the group's table (tree.h) at tab + tree[g]; -1: an explicit inverse
};

// Batched worlds: each scene's residual test, |r_s|^2 <= rtol^2 |b_s|^2, from
// the groups' r.r (groups are numbered scene by scene); first = those of
// iteration 0 (|b_s|^2 = |r_s|^2 then).  One workgroup, SC_L lanes per scene,
// loads in flight together; S_BRUN = 1 while some scene is above its tolerance.
// Solves in two parts: srr takes the first part's |r_s|^2, and the second
// adds it and the first part's |b_s|^2 to its own (a scene whose first part did
// not finish: the second part on its own).
constexpr int SC_L = 4;
__global__ __launch_bounds__(1024) void k_pcg_scene_stop(int S, const int* __restrict__ sc_goff, double rtol2, int first, int part,
                                                         const double* __restrict__ grr, double* __restrict__ sbb,
                                                         double* __restrict__ srr, double* scal) {
    __shared__ int any;
    if (threadIdx.x == 0) any = 0;
    __syncthreads();
    if (scal[S_STOP] == RUN) {
        int mine = 0;
        const int l = threadIdx.x % SC_L;
        for (int s = threadIdx.x / SC_L; s < S; s += blockDim.x / SC_L) {
            const int e = sc_goff[s + 1];
            double rr = 0.0;
            for (int g = sc_goff[s] + l; g < e; g += 8 * SC_L) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = g + SC_L * u < e ? grr[g + SC_L * u] : 0.0;
#pragma unroll
                for (int u = 0; u < 8; u++) rr += v[u];
            }
            for (int m = 1; m < SC_L; m *= 2) rr += __shfl_xor(rr, m);
            double bb = first ? rr : sbb[s], r0 = 0.0;
            if (part == 2) {
                r0 = srr[s];
                if (first) {
                    const double b0 = sbb[s];
                    if (!(r0 <= rtol2 * b0)) r0 = 0.0;
                    bb += b0;
                }
            }
            if (l == 0) {
                if (first) sbb[s] = bb;
                if (part == 1) srr[s] = rr;
                else if (part == 2 && first) srr[s] = r0;
            }
            if (!(rr + r0 <= rtol2 * bb)) mine = 1;
        }
        if (mine) any = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) scal[S_BRUN] = any;
}

// iteration base of the next batch
__global__ void k_pcg_advance(double* scal, int n) { if (threadIdx.x == 0 && blockIdx.x == 0) scal[S_KBASE] += n; }

// A lane's share of one 12 x 12 block of a row: 12 lanes per block (lane r its
// row r), five blocks of the row at a time.
struct RowBlock { double H[12]; double2 z[6], p[6]; };
__device__ __forceinline__ void load_block(RowBlock& b, int k, int col, int r, const double* __restrict__ Hval,
                                           const double* __restrict__ z, const double* __restrict__ pold) {
    const double* H = Hval + 144 * (size_t)k + r;
    const size_t cb = 6 * (size_t)col;
#pragma unroll
    for (int c = 0; c < 12; c++) b.H[c] = H[c * 12];
    const double2* z2 = reinterpret_cast<const double2*>(z) + cb;
    const double2* p2 = reinterpret_cast<const double2*>(pold) + cb;
#pragma unroll
    for (int c = 0; c < 6; c++) { b.z[c] = z2[c]; b.p[c] = p2[c]; }
}
__device__ __forceinline__ double row_product(const RowBlock& b, double beta) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < 6; c++) {
        s += b.H[2 * c] * (b.z[c].x + beta * b.p[c].x);
        s += b.H[2 * c + 1] * (b.z[c].y + beta * b.p[c].y);
    }
    return s;
}
template <int U, bool SPLIT>
__global__ __launch_bounds__(64 * SP_ROWS, U == 8 && !SPLIT ? 3 : 4) void k_pcg_spmv(int B, int kloc, double rtol2, int nbU, int batched,
                                                           const int* __restrict__ row_ptr,
                                                           const int* __restrict__ col_idx, const double* __restrict__ Hval,
                                                           const double* __restrict__ z, const double* __restrict__ pold,
                                                           double* __restrict__ pnew, double* __restrict__ y,
                                                           const double* __restrict__ partB, double* __restrict__ partA,
                                                           double* scal) {
    __shared__ double sh[SP_ROWS], sh2[SP_ROWS][2];
    __shared__ double acc_sh[SP_ROWS][5][12];
    const int team = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int g = lane / 12, r = lane % 12;
    const int stride = gridDim.x * SP_ROWS;
    int row = blockIdx.x * SP_ROWS + team;
    // Three rounds of loads, none of which waits for the scalars: the row's
    // extent (and the next row's), the scalars and the partials; the first
    // block and its column; z and p_old.
    int k0 = 0, k1 = 0;
    if (row < B) { k0 = row_ptr[row]; k1 = row_ptr[row + 1]; }
    int n0 = 0, n1 = 0, ncol = 0;                 // the next row's extent and first column
    if (row + stride < B) { n0 = row_ptr[row + stride]; n1 = row_ptr[row + stride + 1]; }
    const double sc = scal[min(lane, (int)S_COUNT - 1)];
    PartSum<64 * SP_ROWS, U, SPLIT> prz, prr;
    prz.load(partB, nbU);
    prr.load(partB + nbU, nbU);
    RowBlock blk;
    const bool first = g < 5 && k0 + g < k1;
    if (first) load_block(blk, k0 + g, col_idx[k0 + g], r, Hval, z, pold);
    double2 zo = make_double2(0.0, 0.0);          // the row's own z and p_old
    if (row < B && lane < 12) zo = make_double2(z[12 * (size_t)row + lane], pold[12 * (size_t)row + lane]);
    if (lane_value(sc, S_STOP) != RUN) return;
    // scalars of iteration iter - 1 (identical in every wave of every workgroup)
    const int iter = (int)lane_value(sc, S_KBASE) + kloc;
    double rzr[2] = {prz.wave(nbU), prr.wave(nbU)};
    if (SPLIT) add_waves<64 * SP_ROWS>(sh2, rzr);
    const double RZ = rzr[0], RR = rzr[1];
    const double bb = iter == 0 ? RR + lane_value(sc, S_BB0) : lane_value(sc, S_BB);
    int stop = RUN;
    if (!std::isfinite(RR) || !std::isfinite(RZ)) stop = NONFINITE;
    else if (batched ? lane_value(sc, S_BRUN) == 0.0 : RR + lane_value(sc, S_RR0) <= rtol2 * bb) stop = CONVERGED;   // batched: every scene's own test
    else if (!(RZ > 0.0)) stop = BREAKDOWN;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (iter == 0) scal[S_BB] = bb;
        scal[S_RR] = RR;
        scal[S_RZ0 + (iter & 1)] = RZ;
        if (stop != RUN) { scal[S_STOP] = stop; scal[S_ITERS] = iter; }
    }
    if (stop != RUN) return;
    const double beta = iter == 0 ? 0.0 : RZ / lane_value(sc, S_RZ0 + ((iter - 1) & 1));
    double prod = 0.0;
    while (row < B) {
        if (g < 5 && n0 + g < n1) ncol = col_idx[n0 + g];
        if (g < 5) {
            double acc = 0.0;
            if (k0 + g < k1) acc += row_product(blk, beta);
            for (int k = k0 + g + 5; k < k1; k += 5) {
                load_block(blk, k, col_idx[k], r, Hval, z, pold);
                acc += row_product(blk, beta);
            }
            acc_sh[team][g][r] = acc;
        }
        wave_fence();       // a row belongs to one wave
        if (lane < 12) {
            const size_t k = 12 * (size_t)row + lane;
            const double yr = (((acc_sh[team][0][lane] + acc_sh[team][1][lane]) + acc_sh[team][2][lane]) + acc_sh[team][3][lane]) +
                              acc_sh[team][4][lane];
            const double pr = zo.x + beta * zo.y;
            y[k] = yr;
            pnew[k] = pr;
            prod += pr * yr;
        }
        wave_fence();
        row += stride;
        if (row >= B) break;
        k0 = n0; k1 = n1;
        if (g < 5 && k0 + g < k1) load_block(blk, k0 + g, ncol, r, Hval, z, pold);
        if (lane < 12) zo = make_double2(z[12 * (size_t)row + lane], pold[12 * (size_t)row + lane]);
        n0 = n1 = 0;
        if (row + stride < B) { n0 = row_ptr[row + stride]; n1 = row_ptr[row + stride + 1]; }
    }
    prod = wg_sum(prod, sh);
    if (threadIdx.x == 0) partA[blockIdx.x] = prod;
}

// Forms of the update: PLAIN, no tree component (tree.h) in the world; TREES,
// the tree components and, with rest, the other groups; BESIDE, the other
// groups of a world with tree components.  The tree code's registers and
// LDS cost the others 3 us a launch, a tree solve 12 us and more.  The z and p
// of a group that a form leaves out are zero from iteration 0 on, so the
// product with its rows adds nothing; BESIDE keeps its x.
enum { PLAIN = 0, TREES = 1, BESIDE = 2 };
// UPD_T lanes per group: row i = t % GN of the group, column half t / GN of
// z = M^-1 r, the two halves combined in order; groups gi = blockIdx.x,
// + gridDim.x, ....  FIRST: x = 0, r = -g, p_old = 0 (y = the gradient, p
// written) instead of the update of x and r by alpha, and the scalars of a
// new solve.  The loads are issued in three rounds again: group table,
// scalars and partials; body and the lane's part of the inverse (48 values in
// flight); the vectors.
constexpr int UPD_T = 2 * GN, GH = GN / 2;
struct GroupRow { double M[GH]; size_t k; int m, j0, tree; bool on; };      // k: the row's element; columns [j0, j0 + 6 m)
template <int FORM> __device__ __forceinline__ void load_group(GroupRow& q, const Groups& G, int gi, int t, bool rest) {
    const int cnt = *G.count, o0 = G.off[gi], o1 = G.off[gi + 1];
    const double* M = G.Minv + G.moff[gi];
    const int i = t % GN, h = t / GN;
    q.tree = FORM != PLAIN && gi < cnt ? G.tree[gi] : -1;
    q.m = gi < cnt && q.tree < 0 && (FORM != TREES || rest) ? o1 - o0 : 0;
    q.on = i < 12 * q.m;
    q.j0 = h * 6 * q.m;
    q.k = 0;
    if (!q.on) return;
    q.k = 12 * (size_t)G.body[o0 + i / 12] + i % 12;
    M += (size_t)q.j0 * (12 * q.m) + i;
#pragma unroll
    for (int s = 0; s < GN / 12; s++)
        if (s < q.m) {
#pragma unroll
            for (int u = 6 * s; u < 6 * s + 6; u++) q.M[u] = M[u * 12 * q.m];
        }
}
template <bool FIRST, int U, bool SPLIT, int FORM>
__global__ __launch_bounds__(UPD_T) void k_pcg_update(int kloc, int nbS, int rest, int carry, double rtol2, Groups G,
                                                      double* __restrict__ p, const double* __restrict__ y,
                                                      double* __restrict__ x, double* __restrict__ r, double* __restrict__ z,
                                                      const double* __restrict__ partA, double* __restrict__ partB,
                                                      double* __restrict__ grr, double* scal) {
    __shared__ double rs[FORM == TREES ? 12 * TREE_MAX : GN];
    __shared__ int tab[FORM == TREES ? TREE_SOLVE_INTS : 1];
    __shared__ double half2[GN];
    __shared__ double red[UPD_T / 64][2], sh1[UPD_T / 64][1];
    const int t = threadIdx.x;
    double sc = 0.0;
    PartSum<UPD_T, U, SPLIT> pa;
    if (!FIRST) {
        sc = scal[min(t % 64, (int)S_COUNT - 1)];
        pa.load(partA, nbS);
    }
    const int ng = *G.count;
    GroupRow q;
    load_group<FORM>(q, G, blockIdx.x, t, rest);
    const bool vec = t < GN;
    double xk = 0.0, pk = 0.0, yk = 0.0, rk = 0.0;
    if (q.on && vec) {
        yk = y[q.k];
        if (!FIRST) { xk = x[q.k]; pk = p[q.k]; rk = r[q.k]; }
    }
    double alpha = 0.0;
    if (FIRST) {
        if (blockIdx.x == 0 && t == 0) {
            // the second of two parts: what the first left, if it finished
            const double bb = carry ? scal[S_BB] : 0.0, rr = carry && scal[S_RR] <= rtol2 * bb ? scal[S_RR] : 0.0;
            scal[S_BB0] = bb; scal[S_RR0] = rr;
            scal[S_STOP] = RUN; scal[S_ITERS] = 0.0; scal[S_KBASE] = 0.0;
        }
    } else {
        if (lane_value(sc, S_STOP) != RUN) return;
        const int iter = (int)lane_value(sc, S_KBASE) + kloc;
        double s1[1] = {pa.wave(nbS)};
        if (SPLIT) add_waves<UPD_T>(sh1, s1);
        const double pAp = s1[0];
        if (!(pAp > 0.0) || !std::isfinite(pAp)) {
            if (blockIdx.x == 0 && t == 0) { scal[S_STOP] = std::isfinite(pAp) ? BREAKDOWN : NONFINITE; scal[S_ITERS] = iter; }
            return;
        }
        alpha = lane_value(sc, S_RZ0 + (iter & 1)) / pAp;
    }
    double a0 = 0.0, a1 = 0.0;
    for (int gi = blockIdx.x; gi < ng;) {
        double pz = 0.0, pr = 0.0;
        if (FIRST && FORM != PLAIN && (FORM == TREES ? q.tree < 0 && !rest : q.tree >= 0))
            for (int i = 12 * G.off[gi] + t; i < 12 * G.off[gi + 1]; i += UPD_T) {
                const size_t k = 12 * (size_t)G.body[i / 12] + i % 12;
                z[k] = 0.0; p[k] = 0.0;
                if (FORM == TREES) x[k] = 0.0;
            }
        if (FORM == TREES && q.tree >= 0) {
            const int* T = G.tab + q.tree;
            const int ti = tree_solve_ints(T[0], T[1], T[2]);
            for (int i = t; i < ti; i += UPD_T) tab[i] = T[i];
            __syncthreads();
            const TreeTab tt = tree_tab(tab);
            for (int i = t; i < 12 * tt.n; i += UPD_T) {
                const size_t k = 12 * (size_t)tt.body[i / 12] + i % 12;
                const double rn = FIRST ? -y[k] : r[k] - alpha * y[k];
                x[k] = FIRST ? 0.0 : x[k] + alpha * p[k];
                if (FIRST) p[k] = 0.0;
                r[k] = rn;
                rs[i] = rn;
            }
            __syncthreads();
            tree_solve<UPD_T>(tt, G.Minv + G.moff[gi], rs);
            for (int i = t; i < 12 * tt.n; i += UPD_T) {
                const size_t k = 12 * (size_t)tt.body[i / 12] + i % 12;
                const double rn = r[k], zn = rs[i];
                z[k] = zn;
                pz += rn * zn; pr += rn * rn;
            }
        }
        if (q.on && vec) {
            x[q.k] = FIRST ? 0.0 : xk + alpha * pk;
            rk = FIRST ? -yk : rk - alpha * yk;
            if (FIRST) p[q.k] = 0.0;
            r[q.k] = rk;
            rs[t] = rk;
        }
        __syncthreads();
        const int i = t % GN;
        double zi = 0.0;
        if (q.on) {
#pragma unroll
            for (int s = 0; s < GN / 12; s++)
                if (s < q.m) {
#pragma unroll
                    for (int u = 6 * s; u < 6 * s + 6; u++) zi += q.M[u] * rs[q.j0 + u];
                }
        }
        if (!vec && q.on) half2[i] = zi;
        __syncthreads();
        if (vec && q.on) {
            zi += half2[i];
            z[q.k] = zi;
            pz = rk * zi; pr = rk * rk;
        }
        // the next group's loads run under the sums
        const int gj = gi + gridDim.x;
        if (gj < ng) {
            load_group<FORM>(q, G, gj, t, rest);
            if (q.on && vec) {
                yk = y[q.k];
                if (!FIRST) { xk = x[q.k]; pk = p[q.k]; rk = r[q.k]; }
            }
        }
        pz = wave_sum(pz);
        pr = wave_sum(pr);
        if (t % 64 == 0) { red[t / 64][0] = pz; red[t / 64][1] = pr; }
        __syncthreads();
        if (t == 0) {
            double b0 = 0.0, b1 = 0.0;
            for (int w = 0; w < UPD_T / 64; w++) { b0 += red[w][0]; b1 += red[w][1]; }
            a0 += b0; a1 += b1;
            if (grr) grr[gi] = b1;
        }
        gi = gj;
    }
    if (t == 0) { partB[blockIdx.x] = a0; partB[gridDim.x + blockIdx.x] = a1; }
}

static Groups groups_of(World& w) {
    Groups G;
    G.off = w.grp_off; G.body = w.grp_body; G.moff = w.grp_moff; G.Minv = w.Ginv.p; G.count = w.grp_n;
    G.tree = w.grp_tree; G.tab = w.tree_pack.p;
    return G;
}

static int spmv_wgs(int B) { return std::min((B + SP_ROWS - 1) / SP_ROWS, SPMV_WGS); }
static int update_wgs(int B) { return std::min(B, UPD_WGS); }         // at most B groups; their count stays on the device

// kernel k of a batch; the partial counts, so the sums' forms, depend on B only
static void launch_spmv(World& w, int k, const double* pold, double* pnew) {
    const int B = w.B, nbS = spmv_wgs(B), nbU = update_wgs(B);
    double* partA = w.partial.p;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nbS), dim3(64 * SP_ROWS), 0, w.stream, B, k, w.P.pcg_rtol * w.P.pcg_rtol, nbU, (int)(w.S > 1),
                           w.row_ptr.p, w.col_idx.p, w.Hval.p, w.pcg_z.p, pold, pnew, w.pcg_Ap.p, partA + nbS, partA, w.scal.p);
    };
    if (nbU <= 64) go(k_pcg_spmv<1, false>);
    else if (nbU <= 512) go(k_pcg_spmv<8, false>);
    else go(k_pcg_spmv<8, true>);
}
// What one run of the iteration covers: the whole system, its tree
// components or the rest of it (pcg_solve).
enum { WHOLE = 0, TREE_PART = 1, REST_PART = 2 };
static int update_form(const World& w, int part) { return part == REST_PART ? BESIDE : (w.n_trees > 0 ? TREES : PLAIN); }
template <bool FIRST> static void launch_update(World& w, int part, int k, double* p, const double* y) {
    const int B = w.B, nbS = spmv_wgs(B), nbU = update_wgs(B);
    double* partA = w.partial.p;
    double* partB = partA + nbS;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nbU), dim3(UPD_T), 0, w.stream, k, nbS, (int)(part != TREE_PART), (int)(part == REST_PART),
                           w.P.pcg_rtol * w.P.pcg_rtol, groups_of(w), p, y, w.pcg_xo, w.pcg_r.p, w.pcg_z.p,
                           partA, partB, w.S > 1 ? partB + 2 * nbU : (double*)nullptr, w.scal.p);
    };
    auto form = [&](auto f) {
        constexpr int F = decltype(f)::value;
        // (FIRST sums nothing)
        if constexpr (FIRST) go(k_pcg_update<true, 1, false, F>);
        else if (nbS <= 64) go(k_pcg_update<FIRST, 1, false, F>);
        else if (nbS <= 512) go(k_pcg_update<FIRST, 8, false, F>);
        else go(k_pcg_update<FIRST, 8, true, F>);
    };
    switch (update_form(w, part)) {
    case TREES: form(std::integral_constant<int, TREES>{}); break;
    case BESIDE: form(std::integral_constant<int, BESIDE>{}); break;
    default: form(std::integral_constant<int, PLAIN>{});
    }
}
static void launch_scene_stop(World& w, int part, int first) {
    const double* grr = w.partial.p + spmv_wgs(w.B) + 2 * update_wgs(w.B);
    hipLaunchKernelGGL(k_pcg_scene_stop, dim3(1), dim3(1024), 0, w.stream, w.S, w.sc_goff.p, w.P.pcg_rtol * w.P.pcg_rtol, first, part,
                       grr, w.pcg_sbb.p, w.pcg_srr.p, w.scal.p);
}

// One batch = pcg_batch iterations; kernel k of the batch computes iteration
// S_KBASE + k, and the last node advances S_KBASE.  Because the batch is even, the
// p-buffer parity of local iteration k is k & 1 in every batch, so one
// captured graph serves every batch.
static void enqueue_batch(World& w, int part, int nb, bool prof) {
    double* pb[2] = {w.pcg_p.p, w.pcg_p2.p};
    for (int k = 0; k < nb; k++) {
        {
            // H blocks, their column indices, z and p_old read, p_new and y written
            ProfScope ps(w, PK_SPMV, prof ? 1152.0 * w.nnzb + 4.0 * w.nnzb + 4.0 * 96.0 * w.B : 0.0);
            launch_spmv(w, k, pb[k & 1], pb[(k & 1) ^ 1]);
        }
        {
            // the part's inverses or factors read; p, y read; x, r read and written; z written
            const double all = (double)w.h_grp_moff.back(), tree = (double)w.tree_doubles;
            ProfScope ps(w, PK_PCG_UPDATE, prof ? 8.0 * (part == WHOLE ? all : (part == TREE_PART ? tree : all - tree)) + 7.0 * 96.0 * w.B : 0.0);
            launch_update<false>(w, part, k, pb[(k & 1) ^ 1], w.pcg_Ap.p);
        }
        if (w.S > 1) launch_scene_stop(w, part, 0);
    }
    hipLaunchKernelGGL(k_pcg_advance, dim3(1), dim3(64), 0, w.stream, w.scal.p, nb);
}

// A whole batch as a graph, captured when one is first needed and again when a
// buffer it was captured with has moved.  Contact components come and go
// from one iteration to the next, so their number is no part of the key.
static void launch_batch_graph(World& w, int part, int batch) {
    const int form = update_form(w, part);
    World::PcgGraph& gr = w.pcg_graph[form];
    const void* key[] = {w.row_ptr.p, w.col_idx.p, w.Hval.p, w.Ginv.p, w.pcg_xo, w.pcg_r.p, w.pcg_z.p, w.pcg_p.p,
                         w.pcg_p2.p, w.pcg_Ap.p, w.partial.p, w.scal.p, w.grp_off, w.grp_body, w.grp_moff,
                         w.grp_n, w.sc_goff.p, w.pcg_sbb.p, w.pcg_srr.p, form == TREES ? w.tree_pack.p : nullptr};
    static_assert(sizeof key / sizeof key[0] == World::PCG_GRAPH_KEYS, "graph key size");
    bool same = gr.exec != nullptr && gr.batch == batch;
    for (int i = 0; i < World::PCG_GRAPH_KEYS; i++) same = same && gr.key[i] == key[i];
    if (!same) {
        if (gr.exec) { ADB_HIP(hipGraphExecDestroy(gr.exec)); gr.exec = nullptr; }
        hipGraph_t g;
        ADB_HIP(hipStreamBeginCapture(w.stream, hipStreamCaptureModeThreadLocal));
        enqueue_batch(w, part, batch, false);
        ADB_HIP(hipStreamEndCapture(w.stream, &g));
        ADB_HIP(hipGraphInstantiate(&gr.exec, g, nullptr, nullptr, 0));
        ADB_HIP(hipGraphDestroy(g));
        for (int i = 0; i < World::PCG_GRAPH_KEYS; i++) gr.key[i] = key[i];
        gr.batch = batch;
    }
    ADB_HIP(hipGraphLaunch(gr.exec, w.stream));
}

static int solve_part(World& w, int part, double* dq_out, int* iters, const std::function<void()>& after, bool* after_valid) {
    const int B = w.B, n = 12 * B;
    const int nbS = spmv_wgs(B), nbU = update_wgs(B);
    // the iterate x lives in the caller's output (12 B doubles)
    w.pcg_xo = dq_out;
    w.pcg_r.reserve(n); w.pcg_z.reserve(n); w.pcg_p.reserve(n); w.pcg_p2.reserve(n); w.pcg_Ap.reserve(n);
    w.partial.reserve((size_t)nbS + 2 * (size_t)nbU + (w.S > 1 ? (size_t)B : 0)); w.scal.reserve(S_COUNT);
    if (!w.h_scal) ADB_HIP(hipHostMalloc((void**)&w.h_scal, 2 * S_COUNT * sizeof(double), hipHostMallocDefault));
    for (hipEvent_t& e : w.pcg_ev)
        if (!e) ADB_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (w.S > 1) { w.pcg_sbb.reserve(w.S); w.pcg_srr.reserve(w.S); }
    launch_update<true>(w, part, 0, w.pcg_p.p, w.grad.p);
    ADB_HIP(hipGetLastError());
    if (w.S > 1) {
        launch_scene_stop(w, part, 1);
        ADB_HIP(hipGetLastError());
    }
    // batches go out as a captured graph, but not while per-kernel profiling is
    // on, nor with ADB_PCG_GRAPH=0 (for tools that do not support graph capture)
    // (a tree part ends after an iteration or two)
    const bool use_graph = !w.prof.on && w.use_graphs && part != TREE_PART;
    const int BATCH = w.tune.pcg_batch;
    int it = 0, slot = 0;
    bool have_prev = false;
    const int max_it = std::max(w.P.pcg_max_iter, 0);
    // stop test after the last queued update: the spmv of the next iteration
    // tests it first and returns at once when stopped; if not, it does that
    // iteration's spmv, which the next batch's first spmv repeats identically
    // (same iteration, same p-buffer parity: batches are even)
    auto stop_test = [&]() {
        launch_spmv(w, 0, w.pcg_p.p, w.pcg_p2.p);
        ADB_HIP(hipGetLastError());
    };
    // Near the iteration count of the previous solve (Newton steps change the
    // system little) the batches shrink to 4 iterations, so the stop test,
    // read one batch late, leaves few queued iterations that return at once.
    const int pred = part == TREE_PART && w.pcg_prev_its[part] == 0 ? 2 : w.pcg_prev_its[part];
    bool done = false;
    if (pred > 0 && pred <= 4 && max_it > 0) {
        // a short previous solve (the light phase of a scene, where groups are
        // whole components): queue that many iterations (rounded up to even)
        // and test at once, instead of queueing batches ahead of the test
        const int nb0 = std::min(pred + (pred & 1), max_it);
        enqueue_batch(w, part, nb0, w.prof.on);
        it += nb0;
        stop_test();
        ADB_HIP(hipMemcpyAsync(w.h_scal, w.scal.p, S_COUNT * sizeof(double), hipMemcpyDeviceToHost, w.stream));
        // the caller's next work (on x as it stands) is queued ahead of the
        // wait; it is valid when these iterations finished the solve
        if (after) after();
        wait_stream(w);
        done = w.h_scal[S_STOP] != RUN;
        if (after_valid) *after_valid = done && after;
    }
    while (!done && it < max_it) {
        int nb = std::min(BATCH, max_it - it);
        if (pred > 0 && it + BATCH > pred - 8) nb = std::min(nb, 4);
        if (use_graph && nb == BATCH) launch_batch_graph(w, part, BATCH);
        else enqueue_batch(w, part, nb, w.prof.on);
        it += nb;
        ADB_HIP(hipGetLastError());
        ADB_HIP(hipMemcpyAsync(w.h_scal + S_COUNT * slot, w.scal.p, S_COUNT * sizeof(double), hipMemcpyDeviceToHost, w.stream));
        ADB_HIP(hipEventRecord(w.pcg_ev[slot], w.stream));
        if (have_prev) {
            // the batch before this one: stopped already?
            wait_event(w, w.pcg_ev[slot ^ 1]);
            if (w.h_scal[S_COUNT * (slot ^ 1) + S_STOP] != RUN) break;
        }
        have_prev = true;
        slot ^= 1;
    }
    if (!done) {
        stop_test();
        ADB_HIP(hipMemcpyAsync(w.h_scal, w.scal.p, S_COUNT * sizeof(double), hipMemcpyDeviceToHost, w.stream));
        wait_stream(w);
    }
    const double* h = w.h_scal;
    const int stop = (int)h[S_STOP];
    w.pcg_prev_its[part] = stop == RUN ? it : (int)h[S_ITERS];
    *iters += w.pcg_prev_its[part];
    if (stop == NONFINITE) return ADB_E_NAN;
    if (stop == RUN) return ADB_E_NOT_CONVERGED;
    if (stop == BREAKDOWN) return ADB_E_SOLVER;
    return ADB_OK;
}

// The whole system, or its tree components first and then the rest: nothing
// couples them, the tree components are solved after an iteration or two, and
// the rest, where some component is spread over several groups, takes tens
// or hundreds, each of which would repeat the tree solves (8 x 8 cubes in a
// wall, 214 iterations, beside a column of 17: 5137 us a direction against 2790
// in two parts, 3100 with groups of 8 throughout).  The residual test is that
// of the whole: the second part adds what the first left to both its sides.
// Each part has the iteration limit to itself, so that none is refused for the
// other's iterations; the count returned is their sum.
int pcg_solve(World& w, double* dq_out, int* iters, const std::function<void()>& after, bool* after_valid) {
    if (after_valid) *after_valid = false;
    int it = 0, rc;
    if (w.n_trees > 0 && w.tree_rest) {
        const int r1 = solve_part(w, TREE_PART, dq_out, &it, nullptr, nullptr);
        rc = r1 == ADB_E_NAN ? r1 : solve_part(w, REST_PART, dq_out, &it, after, after_valid);
        if (rc != ADB_E_NAN && r1 != ADB_OK) rc = r1;
    } else {
        rc = solve_part(w, WHOLE, dq_out, &it, after, after_valid);
    }
    if (iters) *iters = it;
    return rc;
}

} // namespace adb
