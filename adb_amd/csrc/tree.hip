// tree.hip - block Cholesky factors of the preconditioner's tree components
// (tree.h).  One workgroup per component, a few microseconds per elimination
// round: the bodies of a round are independent, and what bounds it is the
// chain D_j -> L_j -> V_ij (three barriers, the 12 pivots of L_j the longest
// link), not the few hundred blocks of 1.2 KB a component reads and writes.
// Two chains of 32 tori (5 rounds) 80 us and 100 rows of 100 cards (7 rounds)
// 180 us, against 73 and 264 us for the explicit inverses of groups of 8 that
// left 160 and 124 PCG iterations (9 and 32 us each).
//
// A pivot that is not positive and finite (a matrix that is not positive
// definite, or a Schur complement lost to rounding between contacts 1e16 times
// stiffer than the inertia) gives way to the matrix's own diagonal entry there:
// the factors are those of the matrix with that entry raised, a change of rank
// one that costs PCG a few iterations, whatever the component's size.  With the
// inverse diagonal in place of the whole factor a column of 40 cubes with one
// such contact ran to the limit of 2000.
#include "dmath.h"
#include "tree.h"
#include "world.h"

namespace adb {

typedef double d4 __attribute__((ext_vector_type(4)));

// acc -= X Y^T of two column-major 12 x 12 blocks, v_mfma_f64_16x16x4: operand
// lane l holds row l % 16 (rows 12..15 zero) and column k + l / 16; result
// register q of lane l is entry (4 q + l / 16, l % 16)
__device__ __forceinline__ void sub_xyt(const double* X, const double* Y, int lane, d4& acc) {
    const int i = lane % 16, k = lane / 16;
    double x[3], y[3];
#pragma unroll
    for (int s = 0; s < 3; s++) {
        x[s] = i < 12 ? -X[12 * (4 * s + k) + i] : 0.0;
        y[s] = i < 12 ? Y[12 * (4 * s + k) + i] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 3; s++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s], y[s], acc, 0, 0, 0);
}
__device__ __forceinline__ void load_acc(const double* X, int lane, d4& acc) {
#pragma unroll
    for (int q = 0; q < 3; q++) acc[q] = X && lane % 16 < 12 ? X[12 * (lane % 16) + 4 * q + lane / 16] : 0.0;
    acc[3] = 0.0;
}
__device__ __forceinline__ void store_acc(double* X, int lane, const d4& acc) {
    if (lane % 16 < 12)
#pragma unroll
        for (int q = 0; q < 3; q++) X[12 * (lane % 16) + 4 * q + lane / 16] = acc[q];
}

// 1 / sqrt(x) from the hardware approximation and two Newton steps: a rounding
// more than IEEE is nothing to a preconditioner, and the pivots wait for it
__device__ __forceinline__ double rsq2(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    y = fma(y, fma(-h * y, y, 0.5), y);
    return fma(y, fma(-h * y, y, 0.5), y);
}
struct TreeArgs {
    const int* list;                 // the tree groups
    const int* tab; const int* grp_tree; const long long* grp_moff;
    const int* pair_up; const int* pair_low; const int* diag_blk;
    const double* Hval;
    double* Ginv;
};
constexpr int TREE_T = 512, TREE_U = 4;
__global__ __launch_bounds__(TREE_T) void k_tree_factor(TreeArgs a) {
    const int g = a.list[blockIdx.x];
    // the table, but for the contribution lists, in LDS: its indices are links
    // of every chain of loads below
    __shared__ int tab[TREE_FACTOR_INTS];
    const int* T = a.tab + a.grp_tree[g];
    const int ti = tree_solve_ints(T[0], T[1], T[2]) + 2 * T[2] + 1;
    for (int i = threadIdx.x; i < ti; i += TREE_T) tab[i] = T[i];
    __syncthreads();
    TreeTab t = tree_tab(tab);
    t.cona = T + ti;
    t.conb = t.cona + t.nc;
    double* F = a.Ginv + a.grp_moff[g];
    double* V = F + 144 * (size_t)t.n;
    const int lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    for (int l = 0; l < t.nlev; l++) {
        const int p0 = t.lev[l], np = t.lev[l + 1] - p0, e0 = t.up[p0], ne = t.up[p0 + np] - e0;
        // D_j and A_ij = H_ij - sum V V^T of the round's columns, TREE_U blocks
        // a wavefront at a time (their loads in flight together)
        for (int s0 = wv * TREE_U; s0 < np + ne; s0 += TREE_T / 64 * TREE_U) {
            d4 acc[TREE_U];
#pragma unroll
            for (int u = 0; u < TREE_U; u++) {
                const int s = s0 + u, q = s < np ? 0 : (s < np + ne ? t.src[e0 + s - np] : -1);
                const int k = s < np ? a.diag_blk[t.body[p0 + s]] : (q < 0 ? -1 : (q & 1 ? a.pair_low[q >> 1] : a.pair_up[q >> 1]));
                load_acc(k < 0 ? nullptr : a.Hval + 144 * (size_t)k, lane, acc[u]);
            }
#pragma unroll
            for (int u = 0; u < TREE_U; u++) {
                const int s = s0 + u;
                if (s < np) {
                    const int j = p0 + s;
                    for (int x = t.low[j]; x < t.low[j + 1]; x++) {
                        const double* v = V + 144 * (size_t)t.lowe[x];
                        sub_xyt(v, v, lane, acc[u]);
                    }
                    store_acc(F + 144 * (size_t)j, lane, acc[u]);
                } else if (s < np + ne) {
                    const int e = e0 + s - np;
                    for (int x = t.con[e]; x < t.con[e + 1]; x++)
                        sub_xyt(V + 144 * (size_t)t.cona[x], V + 144 * (size_t)t.conb[x], lane, acc[u]);
                    store_acc(V + 144 * (size_t)e, lane, acc[u]);
                }
            }
        }
        __syncthreads();
        // L_j and L_j^-1, 12 lanes a body, lane r holding the rows r of the
        // matrix and of the inverse; five bodies per wavefront
        for (int s = wv * 5; s < np; s += TREE_T / 64 * 5) {
            const int m = lane / 12, r = lane % 12, j = p0 + s + m;
            const bool on = lane < 60 && s + m < np;
            double v[12], x[12];
#pragma unroll
            for (int c = 0; c < 12; c++) {
                v[c] = on ? F[144 * (size_t)j + 12 * c + r] : (c == r ? 1.0 : 0.0);
                x[c] = c == r ? 1.0 : 0.0;
            }
#pragma unroll
            for (int k = 0; k < 12; k++) {
                const int row = min(12 * m, 48);
                double d = __shfl(v[k], row + k);
                if (!(d > 0.0 && d < INFINITY)) {
                    d = on ? fabs(a.Hval[144 * (size_t)a.diag_blk[t.body[j]] + 13 * k]) : 1.0;
                    if (!(d > 0.0 && d < INFINITY)) d = 1.0;
                }
                const double inv = rsq2(d), f = v[k] * inv;            // L_rk
                v[k] = f;
#pragma unroll
                for (int c = k + 1; c < 12; c++) v[c] -= f * __shfl(f, row + c);
#pragma unroll
                for (int c = 0; c <= k; c++) {
                    const double y = __shfl(x[c], row + k) * inv;
                    x[c] = r == k ? y : (r > k ? x[c] - f * y : x[c]);
                }
            }
            // row r of L^-1, and row r of L as column r above the diagonal
            if (on)
#pragma unroll
                for (int c = 0; c < 12; c++) {
                    if (c <= r) F[144 * (size_t)j + 12 * c + r] = x[c];
                    if (c < r) F[144 * (size_t)j + 12 * r + c] = v[c];
                }
        }
        __syncthreads();
        // V_ij = A_ij L_j^-T by substitution, 12 lanes a block, lane r its row r
        for (int s = wv * 5; s < ne; s += TREE_T / 64 * 5) {
            const int r = lane % 12, e = e0 + s + lane / 12;
            if (lane < 60 && e < e0 + ne) {
                double* B = V + 144 * (size_t)e + r;
                const double* L = F + 144 * (size_t)t.own[e];
                double v[12];
#pragma unroll
                for (int c = 0; c < 12; c++) v[c] = B[12 * c];
#pragma unroll
                for (int c = 0; c < 12; c++) {
#pragma unroll
                    for (int d = 0; d < c; d++) v[c] -= v[d] * L[12 * c + d];
                    v[c] *= L[13 * c];
                }
#pragma unroll
                for (int c = 0; c < 12; c++) B[12 * c] = v[c];
            }
        }
        __syncthreads();
    }
}

// factors of the tree groups (build_groups queued their tables' upload)
void tree_factor(World& w) {
    if (w.n_trees == 0) return;
    TreeArgs a;
    a.list = w.tree_list; a.tab = w.tree_pack.p;
    a.grp_tree = w.grp_tree; a.grp_moff = w.grp_moff;
    a.pair_up = w.pair_up.p; a.pair_low = w.pair_low.p; a.diag_blk = w.diag_blk.p;
    a.Hval = w.Hval.p; a.Ginv = w.Ginv.p;
    hipLaunchKernelGGL(k_tree_factor, dim3(w.n_trees), dim3(TREE_T), 0, w.stream, a);
    ADB_HIP(hipGetLastError());
}

} // namespace adb
