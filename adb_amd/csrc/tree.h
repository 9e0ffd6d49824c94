// tree.h - exact preconditioner blocks for whole contact components: the
// elimination plan (host), its table, and the solve with the factors.
//
// The contact graph of a settling scene falls into components that are trees
// or nearly so (rows of leaning cards, chains, stacks: as many pairs as
// bodies less one).  Their diagonal sub-matrix has a block Cholesky factor with hardly
// more blocks than the matrix, so a component is one preconditioner group and
// the preconditioned system decouples: PCG ends after one or two iterations.
// Groups of at most GMAX bodies left 160 iterations on two chains of 32 tori
// and 124 on rows of 100 cards.
//
// Plan: bodies are eliminated in rounds.  A round takes bodies no two of which
// are neighbours, of at most two neighbours each where there are any (of the
// fewest otherwise), so a path of n takes about log2 n rounds and the bodies
// of a round are independent work.  Eliminating a body joins its neighbours
// pairwise.  A component whose cheapest body has more than TREE_DEG
// neighbours, or with more than TREE_MAX bodies, keeps the small groups.
//
// Factors (left-looking, positions in the elimination order):
//     L_j L_j^T = H_jj - sum_k V_jk V_jk^T,   V_ij = (H_ij - sum_k V_ik V_jk^T) L_j^-T
// over the bodies k eliminated before j that neighbour both.  Triangular, not
// D^-1: contacts are 1e5 times stiffer than the inertia and more, and the
// Schur complements lose the square of that ratio through an explicit inverse.
#pragma once
#include <hip/hip_runtime.h>
#include <vector>

namespace adb {

// Components of at most TREE_MIN bodies keep two or three small groups, so that
// the iteration counts which callers (and the tests of truncated solves) see
// on small stacks stay what they were.  Speed is no reason: with factors from 9
// bodies on a direction of one column of 10 cubes takes 326 us instead of 483,
// of 200 of them 636 instead of 2258, of 80 walls of 3 x 4 717 instead of 1198.
constexpr int TREE_MIN = 16;
constexpr int TREE_MAX = 256;        // bodies of a component: its vector stays in LDS
constexpr int TREE_DEG = 8;          // neighbours of a body when it is eliminated
constexpr int TREE_FILL = 6;         // blocks below the diagonal per body
// iteration limits below this keep the small groups, whose truncated iterates
// (and reports of them) are what a caller with such a limit has asked for
constexpr int TREE_MIN_ITER = 16;

// One component's table, ints from T on.  A "block" e is a block below the
// diagonal of column own[e], row node[e] (positions), blocks in column order.
// Its doubles, 144 a block, column-major: of each body L_j^-1 in the lower
// triangle and L_j^T above the diagonal, then V of the ne blocks.
struct TreeTab {
    int n, nlev, ne, nc;
    const int* lev;                  // nlev + 1: first position of each round
    const int* body;                 // n: body at a position
    const int* up;                   // n + 1: first block of each column
    const int* node; const int* own; // ne
    const int* low;                  // n + 1: first entry of lowe of each row
    const int* lowe;                 // ne: the blocks of a row, in block order
    // (up to here what the solve reads)
    const int* src;                  // ne: 2 pair + (0: BSR block (lo, hi), 1: (hi, lo)); -1: no contacts of its own
    const int* con;                  // ne + 1: first entry of cona / conb of each block
    const int* cona; const int* conb;     // nc: the block loses V_cona V_conb^T
};
constexpr int TREE_HEAD = 4;
__host__ __device__ constexpr int tree_solve_ints(int n, int nlev, int ne) { return TREE_HEAD + nlev + 1 + n + 2 * (n + 1) + 3 * ne; }
constexpr int TREE_SOLVE_INTS = tree_solve_ints(TREE_MAX, TREE_MAX, TREE_FILL * TREE_MAX);
constexpr int TREE_FACTOR_INTS = TREE_SOLVE_INTS + 2 * TREE_FILL * TREE_MAX + 1;
__host__ __device__ __forceinline__ TreeTab tree_tab(const int* T) {
    TreeTab t;
    t.n = T[0]; t.nlev = T[1]; t.ne = T[2]; t.nc = T[3];
    const int* q = T + TREE_HEAD;
    t.lev = q; q += t.nlev + 1;
    t.body = q; q += t.n;
    t.up = q; q += t.n + 1;
    t.node = q; q += t.ne;
    t.own = q; q += t.ne;
    t.low = q; q += t.n + 1;
    t.lowe = q; q += t.ne;
    t.src = q; q += t.ne;
    t.con = q; q += t.ne + 1;
    t.cona = q; q += t.nc;
    t.conb = q;
    return t;
}

// Host: the plan of one component.
struct TreePlan {
    struct Half { int to, edge; };
    struct Con { int a, b, next; };          // edge {u, v}, u < v: the edges (u, k), (v, k) of an eliminated k
    std::vector<std::vector<Half>> adj;
    std::vector<int> eu, ev, esrc, ehead, etail, alive, pos, blocked, lev, seq, upp, upe, slot;
    std::vector<Con> cons;

    void start(int n) {
        if ((int)adj.size() < n) adj.resize(n);
        for (int u = 0; u < n; u++) adj[u].clear();
        eu.clear(); ev.clear(); esrc.clear(); ehead.clear(); etail.clear(); cons.clear();
    }
    // pair p between local bodies u < v (u the pair's lo body); src = 2 p or -1
    int edge(int u, int v, int src) {
        const int e = (int)eu.size();
        eu.push_back(u); ev.push_back(v); esrc.push_back(src); ehead.push_back(-1); etail.push_back(-1);
        adj[u].push_back({v, e});
        adj[v].push_back({u, e});
        return e;
    }
    // appends the table of the component of n bodies (global ids bodies[0..n),
    // ascending) to out; false (nothing appended) when its elimination would
    // fill in too much
    bool finish(int n, const int* bodies, std::vector<int>& out) {
        alive.resize(n); pos.assign(n, -1); blocked.assign(n, -1);
        lev.clear(); seq.clear(); upp.clear(); upe.clear();
        for (int u = 0; u < n; u++) alive[u] = u;
        upp.push_back(0);
        for (int round = 0; !alive.empty(); round++) {
            size_t dmin = ~(size_t)0;
            for (int u : alive) dmin = adj[u].size() < dmin ? adj[u].size() : dmin;
            if (dmin > TREE_DEG) return false;
            const size_t lim = dmin > 2 ? dmin : 2;
            const int first = (int)seq.size();
            lev.push_back(first);
            for (int u : alive) {
                if (blocked[u] == round || adj[u].size() > lim) continue;
                pos[u] = (int)seq.size();
                seq.push_back(u);
                for (const Half& h : adj[u]) blocked[h.to] = round;
            }
            for (int q = first; q < (int)seq.size(); q++) {
                const int k = seq[q];
                std::vector<Half>& L = adj[k];
                for (const Half& h : L) {
                    upe.push_back(h.edge);
                    std::vector<Half>& M = adj[h.to];
                    for (size_t i = 0; i < M.size(); i++)
                        if (M[i].to == k) { M.erase(M.begin() + i); break; }
                }
                upp.push_back((int)upe.size());
                for (size_t x = 0; x < L.size(); x++)
                    for (size_t y = x + 1; y < L.size(); y++) {
                        const Half a = L[x].to < L[y].to ? L[x] : L[y], b = L[x].to < L[y].to ? L[y] : L[x];
                        int e = -1;
                        for (const Half& h : adj[a.to])
                            if (h.to == b.to) { e = h.edge; break; }
                        if (e < 0) e = edge(a.to, b.to, -1);
                        cons.push_back({a.edge, b.edge, -1});
                        const int c = (int)cons.size() - 1;
                        if (ehead[e] < 0) ehead[e] = c; else cons[etail[e]].next = c;
                        etail[e] = c;
                    }
                if ((int)eu.size() > TREE_FILL * n) return false;
            }
            size_t keep = 0;
            for (int u : alive)
                if (pos[u] < 0) alive[keep++] = u;
            alive.resize(keep);
        }
        lev.push_back(n);
        const int ne = (int)upe.size(), nc = (int)cons.size();
        slot.resize(eu.size());
        for (int s = 0; s < ne; s++) slot[upe[s]] = s;
        const size_t at = out.size();
        out.resize(at + TREE_HEAD + lev.size() + n + 2 * (size_t)(n + 1) + 4 * (size_t)ne + ne + 1 + 2 * (size_t)nc);
        int* T = out.data() + at;
        T[0] = n; T[1] = (int)lev.size() - 1; T[2] = ne; T[3] = nc;
        int* q = T + TREE_HEAD;
        for (int v : lev) *q++ = v;
        for (int p = 0; p < n; p++) *q++ = bodies[seq[p]];
        for (int v : upp) *q++ = v;
        int* node = q; q += ne;
        int* own = q; q += ne;
        int* low = q; q += n + 1;
        int* lowe = q; q += ne;
        int* src = q; q += ne;
        int* con = q; q += ne + 1;
        int* cona = q; q += nc;
        int* conb = q;
        for (int p = 0; p <= n; p++) low[p] = 0;
        int c = 0;
        for (int j = 0; j < n; j++)
            for (int s = upp[j]; s < upp[j + 1]; s++) {
                const int e = upe[s], u = seq[j], v = eu[e] == u ? ev[e] : eu[e];
                node[s] = pos[v]; own[s] = j;
                // row v, column u: (lo, hi) when v is the pair's lo body
                src[s] = esrc[e] < 0 ? -1 : esrc[e] + (v == eu[e] ? 0 : 1);
                low[pos[v] + 1]++;
                con[s] = c;
                for (int i = ehead[e]; i >= 0; i = cons[i].next) {
                    // cons: a is the edge of eu[e] (the smaller), b that of ev[e]
                    cona[c] = slot[v == eu[e] ? cons[i].a : cons[i].b];
                    conb[c] = slot[v == eu[e] ? cons[i].b : cons[i].a];
                    c++;
                }
            }
        con[ne] = c;
        for (int p = 0; p < n; p++) low[p + 1] += low[p];
        // rows' blocks in block order (upp is free to hold the fill positions)
        upp.assign(low, low + n);
        for (int s = 0; s < ne; s++) lowe[upp[node[s]]++] = s;
        return true;
    }
    static long long doubles(int n, int ne) { return 144ll * (n + (long long)ne); }
};

// a team of 12 lanes lies in one wavefront: only the order of its LDS accesses matters
__device__ __forceinline__ void team_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Device: rs (LDS, 12 n, by position) <- M^-1 rs with the factors F, by the
// workgroup's NT lanes in teams of 12 (five per wavefront).  Bound by the
// rounds' dependent loads: two passes over the rounds, one barrier each.
template <int NT> __device__ __forceinline__ void tree_solve(const TreeTab& t, const double* F, double* rs) {
    constexpr int TEAMS = NT / 64 * 5;
    const int lane = threadIdx.x % 64, team = threadIdx.x / 64 * 5 + lane / 12, r = lane % 12;
    const double* V = F + 144 * (size_t)t.n;
    // y_j = L_j^-1 (r_j - sum V_jk y_k), then z_j = L_j^-T (y_j - sum V_ij^T z_i)
    for (int l = 0; l < t.nlev; l++) {
        const int p1 = t.lev[l + 1];
        for (int q = t.lev[l]; q < p1; q += TEAMS) {
            const int j = q + team;
            const bool on = lane < 60 && j < p1;
            double s = 0.0, d[12];
            if (on) {
#pragma unroll
                for (int c = 0; c < 12; c++) d[c] = F[144 * (size_t)j + 12 * c + r];
                s = rs[12 * j + r];
                for (int x = t.low[j]; x < t.low[j + 1]; x++) {
                    const int e = t.lowe[x];
                    const double* w = V + 144 * (size_t)e + r;
                    const double* v = rs + 12 * t.own[e];
#pragma unroll
                    for (int c = 0; c < 12; c++) s -= w[12 * c] * v[c];
                }
                rs[12 * j + r] = s;
            }
            team_fence();
            if (on) {
                s = 0.0;
#pragma unroll
                for (int c = 0; c < 12; c++)
                    if (c <= r) s += d[c] * rs[12 * j + c];
            }
            team_fence();
            if (on) rs[12 * j + r] = s;
        }
        __syncthreads();
    }
    for (int l = t.nlev - 1; l >= 0; l--) {
        const int p1 = t.lev[l + 1];
        for (int q = t.lev[l]; q < p1; q += TEAMS) {
            const int j = q + team;
            const bool on = lane < 60 && j < p1;
            double s = 0.0, d[12];
            if (on) {
#pragma unroll
                for (int c = 0; c < 12; c++) d[c] = F[144 * (size_t)j + 12 * r + c];
                s = rs[12 * j + r];
                for (int e = t.up[j]; e < t.up[j + 1]; e++) {
                    const double* w = V + 144 * (size_t)e + 12 * r;
                    const double* v = rs + 12 * t.node[e];
#pragma unroll
                    for (int c = 0; c < 12; c++) s -= w[c] * v[c];
                }
                rs[12 * j + r] = s;
            }
            team_fence();
            if (on) {
                s = 0.0;
#pragma unroll
                for (int c = 0; c < 12; c++)
                    if (c >= r) s += d[c] * rs[12 * j + c];
            }
            team_fence();
            if (on) rs[12 * j + r] = s;
        }
        __syncthreads();
    }
}

} // namespace adb
