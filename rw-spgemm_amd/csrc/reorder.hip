// reorder.hip -- matrix orderings and permutations on the device.
//
//  * degree order: vertices sorted by (-degree, id)
//    (reorder_algorithm/common/order_utils.py:78-81)
//  * Cuthill-McKee / RCM on the symmetrised pattern, the structure of the
//    reference's native_rcm (order_utils.py:84-104) with every tie broken by
//    (degree, id): components are labelled by their lowest-(degree, id)
//    vertex, all components are traversed by one multi-source
//    level-synchronous BFS (a vertex is claimed by its first parent in
//    level order, children ordered by (parent, degree, id)), and the
//    concatenated levels are grouped by component and reversed.
//  * seeded random order
//  * P*A*Q^T with sorted rows: apply_bipermutation_csr / restore
//    (src/reorder.h:2429-2551), done with the library's radix sort.
#include <string.h>

#include "tsg_internal.h"

static int bits_of(long long v) {
    int b = 1;
    while ((1ll << b) <= v) b++;
    return b;
}

__global__ void k_iota2(int *v, long long n) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) v[i] = (int)i;
}
__global__ void k_scatter_inverse(const int *__restrict__ old_id, int n, int *__restrict__ new_id) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) new_id[old_id[i]] = i;
}
__global__ void k_gather_i32_r(const int *__restrict__ src, const int *__restrict__ idx, int n, int *__restrict__ dst) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[idx[i]];
}
__global__ void k_perm_check(const int *__restrict__ p, int n, int *__restrict__ seen, int *__restrict__ bad) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int v = p[i];
    if (v < 0 || v >= n) { atomicOr(bad, 1); return; }
    if (atomicAdd(&seen[v], 1) != 0) atomicOr(bad, 1);
}

// TSG_OK when d_perm[0..n) is a permutation of 0..n-1.
extern "C" int tsg_perm_validate(tsg_ctx *ctx, int n, const int *d_perm) {
    if (n <= 0) return TSG_OK;
    int *seen;
    TSG_TRY(tsg_alloc_t(ctx, &seen, (size_t)n + 1));
    TSG_HIP(hipMemsetAsync(seen, 0, ((size_t)n + 1) * 4, ctx->stream));
    hipLaunchKernelGGL(k_perm_check, dim3(tsg_div_up(n, 256)), dim3(256), 0, ctx->stream, d_perm, n, seen, seen + n);
    TSG_LAUNCH_CHECK();
    long long bad = 0;
    TSG_TRY(tsg_read_scalar_i64(ctx, seen + n, 0, &bad));
    tsg_free(ctx, seen);
    if (bad) { tsg_set_error("not a permutation of 0..%d", n - 1); return TSG_ERR_ARG; }
    return TSG_OK;
}

extern "C" int tsg_perm_invert(tsg_ctx *ctx, int n, const int *d_old_id, int *d_new_id) {
    if (n > 0) {
        hipLaunchKernelGGL(k_scatter_inverse, dim3(tsg_div_up(n, 256)), dim3(256), 0, ctx->stream, d_old_id, n, d_new_id);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

// ------------------------------------------------------------------ degree
__global__ void k_rowlen(const int *__restrict__ rowptr, int m, int *__restrict__ deg) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < m) deg[i] = rowptr[i + 1] - rowptr[i];
}
__global__ void k_mirror_deg(const int *__restrict__ rowptr, const int *__restrict__ col, int m, int *__restrict__ deg) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    for (int e = rowptr[i]; e < rowptr[i + 1]; e++)
        if (col[e] != i) atomicAdd(&deg[col[e]], 1);
}
// (few large blocks: the atomics on one address are what this costs)
__global__ void __launch_bounds__(1024)
k_max_i32(const int *__restrict__ v, int n, int *__restrict__ out) {
    __shared__ int s_m[16];
    int mx = 0;
    for (int i = blockIdx.x * 1024 + threadIdx.x; i < n; i += gridDim.x * 1024) mx = max(mx, v[i]);
    mx = tsg_wave_max(mx);
    if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) mx = max(mx, s_m[w]);
        atomicMax(out, mx);
    }
}
__global__ void k_deg_key(const int *__restrict__ deg, int n, int maxdeg, int descending, unsigned *__restrict__ key) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) key[i] = descending ? (unsigned)(maxdeg - deg[i]) : (unsigned)deg[i];
}

static int max_of(tsg_ctx *ctx, const int *v, int n, int *out) {
    void *scr;
    TSG_TRY(tsg_scratch(ctx, 64, &scr));
    TSG_HIP(hipMemsetAsync(scr, 0, 4, ctx->stream));
    if (n > 0) {
        hipLaunchKernelGGL(k_max_i32, dim3(std::min<unsigned>(64, tsg_div_up(n, 1024))), dim3(1024), 0, ctx->stream, v, n,
                           (int *)scr);
        TSG_LAUNCH_CHECK();
    }
    long long m;
    TSG_TRY(tsg_read_scalar_i64(ctx, scr, 0, &m));
    *out = (int)m;
    return TSG_OK;
}

// ids sorted by degree (ascending or descending), ties by ascending id
static int sort_ids_by_degree(tsg_ctx *ctx, const int *deg, int n, int descending, int *ids, int *most = nullptr) {
    int maxdeg = 0;
    TSG_TRY(max_of(ctx, deg, n, &maxdeg));
    if (most) *most = maxdeg;
    unsigned *key;
    TSG_TRY(tsg_alloc_t(ctx, &key, (size_t)n + 1));
    if (n > 0) {
        hipLaunchKernelGGL(k_deg_key, dim3(tsg_div_up(n, 256)), dim3(256), 0, ctx->stream, deg, n, maxdeg, descending, key);
        hipLaunchKernelGGL(k_iota2, dim3(tsg_div_up(n, 256)), dim3(256), 0, ctx->stream, ids, (long long)n);
        TSG_LAUNCH_CHECK();
        TSG_TRY(tsg_sort_pairs_u32(ctx, key, ids, n, bits_of(maxdeg)));
    }
    tsg_free(ctx, key);
    return TSG_OK;
}

extern "C" int tsg_order_degree(tsg_ctx *ctx, const tsg_dcsr *a, int symmetric_header, int *d_old_id) {
    if (a->m != a->n) { tsg_set_error("degree order needs a square matrix"); return TSG_ERR_ARG; }
    // only row lengths (and, for the mirror count, column ids) are read:
    // a CSR straight from mmio_allinone, repeated entries included, is
    // ranked by its row lengths as given
    TSG_TRY(tsg_validate_csr_mode(ctx, a, 0));
    int *deg;
    TSG_TRY(tsg_alloc_t(ctx, &deg, (size_t)a->m + 1));
    const unsigned g = tsg_div_up(a->m, 256);
    if (a->m > 0) {
        hipLaunchKernelGGL(k_rowlen, dim3(g), dim3(256), 0, ctx->stream, a->rowptr, a->m, deg);
        if (symmetric_header) hipLaunchKernelGGL(k_mirror_deg, dim3(g), dim3(256), 0, ctx->stream, a->rowptr, a->colidx, a->m, deg);
        TSG_LAUNCH_CHECK();
    }
    TSG_TRY(sort_ids_by_degree(ctx, deg, a->m, 1, d_old_id));
    tsg_free(ctx, deg);
    return TSG_OK;
}

// ------------------------------------------------------------------ random
__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
    x += 0x9e3779b97f4a7c15ULL;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ULL;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebULL;
    return x ^ (x >> 31);
}
__global__ void k_rand_key(int n, unsigned long long seed, unsigned long long *__restrict__ key, int *__restrict__ ids) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    // high bits random, low bits the id: distinct keys, uniform order
    key[i] = (mix64(seed ^ mix64((unsigned long long)i)) & 0xffffffff00000000ULL) | (unsigned)i;
    ids[i] = i;
}

extern "C" int tsg_order_random(tsg_ctx *ctx, int n, unsigned long long seed, int *d_old_id) {
    unsigned long long *key;
    TSG_TRY(tsg_alloc_t(ctx, &key, (size_t)n + 1));
    if (n > 0) {
        hipLaunchKernelGGL(k_rand_key, dim3(tsg_div_up(n, 256)), dim3(256), 0, ctx->stream, n, seed, key, d_old_id);
        TSG_LAUNCH_CHECK();
        TSG_TRY(tsg_sort_pairs_u64(ctx, key, d_old_id, n, 64));
    }
    tsg_free(ctx, key);
    return TSG_OK;
}

// ------------------------------------------------------------------ symmetrised pattern
__global__ void k_fill_f64(double *v, long long n, double x) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) v[i] = x;
}

// First index in [lo, hi) with list[index] >= key.
__device__ __forceinline__ int lower_bound_r(const int *__restrict__ list, int lo, int hi, int key) {
    while (lo < hi) {
        const int mid = (int)(((unsigned)lo + (unsigned)hi) >> 1);
        if (list[mid] < key) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Union of two sorted rows, L lanes per row: an entry's place is its index
// plus the other row's smaller entries, less those of both rows before it.
// (One thread merging a row: 27-point mesh of 230k rows 357 -> 87 us with 16.
// Rows of one entry, 4,000,000 of them: 16 lanes 433 us, 4 lanes 150.)
template <bool FILL, int L>
__global__ void __launch_bounds__(256)
k_union_rows(int m, const int *__restrict__ ap, const int *__restrict__ ac, const int *__restrict__ tp,
             const int *__restrict__ tc, int *__restrict__ cnt_or_ptr, int *__restrict__ gc) {
    const unsigned i = tsg_block() * (256 / L) + threadIdx.x / L, l = threadIdx.x % L, gb = (threadIdx.x & 63) / L * L;
    if (i >= (unsigned)m) return;  // whole groups
    const unsigned lanes = (1u << L) - 1u;
    const int a0 = ap[i], a1 = ap[i + 1], b0 = tp[i], b1 = tp[i + 1];
    const int out = FILL ? cnt_or_ptr[i] : 0;
    int both = 0;  // entries of both rows so far
    for (int e0 = a0; e0 < a1; e0 += L) {
        const int e = e0 + l;
        bool dup = false;
        int x = 0, at = 0;
        if (e < a1) {
            x = ac[e];
            at = lower_bound_r(tc, b0, b1, x);
            dup = at < b1 && tc[at] == x;
        }
        const unsigned d = (unsigned)(__ballot(dup) >> gb) & lanes;
        if (FILL && e < a1) gc[out + (e - a0) + (at - b0) - both - __popc(d & ((1u << l) - 1u))] = x;
        both += __popc(d);
    }
    if (!FILL) {
        if (l == 0) cnt_or_ptr[i] = (a1 - a0) + (b1 - b0) - both;
        return;
    }
    both = 0;
    for (int e0 = b0; e0 < b1; e0 += L) {  // entries of the second row alone
        const int e = e0 + l;
        bool dup = false;
        int x = 0, at = 0;
        if (e < b1) {
            x = tc[e];
            at = lower_bound_r(ac, a0, a1, x);
            dup = at < a1 && ac[at] == x;
        }
        const unsigned d = (unsigned)(__ballot(dup) >> gb) & lanes;
        if (e < b1 && !dup) gc[out + (e - b0) + (at - a0) - both - __popc(d & ((1u << l) - 1u))] = x;
        both += __popc(d);
    }
}
// Whether four lanes per row are enough: entries few on the whole and in every
// row (asked of large matrices only: it costs a launch and a wait).
#define UNION_LOW_ROWS (1 << 18)
#define UNION_LOW_MEAN 4  // entries of A per row
#define UNION_LOW_MAX 64  // of a row of A and of A^T together
__global__ void __launch_bounds__(256)
k_both_lengths(int m, const int *__restrict__ ap, const int *__restrict__ tp, int *__restrict__ len) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < (unsigned)m) len[i] = ap[i + 1] - ap[i] + (tp[i + 1] - tp[i]);
}
static int union_is_low(tsg_ctx *ctx, const tsg_dcsr *a, const tsg_dcsr *at, int *len, bool *low) {
    *low = false;
    if (a->m < UNION_LOW_ROWS || a->nnz > UNION_LOW_MEAN * (long long)a->m) return TSG_OK;
    hipLaunchKernelGGL(k_both_lengths, dim3(tsg_div_up(a->m, 256)), dim3(256), 0, ctx->stream, a->m, a->rowptr, at->rowptr, len);
    TSG_LAUNCH_CHECK();
    int most = 0;
    TSG_TRY(max_of(ctx, len, a->m, &most));
    *low = most <= UNION_LOW_MAX;
    return TSG_OK;
}

// pattern(A + A^T), sorted rows, self loops kept
extern "C" int tsg_dcsr_symmetrize(tsg_ctx *ctx, const tsg_dcsr *a, tsg_dcsr *g) {
    memset(g, 0, sizeof(*g));
    if (a->m != a->n) { tsg_set_error("symmetrize needs a square matrix"); return TSG_ERR_ARG; }
    tsg_dcsr at;
    TSG_TRY(tsg_dcsr_transpose(ctx, a, &at));
    g->m = g->n = a->m;
    TSG_TRY(tsg_alloc_t(ctx, &g->rowptr, (size_t)a->m + 1));
    bool low;
    TSG_TRY(union_is_low(ctx, a, &at, g->rowptr, &low));
    const dim3 gr = tsg_grid(tsg_div_up(a->m, low ? 64 : 16), 256);
    if (a->m > 0) {
        hipLaunchKernelGGL((low ? k_union_rows<false, 4> : k_union_rows<false, 16>), gr, dim3(256), 0, ctx->stream, a->m, a->rowptr, a->colidx,
                           at.rowptr, at.colidx, g->rowptr, (int *)nullptr);
        TSG_LAUNCH_CHECK();
    }
    long long nnz = 0;
    TSG_TRY(tsg_scan_i32(ctx, g->rowptr, g->rowptr, a->m, &nnz));
    g->nnz = (int)nnz;
    TSG_TRY(tsg_alloc_t(ctx, &g->colidx, (size_t)nnz + 1));
    TSG_TRY(tsg_alloc_t(ctx, &g->val, (size_t)nnz + 1));
    if (a->m > 0 && nnz > 0) {
        hipLaunchKernelGGL((low ? k_union_rows<true, 4> : k_union_rows<true, 16>), gr, dim3(256), 0, ctx->stream, a->m, a->rowptr, a->colidx,
                           at.rowptr, at.colidx, g->rowptr, g->colidx);
        hipLaunchKernelGGL(k_fill_f64, dim3(tsg_div_up(nnz, 256)), dim3(256), 0, ctx->stream, g->val, nnz, 1.0);
        TSG_LAUNCH_CHECK();
    }
    tsg_dcsr_free(ctx, &at);
    return TSG_OK;
}

// ------------------------------------------------------------------ RCM
// degree as SciPy's _node_degrees: row length + 1 when the diagonal is stored
__global__ void k_rcm_deg(const int *__restrict__ gp, const int *__restrict__ gc, int n, int *__restrict__ deg) {
    int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= n) return;
    const int e1 = gp[v + 1];
    const int e = lower_bound_r(gc, gp[v], e1, v);
    deg[v] = e1 - gp[v] + (e < e1 && gc[e] == v);
}
__global__ void k_scatter_rank(const int *__restrict__ order, int n, int *__restrict__ rank) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r < n) rank[order[r]] = r;
}
// Connected components as a forest over the ranks whose parents only ever get
// smaller, so a component's root ends as its lowest rank whatever order the
// edges are taken in.  CC_ROUNDS rounds hook every vertex, then every tree, to
// the lowest rank next to it (a minimum, no retries) and flatten the forest;
// a last pass joins what is left, root to root by compare-and-swap, and is
// what the result rests on.  No read-back in between.  Label propagation with
// pointer jumping took 26 rounds with a read-back each on a shuffled 27-point
// mesh (27d 61x64x59; 1.5 ms of kernels), the last pass alone 2.9 ms (every
// tree's root swapped at once), after 3 / 4 / 5 rounds 0.97 / 0.48 / 0.33 ms.
#define CC_ROUNDS 5
// Parents are read past the caches of the other XCDs; an older parent is
// still an ancestor, and a failed swap returns the current one, so every
// step moves down.
__device__ __forceinline__ int cc_load(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int cc_root(const int *parent, int x) {
    int p = cc_load(&parent[x]);
    while (p != x) {  // p < x
        const int g = cc_load(&parent[p]);
        x = p;
        p = g;
    }
    return x;
}
// Lanes per vertex of the kernels that walk adjacency lists: VERT_LANES, and a
// wave where children are put in order; VERT_LANES_LOW and VERT_LANES where every
// list is short and most are shorter than a line (RCM of 2,000,000 pairs 7.3 -> 3.1
// ms with the scan by runs below, of ER 1,000,000, two a row, 4.0 -> 2.5).
#define VERT_LANES 16
#define VERT_LANES_LOW 4
#define VERT_LOW_MAX 64   // longest list
#define VERT_LOW_MEAN 8
// FIRST: parent of each vertex = the lowest rank among itself and its
// neighbours.  Else: the parent of its tree's root, label[v], lowered to the
// lowest label next to it.
template <bool FIRST, int VL>
__global__ void __launch_bounds__(256)
k_cc_hook(const int *__restrict__ gp, const int *__restrict__ gc, int n, const int *__restrict__ id, int *parent) {
    const unsigned v = tsg_block() * (256 / VL) + threadIdx.x / VL, l = threadIdx.x % VL;
    if (v >= (unsigned)n) return;
    const int iv = id[v], e1 = gp[v + 1];
    int mn = iv;
    for (int e = gp[v] + l; e < e1; e += VL) mn = min(mn, id[gc[e]]);
#pragma unroll
    for (int o = VL / 2; o > 0; o >>= 1) mn = min(mn, __shfl_xor(mn, o, VL));
    if (l == 0) {
        if (FIRST) parent[iv] = mn;
        else if (mn < iv && mn < cc_load(&parent[iv])) atomicMin(&parent[iv], mn);  // few trees: one address for many
    }
}
// label[v] = root of v's tree, and v's parent set to it.
__global__ void __launch_bounds__(256)
k_cc_label(const int *__restrict__ rank, int n, int *parent, int *__restrict__ label) {
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= n) return;
    const int r = rank[v], t = cc_root(parent, r);
    label[v] = t;
    if (t != r) __hip_atomic_store(&parent[r], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int VL>
__global__ void __launch_bounds__(256)
k_cc_link(const int *__restrict__ gp, const int *__restrict__ gc, int n, const int *__restrict__ label, int *parent) {
    const unsigned v = tsg_block() * (256 / VL) + threadIdx.x / VL, l = threadIdx.x % VL;
    if (v >= (unsigned)n) return;
    const int lv = label[v], e1 = gp[v + 1];
    for (int e = gp[v] + l; e < e1; e += VL) {
        const int lu = label[gc[e]];
        if (lu >= lv) continue;  // one tree, or the edge's other end takes it (the pattern is symmetric)
        int a = cc_root(parent, lv), b = cc_root(parent, lu);
        while (a != b) {
            if (a < b) { const int t = a; a = b; b = t; }
            const int old = atomicCAS(&parent[a], a, b);
            if (old == a) break;
            a = cc_root(parent, old);
        }
    }
}
// seeds (component minima) in rank order: flag, scan, compact
__global__ void k_seed_flag(const int *__restrict__ order, const int *__restrict__ label, int n, int *__restrict__ flag) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r < n) flag[r] = label[order[r]] == r;
}
__global__ void k_seed_compact(const int *__restrict__ order, const int *__restrict__ label, const int *__restrict__ pos,
                               int n, int *__restrict__ front, int *__restrict__ visited) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r < n && label[order[r]] == r) {
        front[pos[r]] = order[r];
        visited[order[r]] = 1;
    }
}
// One BFS level: every unvisited neighbour is claimed by its first parent in
// level order (its position q), the claimed ones are counted per parent, and
// put in (degree, id) order behind one another.  VL lanes per parent
// for the first two, EL for the last, which sorts a parent's children by
// counting the smaller keys; a level with more than RCM_KIDS children of one
// parent (word[0] then) goes through the radix sort instead.  Against sorting
// every level (62 of a 27-point 61x64x59 mesh, some 40 launches each, 18 ms for
// the call): 4 launches, 1.9 ms.
//   A block counts the parents of one run of positions and leaves each its
// children's place within the run; the runs' totals (at most RCM_BLOCKS) are all
// that is left to scan, whatever the level's size (scanning every count in
// one block took 1.3 ms of a level of 2,000,000).
#define RCM_KIDS 64
#define RCM_AHEAD 8  // levels enqueued behind one another
#define RCM_BLOCKS 1024
// Positions per block of a level of nf: whole steps of `step` parents.
__device__ __forceinline__ int rcm_run(int nf, int blocks, int step) {
    const int per = (int)(((unsigned)nf + (unsigned)blocks - 1u) / (unsigned)blocks);
    return (per + step - 1) / step * step;
}
// Where parent q's children go in the level's (q < nf), from k_count_children's
// places and k_level_scan's totals.
__device__ __forceinline__ int rcm_place(const int *__restrict__ cnt, const int *__restrict__ first, int run, int q) {
    return first[q / run] + cnt[q];
}
template <int VL>
__global__ void __launch_bounds__(256)
k_claim(const int *__restrict__ gp, const int *__restrict__ gc, const int *__restrict__ seq, int2 *__restrict__ level,
        int2 given, const int *__restrict__ visited, int *__restrict__ claim, int *__restrict__ word) {
    const int2 lv = given.y > 0 ? given : *level;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        word[0] = 0;
        if (given.y > 0) *level = given;
    }
    const int l = threadIdx.x % VL;
    for (int q = (int)(((long long)blockIdx.x * 256 + threadIdx.x) / VL); q < lv.y; q += (int)(gridDim.x * (256 / VL))) {
        const int p = seq[lv.x + q], e1 = gp[p + 1];
        for (int e = gp[p] + l; e < e1; e += VL) {
            const int u = gc[e];
            if (!visited[u]) atomicMin(&claim[u], q);
        }
    }
}
template <int VL>
__global__ void __launch_bounds__(256)
k_count_children(const int *__restrict__ gp, const int *__restrict__ gc, const int *__restrict__ seq,
                 const int2 *__restrict__ level, const int *__restrict__ visited, const int *__restrict__ claim,
                 int *__restrict__ cnt, int *__restrict__ total, int *__restrict__ word) {
    __shared__ int s_w[2][4];
    const int2 lv = *level;
    if (lv.y == 0) return;  // (an empty level leaves the places of the one before)
    constexpr int STEP = 256 / VL;
    const int l = threadIdx.x % VL, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int run = rcm_run(lv.y, gridDim.x, STEP);
    const long long q0 = (long long)blockIdx.x * run, q1 = min((long long)lv.y, q0 + run);
    int before = 0, k = 0;
    for (long long b = q0; b < q1; b += STEP, k ^= 1) {  // block-uniform
        const int q = (int)b + threadIdx.x / VL;
        int c = 0;
        if (q < q1) {
            const int p = seq[lv.x + q], e1 = gp[p + 1];
            for (int e = gp[p] + l; e < e1; e += VL) {
                const int u = gc[e];
                c += !visited[u] && claim[u] == q;
            }
        }
#pragma unroll
        for (int o = VL / 2; o > 0; o >>= 1) c += __shfl_xor(c, o, VL);
        const int mx = tsg_wave_max(c);
        if (lane == 0 && mx > RCM_KIDS) atomicMax(&word[0], mx);
        const int mine = l == 0 ? c : 0, incl = tsg_wave_incl_scan_dpp(mine);
        if (lane == 63) s_w[k][wave] = incl;
        __syncthreads();
        int at = before + incl - mine;
        for (int w = 0; w < 4; w++) {
            if (w < wave) at += s_w[k][w];
            before += s_w[k][w];
        }
        if (q < q1 && l == 0) cnt[q] = at;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = before;
}

// One block: the runs' totals to their first places, the next level
// behind this one (empty when a parent has too many children for
// k_emit_children), {children, most of one parent beyond RCM_KIDS} to the host.
__global__ void __launch_bounds__(RCM_BLOCKS)
k_level_scan(int *total, int blocks, int2 *level, const int *__restrict__ word, int *__restrict__ host) {
    __shared__ int s_w[RCM_BLOCKS / 64];
    const int2 lv = level[0];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (lv.y == 0) {  // block-uniform
        if (tid == 0) {
            level[1] = make_int2(0, 0);
            host[0] = host[1] = 0;
        }
        return;
    }
    const int c = tid < blocks ? total[tid] : 0, incl = tsg_wave_incl_scan_dpp(c);
    if (lane == 63) s_w[wave] = incl;
    __syncthreads();
    int at = incl - c;
    for (int w = 0; w < wave; w++) at += s_w[w];
    if (tid < blocks) total[tid] = at;
    if (tid == RCM_BLOCKS - 1) {
        const int all = at + c, most = word[0];
        level[1] = most > RCM_KIDS ? make_int2(0, 0) : make_int2(lv.x + lv.y, all);
        host[0] = all;
        host[1] = most;
    }
}
// Children of parent q, EL lanes', into their places, marked visited (only q's
// own claims are, so the other parents' tests do not change).
template <int EL>
__global__ void __launch_bounds__(256)
k_emit_children(const int *__restrict__ gp, const int *__restrict__ gc, const int2 *__restrict__ level, const int *__restrict__ word,
                int *__restrict__ visited, const int *__restrict__ claim, const int *__restrict__ deg,
                const int *__restrict__ cnt, const int *__restrict__ first, int blocks, int step, int *__restrict__ seq) {
    __shared__ unsigned long long s_key[256 / EL][RCM_KIDS];
    const int g = threadIdx.x / EL, l = threadIdx.x % EL, gb = (threadIdx.x & 63) / EL * EL;
    const unsigned long long mask = EL == 64 ? ~0ull : (1ull << (EL & 63)) - 1ull;
    const int2 lv = *level;
    if (lv.y == 0 || *word > RCM_KIDS) return;
    const int run = rcm_run(lv.y, blocks, step);
    int *out = seq + lv.x + lv.y;
    for (int q = blockIdx.x * (256 / EL) + g; q < lv.y; q += gridDim.x * (256 / EL)) {
        const int p = seq[lv.x + q], e0 = gp[p], e1 = gp[p + 1];
        int n = 0;  // at most RCM_KIDS
        for (int eb = e0; eb < e1; eb += EL) {
            const int e = eb + l;
            int u = 0;
            bool mine = false;
            if (e < e1) {
                u = gc[e];
                mine = !visited[u] && claim[u] == q;
            }
            const unsigned long long b = (__ballot(mine) >> gb) & mask;
            if (mine) s_key[g][n + __popcll(b & ((1ull << l) - 1ull))] = ((unsigned long long)(unsigned)deg[u] << 32) | (unsigned)u;
            n += __popcll(b);
        }
        tsg_wave_sync();
        const int at = n > 0 ? rcm_place(cnt, first, run, q) : 0;
        for (int i = l; i < n; i += EL) {
            const unsigned long long key = s_key[g][i];
            int r = 0;
            for (int j = 0; j < n; j++) r += s_key[g][j] < key;  // ids differ, so keys do
            const int u = (int)(key & 0xffffffffu);
            out[at + r] = u;
            visited[u] = 1;
        }
        tsg_wave_sync();  // the next parent rewrites the keys
    }
}
// The children of a level as sort keys (degree, id) with their parents.
__global__ void __launch_bounds__(256)
k_list_children(const int *__restrict__ gp, const int *__restrict__ gc, const int *__restrict__ front, int nf,
                const int *__restrict__ visited, const int *__restrict__ claim, const int *__restrict__ deg,
                const int *__restrict__ cnt, const int *__restrict__ first, int blocks, int step,
                unsigned long long *__restrict__ key, int *__restrict__ par) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned q = tsg_block() * 4 + wave;
    if (q >= (unsigned)nf) return;
    const int p = front[q], e1 = gp[p + 1];
    int k = rcm_place(cnt, first, rcm_run(nf, blocks, step), (int)q);
    for (int e0 = gp[p]; e0 < e1; e0 += 64) {
        const int e = e0 + lane;
        int u = 0;
        bool mine = false;
        if (e < e1) {
            u = gc[e];
            mine = !visited[u] && claim[u] == (int)q;
        }
        const unsigned long long b = __ballot(mine);
        if (mine) {
            const int at = k + __popcll(b & ((1ull << lane) - 1ull));
            key[at] = ((unsigned long long)(unsigned)deg[u] << 32) | (unsigned)u;
            par[at] = (int)q;
        }
        k += __popcll(b);
    }
}
__global__ void k_mark_children(const unsigned long long *__restrict__ key, int nc, int *__restrict__ visited) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nc) visited[(int)(key[i] & 0xffffffffu)] = 1;
}
__global__ void k_gather_children(const unsigned long long *__restrict__ key, const int *__restrict__ idx, int nc,
                                  int *__restrict__ out) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < nc) out[i] = (int)(key[idx[i]] & 0xffffffffu);
}
__global__ void k_comp_key(const int *__restrict__ seq, const int *__restrict__ label, int n, unsigned *__restrict__ k) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) k[i] = (unsigned)label[seq[i]];
}
__global__ void k_reverse_gather(const int *__restrict__ seq, const int *__restrict__ idx, int n, int *__restrict__ out) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = seq[idx[n - 1 - i]];
}
__global__ void k_fill_i32(int *v, long long n, int x) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) v[i] = x;
}

extern "C" int tsg_order_rcm(tsg_ctx *ctx, const tsg_dcsr *a, int *d_old_id, int *levels_out) {
    if (a->m != a->n) { tsg_set_error("RCM needs a square matrix"); return TSG_ERR_ARG; }
    const int n = a->m;
    if (n == 0) return TSG_OK;
    tsg_dcsr g;
    TSG_TRY(tsg_dcsr_symmetrize(ctx, a, &g));
    int *deg, *order, *rank, *label, *visited, *claim, *seq, *flag, *pos, *word, *first;
    TSG_TRY(tsg_alloc_t(ctx, &word, RCM_AHEAD));
    TSG_TRY(tsg_alloc_t(ctx, &first, RCM_BLOCKS));
    TSG_TRY(tsg_alloc_t(ctx, &deg, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &order, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &rank, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &label, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &visited, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &claim, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &seq, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &flag, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &pos, (size_t)n + 1));
    hipStream_t s = ctx->stream;
    const unsigned gn = tsg_div_up(n, 256);
    hipLaunchKernelGGL(k_rcm_deg, dim3(gn), dim3(256), 0, s, g.rowptr, g.colidx, n, deg);
    TSG_LAUNCH_CHECK();
    int longest = 0;
    TSG_TRY(sort_ids_by_degree(ctx, deg, n, 0, order, &longest));  // ascending (degree, id)
    const bool low = longest <= VERT_LOW_MAX && g.nnz <= VERT_LOW_MEAN * (long long)n;
    const int vl = low ? VERT_LANES_LOW : VERT_LANES, el = low ? VERT_LANES : 64, step = 256 / vl;
    // connected components: label = lowest rank in the component (parents in
    // claim, which is set up for the traversal below)
    const dim3 gv = tsg_grid(tsg_div_up(n, 256 / vl), 256);
    hipLaunchKernelGGL(k_scatter_rank, dim3(gn), dim3(256), 0, s, order, n, rank);
    for (int round = 0; round < CC_ROUNDS; round++) {
        auto hook = low ? (round == 0 ? k_cc_hook<true, VERT_LANES_LOW> : k_cc_hook<false, VERT_LANES_LOW>)
                        : (round == 0 ? k_cc_hook<true, VERT_LANES> : k_cc_hook<false, VERT_LANES>);
        hipLaunchKernelGGL(hook, gv, dim3(256), 0, s, g.rowptr, g.colidx, n, (const int *)(round == 0 ? rank : label), claim);
        hipLaunchKernelGGL(k_cc_label, dim3(gn), dim3(256), 0, s, (const int *)rank, n, claim, label);
    }
    hipLaunchKernelGGL(low ? k_cc_link<VERT_LANES_LOW> : k_cc_link<VERT_LANES>, gv, dim3(256), 0, s, g.rowptr, g.colidx, n, (const int *)label, claim);
    hipLaunchKernelGGL(k_cc_label, dim3(gn), dim3(256), 0, s, (const int *)rank, n, claim, label);
    TSG_LAUNCH_CHECK();
    // level 0: all component seeds, in rank order
    TSG_HIP(hipMemsetAsync(visited, 0, (size_t)n * 4, s));
    hipLaunchKernelGGL(k_fill_i32, dim3(gn), dim3(256), 0, s, claim, (long long)n, 0x7fffffff);
    hipLaunchKernelGGL(k_seed_flag, dim3(gn), dim3(256), 0, s, order, label, n, flag);
    TSG_LAUNCH_CHECK();
    long long nseed = 0;
    TSG_TRY(tsg_scan_i32(ctx, flag, pos, n, &nseed));
    hipLaunchKernelGGL(k_seed_compact, dim3(gn), dim3(256), 0, s, order, label, pos, n, seq, visited);
    TSG_LAUNCH_CHECK();
    long long done = nseed, fstart = 0, nf = nseed;
    int levels = 1;
    unsigned long long *key = nullptr;
    int *par = nullptr, *cnt = nullptr, *idx = nullptr;
    unsigned *k2 = nullptr;
    TSG_TRY(tsg_alloc_t(ctx, &key, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &par, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &cnt, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &idx, (size_t)n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &k2, (size_t)n + 1));
    const int nbits = bits_of(n);
    // Levels are enqueued up to RCM_AHEAD at a time, as many as the growth of the
    // last ones suggests (an empty one costs four launches): each finds its place
    // and size where the one before left them, and the host waits once for all.
    // Against a wait per level: RCM + permute of 27d 61x64x59, 64 levels, 3.65 ->
    // 3.41 ms, banded 8000, 365 levels, 10.0 -> 7.3 ms.  Always eight at a time lost 50
    // to 70 us on graphs of 5 to 11 levels.
    int2 *lvl = nullptr;
    TSG_TRY(tsg_alloc_t(ctx, &lvl, RCM_AHEAD + 1));
    int *host = (int *)ctx->pinned;
    static_assert(2 * RCM_AHEAD <= 128, "the pinned words hold every level's");
    double growth = 1.0;  // of the last level against the one before
    for (int ahead = 2; nf > 0 && done < n;) {
        const unsigned gf = std::min<unsigned>(RCM_BLOCKS, std::max(64u, tsg_div_up(2 * nf * vl, 256)));
        const unsigned gw = std::min(2048u, std::max(64u, tsg_div_up(2 * nf * el, 256)));
        for (int i = 0; i < ahead; i++) {
            hipLaunchKernelGGL(low ? k_claim<VERT_LANES_LOW> : k_claim<VERT_LANES>, dim3(gf), dim3(256), 0, s, g.rowptr, g.colidx,
                               (const int *)seq, lvl + i, i ? make_int2(0, 0) : make_int2((int)fstart, (int)nf), visited, claim,
                               word + i);
            hipLaunchKernelGGL(low ? k_count_children<VERT_LANES_LOW> : k_count_children<VERT_LANES>, dim3(gf), dim3(256), 0, s,
                               g.rowptr, g.colidx, (const int *)seq, (const int2 *)(lvl + i), visited, claim, cnt, first,
                               word + i);
            hipLaunchKernelGGL(k_level_scan, dim3(1), dim3(RCM_BLOCKS), 0, s, first, (int)gf, lvl + i, (const int *)(word + i),
                               host + 2 * i);
            hipLaunchKernelGGL(low ? k_emit_children<VERT_LANES> : k_emit_children<64>, dim3(gw), dim3(256), 0, s, g.rowptr,
                               g.colidx, (const int2 *)(lvl + i), (const int *)(word + i), visited, claim, deg,
                               (const int *)cnt, (const int *)first, (int)gf, step, seq);
            TSG_LAUNCH_CHECK();
        }
        TSG_HIP(hipStreamSynchronize(s));
        int kids[2 * RCM_AHEAD];
        memcpy(kids, host, sizeof(kids));
        bool big = false;
        long long nc = 0;
        for (int i = 0; i < ahead && nf > 0; i++) {
            nc = kids[2 * i];
            big = kids[2 * i + 1] > RCM_KIDS;
            if (big) break;
            growth = (double)nc / (double)nf;
            fstart += nf;
            nf = nc;
            done += nc;
            levels += nc > 0;
        }
        // as many as cover the rest if the levels go on like this
        double left = (double)(n - done), next = (double)nf * growth;
        for (ahead = 1; ahead < RCM_AHEAD && left > next; ahead++) {
            left -= next;
            next *= growth;
        }
        if (!big) continue;
        ahead = 2;
        // a parent with many children: the level's by sorting
        const int *front = seq + fstart;
        const dim3 gl = tsg_grid(tsg_div_up(nf, 4), 256);
        {
            hipLaunchKernelGGL(k_list_children, gl, dim3(256), 0, s, g.rowptr, g.colidx, front, (int)nf, visited,
                               claim, deg, (const int *)cnt, (const int *)first, (int)gf, step, key, par);
            TSG_LAUNCH_CHECK();
            const unsigned gc2 = tsg_div_up(nc, 256);
            hipLaunchKernelGGL(k_mark_children, dim3(gc2), dim3(256), 0, s, key, (int)nc, visited);
            // order children by (parent position, degree, id): sort by (degree,
            // id), then stably by parent position
            hipLaunchKernelGGL(k_iota2, dim3(gc2), dim3(256), 0, s, idx, nc);
            TSG_LAUNCH_CHECK();
            TSG_TRY(tsg_sort_pairs_u64(ctx, key, idx, nc, 32 + bits_of((long long)n + 1)));
            // after the sort, idx[i] is the emit slot of the i-th smallest key:
            // parent of the i-th smallest key is par[idx[i]]
            hipLaunchKernelGGL(k_gather_i32_r, dim3(gc2), dim3(256), 0, s, par, idx, (int)nc, (int *)k2);
            hipLaunchKernelGGL(k_iota2, dim3(gc2), dim3(256), 0, s, idx, nc);
            TSG_LAUNCH_CHECK();
            TSG_TRY(tsg_sort_pairs_u32(ctx, k2, idx, nc, bits_of(nf)));
            hipLaunchKernelGGL(k_gather_children, dim3(gc2), dim3(256), 0, s, key, idx, (int)nc, seq + fstart + nf);
            TSG_LAUNCH_CHECK();
        }
        fstart += nf;
        nf = nc;
        done += nc;
        levels++;
    }
    if (done != n) { tsg_set_error("RCM: traversal covered %lld of %d vertices", done, n); return TSG_ERR_STATE; }
    // group the level-ordered sequence by component (stable), then reverse
    unsigned *ck;
    TSG_TRY(tsg_alloc_t(ctx, &ck, (size_t)n + 1));
    hipLaunchKernelGGL(k_comp_key, dim3(gn), dim3(256), 0, s, seq, label, n, ck);
    hipLaunchKernelGGL(k_iota2, dim3(gn), dim3(256), 0, s, idx, (long long)n);
    TSG_LAUNCH_CHECK();
    TSG_TRY(tsg_sort_pairs_u32(ctx, ck, idx, n, nbits));
    hipLaunchKernelGGL(k_reverse_gather, dim3(gn), dim3(256), 0, s, seq, idx, n, d_old_id);
    TSG_LAUNCH_CHECK();
    if (levels_out) *levels_out = levels;
    void *ps[] = {deg, order, rank, label, visited, claim, seq, flag, pos, word, first, key, par, cnt, idx, k2, ck, lvl};
    for (void *p : ps) tsg_free(ctx, p);
    tsg_dcsr_free(ctx, &g);
    return TSG_OK;
}

// ------------------------------------------------------------------ P A Q^T
#define PERM_WAVE 64
#define PERM_BLOCK 4096
// Row lengths of the result; word[0] (zeroed beforehand) = the longest over
// PERM_WAVE, if any, word[1] = the number of such rows, listed in rows (in no
// order).  (An atomic per wave on one address is 43 us of its own.)
__global__ void __launch_bounds__(256)
k_perm_counts(const int *__restrict__ rowptr, const int *__restrict__ row_old, int m, int *__restrict__ cnt,
              int *__restrict__ word, int *__restrict__ rows) {
    const int lane = threadIdx.x & 63;
    int mx = 0;
    for (unsigned r0 = blockIdx.x * 256; r0 < (unsigned)m; r0 += gridDim.x * 256) {  // block-uniform
        const unsigned r = r0 + threadIdx.x;
        int c = 0;
        if (r < (unsigned)m) {
            c = rowptr[row_old[r] + 1] - rowptr[row_old[r]];
            cnt[r] = c;
        }
        mx = max(mx, c);
        const unsigned long long b = __ballot(c > PERM_WAVE);
        if (!b) continue;
        int at = 0;
        if (lane == 0) at = atomicAdd(&word[1], __popcll(b));
        at = __builtin_amdgcn_readfirstlane(at);
        if (c > PERM_WAVE) rows[at + __popcll(b & ((1ull << lane) - 1ull))] = (int)r;
    }
    mx = tsg_wave_max(mx);
    if (lane == 0 && mx > PERM_WAVE) atomicMax(&word[0], mx);
}
// Rows of at most PERM_WAVE entries: each entry's place by counting the
// smaller columns, one wave per row, or 16 lanes where rows have at most 16
// entries on average (4,000,000 rows of one entry 2.43 -> 1.74 ms for the call,
// 5-point 1500x1000 1.02 -> 0.77).  Longer ones, up to PERM_BLOCK: one block per
// listed row (a block for every row: 3.51 / 1.74 ms with one row of 100), bitonic
// sort in LDS.  A matrix with a longer row has all its entries sorted by
// (row, column) with the radix sort (two words an entry, five passes and
// more): 27-point 61x64x59 (5.9M entries) some 0.9 ms of kernels
// -> 0.11.
__global__ void __launch_bounds__(256)
k_perm_rows(const int *__restrict__ rowptr, const int *__restrict__ col, const double *__restrict__ val,
            const int *__restrict__ row_old, const int *__restrict__ col_new, int m, const int *__restrict__ optr,
            int *__restrict__ ocol, double *__restrict__ oval) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned r = tsg_block() * 4 + wave;
    if (r >= (unsigned)m) return;
    const int e0 = rowptr[row_old[r]], o0 = optr[r], n = optr[r + 1] - o0;
    if (n == 0 || n > PERM_WAVE) return;  // wave-uniform
    int c = 0x7fffffff;
    double v = 0.0;
    if (lane < n) {
        c = col_new[col[e0 + lane]];
        v = val[e0 + lane];
    }
    int at = 0;
    for (int j = 0; j < n; j++) at += __builtin_amdgcn_readlane(c, j) < c;  // columns differ inside a row
    if (lane < n) {
        ocol[o0 + at] = c;
        oval[o0 + at] = v;
    }
}
__global__ void __launch_bounds__(256)
k_perm_rows16(const int *__restrict__ rowptr, const int *__restrict__ col, const double *__restrict__ val,
              const int *__restrict__ row_old, const int *__restrict__ col_new, int m, const int *__restrict__ optr,
              int *__restrict__ ocol, double *__restrict__ oval) {
    constexpr int Q = PERM_WAVE / 16;  // entries of a lane
    const unsigned r = tsg_block() * 16 + (threadIdx.x >> 4);
    const int l = threadIdx.x & 15;
    int e0 = 0, o0 = 0, n = 0;
    if (r < (unsigned)m) {
        e0 = rowptr[row_old[r]];
        o0 = optr[r];
        n = optr[r + 1] - o0;
        if (n > PERM_WAVE) n = 0;
    }
    int c[Q], at[Q];
    double v[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        c[q] = 0x7fffffff;
        at[q] = 0;
        v[q] = 0.0;
        if (l + 16 * q < n) {
            c[q] = col_new[col[e0 + l + 16 * q]];
            v[q] = val[e0 + l + 16 * q];
        }
    }
#pragma unroll
    for (int s = 0; s < Q; s++) {
        if (!__any(n > 16 * s)) break;  // wave-uniform; every lane is active in the broadcasts
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int x = tsg_row16_bcast(c[s], j);
#pragma unroll
            for (int q = 0; q < Q; q++) at[q] += x < c[q];
        }
    }
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (l + 16 * q < n) {
            ocol[o0 + at[q]] = c[q];
            oval[o0 + at[q]] = v[q];
        }
}
__global__ void __launch_bounds__(256)
k_perm_rows_block(const int *__restrict__ rowptr, const int *__restrict__ col, const double *__restrict__ val,
                  const int *__restrict__ row_old, const int *__restrict__ col_new, const int *__restrict__ rows, int nrows,
                  const int *__restrict__ optr, int *__restrict__ ocol, double *__restrict__ oval) {
    __shared__ unsigned long long s_key[PERM_BLOCK];
    const int tid = threadIdx.x;
    for (int w = blockIdx.x; w < nrows; w += gridDim.x) {
        const int r = rows[w];
        const int e0 = rowptr[row_old[r]], o0 = optr[r], n = optr[r + 1] - o0;
        int p2 = 2 * PERM_WAVE;
        while (p2 < n) p2 <<= 1;
        for (int i = tid; i < p2; i += 256)
            s_key[i] = i < n ? ((unsigned long long)(unsigned)col_new[col[e0 + i]] << 32) | (unsigned)i : ~0ull;
        __syncthreads();
        for (int k = 2; k <= p2; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int i = tid; i < p2; i += 256) {
                    const int x = i ^ j;
                    if (x > i) {
                        const unsigned long long a = s_key[i], b = s_key[x];
                        if ((a > b) == ((i & k) == 0)) {
                            s_key[i] = b;
                            s_key[x] = a;
                        }
                    }
                }
                __syncthreads();
            }
        for (int i = tid; i < n; i += 256) {
            const unsigned long long key = s_key[i];
            ocol[o0 + i] = (int)(key >> 32);
            oval[o0 + i] = val[e0 + (int)(key & 0xffffffffu)];
        }
        __syncthreads();  // the next row rewrites the keys
    }
}
__global__ void k_perm_emit(const int *__restrict__ rowptr, const int *__restrict__ col, const int *__restrict__ row_old,
                            const int *__restrict__ col_new, int m, int n, const int *__restrict__ optr,
                            unsigned long long *__restrict__ key, int *__restrict__ src) {
    const unsigned r = tsg_block() * 16 + (threadIdx.x >> 4);  // 16 lanes per row
    const int l = threadIdx.x & 15;
    if (r >= (unsigned)m) return;
    const int e0 = rowptr[row_old[r]], w0 = optr[r], len = optr[r + 1] - w0;
    for (int j = l; j < len; j += 16) {
        key[w0 + j] = (unsigned long long)r * (unsigned long long)n + (unsigned)col_new[col[e0 + j]];
        src[w0 + j] = e0 + j;
    }
}
__global__ void k_perm_gather(const unsigned long long *__restrict__ key, const int *__restrict__ src,
                              const double *__restrict__ val, int nnz, int n, int *__restrict__ ocol, double *__restrict__ oval) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nnz) return;
    ocol[i] = (int)(key[i] % (unsigned long long)n);
    oval[i] = val[src[i]];
}

// out row r = a row row_old[r], columns relabelled c -> col_new[c], rows sorted.
extern "C" int tsg_dcsr_permute(tsg_ctx *ctx, const tsg_dcsr *a, const int *d_row_old, const int *d_col_new,
                                tsg_dcsr *out) {
    memset(out, 0, sizeof(*out));
    TSG_TRY(tsg_validate_csr(ctx, a));
    TSG_TRY(tsg_perm_validate(ctx, a->m, d_row_old));
    TSG_TRY(tsg_perm_validate(ctx, a->n, d_col_new));
    const int m = a->m, n = a->n, nnz = a->nnz;
    out->m = m;
    out->n = n;
    out->nnz = nnz;
    TSG_TRY(tsg_alloc_t(ctx, &out->rowptr, (size_t)m + 1));
    TSG_TRY(tsg_alloc_t(ctx, &out->colidx, (size_t)nnz + 1));
    TSG_TRY(tsg_alloc_t(ctx, &out->val, (size_t)nnz + 1));
    int *word, *rows;  // {longest row, rows of more than PERM_WAVE entries}, those rows
    TSG_TRY(tsg_alloc_t(ctx, &word, 4));
    TSG_TRY(tsg_alloc_t(ctx, &rows, (size_t)nnz / (PERM_WAVE + 1) + 1));
    TSG_HIP(hipMemsetAsync(word, 0, 8, ctx->stream));
    if (m > 0) {
        hipLaunchKernelGGL(k_perm_counts, dim3(std::min<unsigned>(1024, tsg_div_up(m, 256))), dim3(256), 0, ctx->stream,
                           a->rowptr, d_row_old, m, out->rowptr, word, rows);
        TSG_LAUNCH_CHECK();
    }
    long long tot = 0;
    const int sc = tsg_scan_i32(ctx, out->rowptr, out->rowptr, m, &tot, word, 2);
    const int longest = ((volatile int *)(ctx->pinned + 1))[0], nlong = ((volatile int *)(ctx->pinned + 1))[1];
    tsg_free(ctx, word);
    tsg_free(ctx, rows);  // (what frees and allocates later is behind these kernels on the stream)
    TSG_TRY(sc);
    if (tot != nnz) { tsg_set_error("permute: row permutation is not a bijection"); return TSG_ERR_ARG; }
    if (nnz > 0 && longest <= PERM_BLOCK) {
        if (nlong < m && nnz <= 16LL * m)
            hipLaunchKernelGGL(k_perm_rows16, tsg_grid(tsg_div_up(m, 16), 256), dim3(256), 0, ctx->stream, a->rowptr, a->colidx,
                               a->val, d_row_old, d_col_new, m, out->rowptr, out->colidx, out->val);
        else if (nlong < m)
            hipLaunchKernelGGL(k_perm_rows, tsg_grid(tsg_div_up(m, 4), 256), dim3(256), 0, ctx->stream, a->rowptr, a->colidx,
                               a->val, d_row_old, d_col_new, m, out->rowptr, out->colidx, out->val);
        if (nlong > 0)
            hipLaunchKernelGGL(k_perm_rows_block, dim3((unsigned)std::min(nlong, 1 << 16)), dim3(256), 0, ctx->stream,
                               a->rowptr, a->colidx, a->val, d_row_old, d_col_new, (const int *)rows, nlong, out->rowptr,
                               out->colidx, out->val);
        TSG_LAUNCH_CHECK();
    } else if (nnz > 0) {
        unsigned long long *key;
        int *src;
        TSG_TRY(tsg_alloc_t(ctx, &key, (size_t)nnz));
        TSG_TRY(tsg_alloc_t(ctx, &src, (size_t)nnz));
        hipLaunchKernelGGL(k_perm_emit, tsg_grid(tsg_div_up(m, 16), 256), dim3(256), 0, ctx->stream, a->rowptr, a->colidx, d_row_old, d_col_new,
                           m, n, out->rowptr, key, src);
        TSG_LAUNCH_CHECK();
        TSG_TRY(tsg_sort_pairs_u64(ctx, key, src, nnz, bits_of((long long)m * n)));
        hipLaunchKernelGGL(k_perm_gather, dim3(tsg_div_up(nnz, 256)), dim3(256), 0, ctx->stream, key, src, a->val, nnz, n,
                           out->colidx, out->val);
        TSG_LAUNCH_CHECK();
        tsg_free(ctx, key);
        tsg_free(ctx, src);
    }
    return TSG_OK;
}
