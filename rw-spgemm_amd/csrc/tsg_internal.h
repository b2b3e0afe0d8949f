// tsg_internal.h -- shared internals of the gfx950 TileSpGEMM library:
// context, caching device allocator, error plumbing and wave64 helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/tsg.h"

#define TSG_TILE 16

// ------------------------------------------------------------------ errors
void tsg_set_error(const char *fmt, ...);

#define TSG_HIP(call)                                                          \
    do {                                                                       \
        hipError_t e_ = (call);                                                \
        if (e_ != hipSuccess) {                                                \
            tsg_set_error("%s:%d %s -> %s", __FILE__, __LINE__, #call,         \
                          hipGetErrorString(e_));                              \
            return TSG_ERR_HIP;                                                \
        }                                                                      \
    } while (0)

#define TSG_TRY(expr)                                                          \
    do {                                                                       \
        int s_ = (expr);                                                       \
        if (s_ != TSG_OK) return s_;                                           \
    } while (0)

#define TSG_LAUNCH_CHECK()                                                     \
    do {                                                                       \
        hipError_t e_ = hipGetLastError();                                     \
        if (e_ != hipSuccess) {                                                \
            tsg_set_error("%s:%d kernel launch -> %s", __FILE__, __LINE__,     \
                          hipGetErrorString(e_));                              \
            return TSG_ERR_HIP;                                                \
        }                                                                      \
    } while (0)

// ------------------------------------------------------------------ arena
// One device allocation handed out in pieces (best fit; released pieces
// coalesce with free neighbours); shared by contexts on several threads.
// Memory returned to an arena stays mapped, so a workload that keeps
// allocating and releasing large blocks does not go back to the driver.
struct tsg_arena {
    int device = 0;
    char *base = nullptr;
    size_t size = 0;
    std::mutex mu;
    std::map<size_t, size_t> free_by_off;       // offset -> length
    std::multimap<size_t, size_t> free_by_len;  // length -> offset
    size_t bytes_free = 0;
};
int tsg_arena_create(int device, size_t bytes, tsg_arena **out);
void tsg_arena_destroy(tsg_arena *a);
void *tsg_arena_alloc(tsg_arena *a, size_t bytes);  // nullptr when no free piece fits
void tsg_arena_free(tsg_arena *a, void *p, size_t bytes);
inline bool tsg_arena_owns(const tsg_arena *a, const void *p) {
    return a && (const char *)p >= a->base && (const char *)p < a->base + a->size;
}

// ------------------------------------------------------------------ context
#define TSG_STAGE_WORKERS 4
struct tsg_ctx {
    int device;
    hipStream_t stream;
    // caching allocator: size -> blocks (stream-ordered reuse on `stream`)
    std::multimap<size_t, void *> free_blocks;
    std::map<void *, size_t> live;
    long long bytes_live = 0;
    long long bytes_cached = 0;
    // small pinned host buffer for scalar read-backs
    long long *pinned = nullptr;
    // persistent small device scratch (scan partials, counters)
    void *scratch = nullptr;
    size_t scratch_bytes = 0;
    // pinned slots of large copies to the host, two per worker
    char *stage = nullptr;
    hipEvent_t stage_ev[2 * TSG_STAGE_WORKERS] = {};
    // when set, blocks come from this arena (hipMalloc only if it is full)
    tsg_arena *arena = nullptr;
};
// Routes ctx's allocations through an arena; call before it allocates.
void tsg_ctx_set_arena(tsg_ctx *ctx, tsg_arena *a);

int tsg_alloc(tsg_ctx *ctx, void **p, size_t bytes);
void tsg_free(tsg_ctx *ctx, void *p);
template <typename T>
static inline int tsg_alloc_t(tsg_ctx *ctx, T **p, size_t count) {
    return tsg_alloc(ctx, (void **)p, count * sizeof(T));
}
int tsg_scratch(tsg_ctx *ctx, size_t bytes, void **p);
int tsg_read_scalar_i64(tsg_ctx *ctx, const void *dptr, int is64, long long *out);
// Device to fresh host memory, all parts, finished on return.
struct tsg_part {
    void *dst;
    const void *src;
    size_t bytes;
};
int tsg_download_parts(tsg_ctx *ctx, const tsg_part *parts, int n);
// Host memory for a result (free() it): huge pages asked for when it is large.
void *tsg_host_alloc(size_t bytes);
// Bytes the allocator reserved for a live block of ctx (0 if none).
size_t tsg_alloc_size(const tsg_ctx *ctx, const void *p);

// ------------------------------------------------------------------ scans
// Exclusive scan of n non-negative int32 counts into out[0..n] (out[n] =
// total).  `in` may alias `out`.  total (may be NULL) is read back to the
// host; TSG_ERR_OVERFLOW when the total exceeds INT32_MAX.  With total,
// nwords device ints are read back behind it (ctx->pinned + 1).
int tsg_scan_i32(tsg_ctx *ctx, const int *in, int *out, long long n, long long *total, const int *words = nullptr,
                 int nwords = 0);
// Enqueue-only form (no host read-back, no memset: graph-capturable).
// `partial` holds tsg_scan_partial_count(n) int64 values; the int64 total
// is left in partial[tsg_scan_partial_count(n) - 1].  With pub.host (pinned
// memory) the scan's last block also writes the total there and nwords
// device ints behind it: valid once the stream has been waited for.
struct tsg_scan_publish {
    long long *host = nullptr;
    const int *words = nullptr;
    int nwords = 0;
};
long long tsg_scan_partial_count(long long n);
int tsg_scan_i32_enqueue(hipStream_t stream, const int *in, int *out, long long n, long long *partial,
                         tsg_scan_publish pub = {});

// ------------------------------------------------------------------ spgemm
// Decisions of one SpGEMM that depend only on the operand patterns (sizes
// of C, which step-2 / step-3 kernels run, the LDS layout of the row-wise
// step 3).  A plan made by tsg_spgemm_planned lets tsg_spgemm_enqueue
// recompute the same product into the same C buffers with no host
// read-back, allocation or memset (so the sequence can be captured in a
// HIP graph).
struct tsg_spgemm_plan {
    long long numtileC, nnzC;
    int maxrow;     // C tiles of the longest tile-row
    int all;        // every tile-row through the tile-parallel kernels
    int s3_rows;    // some tile-row runs the row-wise step 3
    int s3_unfit;   // some tile-row runs the tile-parallel step 3
    int dense_min;  // dense accumulator threshold of the tile-parallel step 3
    int s3_elem;    // the tile-rows the row-wise kernel cannot hold go element-wise
    int elem_all;   // every tile-row goes element-wise
    int g3[6];      // row-wise step-3 LDS layout maxima
    int s1w;        // step-1 bitmap window, 32-bit words per wave
    int s2u;        // most C tiles of a step-2 tile-pair segment (LDS sizing)
    int s2map;      // bytes of the step-2 column -> slot map (0: binary search)
    int n2[4];      // step-2 segments per kernel (step2_kind)
    int s2w;        // widest tile-row span of the dense step 2's small blocks
    int lines;      // tile-rows may go by row lines
    int s3_lines;   // some tile-row does
    int ln[4];      // row lines: C nonzeros, C tiles, map bytes, threads of a block
    int s3span;     // widest tile-column span of a tile-row (hash key widths of step 3)
};
// symbolic = true runs steps 1-2 and the step-3 plan only (C's values and
// in-tile columns stay unallocated); stats (when given) then holds C's exact
// tile and nonzero counts and the numeric step's heavy-row scratch bytes.
// may_index = true lets it make row indices of its own, for this product, where
// the operands have none and it pays.
// On any error every temporary and every array of C allocated so far is
// freed (C is left zeroed).
int tsg_spgemm_planned(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, const tsg_tune *tune,
                       tsg_dtiles *C, tsg_stats *stats, tsg_spgemm_plan *plan_out, bool symbolic = false,
                       bool may_index = false);
// tsg_spgemm_tile_rows with the symbolic option above.
int tsg_spgemm_tile_rows_ex(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, int r0, int r1,
                            const tsg_tune *tune, tsg_dtiles *C, tsg_stats *stats, bool symbolic);
// Intermediate products of each A tile-row (device u64[A->tilem]).
int tsg_tile_row_products(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, unsigned long long *d_out);
// Device scratch bytes tsg_spgemm_enqueue needs for this C and B (B may be
// NULL: no room for B's tile-row bitmaps, counted for a product with B).
size_t tsg_spgemm_work_bytes(const tsg_dtiles *C, const tsg_dtiles *B, int s1w);
// Step-1 bitmap window (32-bit words per wave) for products with this B.
int tsg_s1_words(const tsg_dtiles *B, const tsg_tune &t);
int tsg_spgemm_enqueue(hipStream_t s, const tsg_dtiles *A, const tsg_dtiles *B, tsg_dtiles *C,
                       const tsg_spgemm_plan &P, void *work);

// ------------------------------------------------------------------ conversions
int tsg_tile2csr_view(tsg_ctx *ctx, const tsg_dtiles *t, int jbase, tsg_dcsr *out);
// Block-diagonal packing of tile matrices on 16-row/column boundaries.
int tsg_tiles_pack(tsg_ctx *ctx, const tsg_dtiles *const *parts, int count, tsg_dtiles *out);

// ------------------------------------------------------------------ sort
// Stable ascending sort of (key,value) pairs, 32-bit keys, using the
// library's own LSD radix sort.  Keys must be < (1u << key_bits).
int tsg_sort_pairs_u32(tsg_ctx *ctx, unsigned *keys, int *vals, long long n,
                       int key_bits);
int tsg_sort_pairs_u64(tsg_ctx *ctx, unsigned long long *keys, int *vals, long long n,
                       int key_bits);

// ------------------------------------------------------------------ device helpers
__device__ __forceinline__ void tsg_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int tsg_lane() { return __lane_id(); }

template <typename T>
__device__ __forceinline__ T tsg_wave_sum(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
template <typename T>
__device__ __forceinline__ T tsg_wave_min(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { T w = __shfl_xor(v, o, 64); v = w < v ? w : v; }
    return v;
}
template <typename T>
__device__ __forceinline__ T tsg_wave_max(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { T w = __shfl_xor(v, o, 64); v = w > v ? w : v; }
    return v;
}
// inclusive scan across the 64 lanes
template <typename T>
__device__ __forceinline__ T tsg_wave_incl_scan(T v) {
    const int lane = __lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        T w = __shfl_up(v, o, 64);
        if (lane >= o) v += w;
    }
    return v;
}
// The same for 32-bit values by DPP (six VALU moves, no LDS traffic); every
// lane of the wave must be active.  Row shifts inside the 16-lane rows, then
// row 0's last lane into row 1 and row 2's into row 3, then lane 31 into
// rows 2 and 3; lanes without a source take 0.
__device__ __forceinline__ int tsg_wave_incl_scan_dpp(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}
// inclusive scan inside each row of 16 lanes, likewise
__device__ __forceinline__ int tsg_row16_incl_scan_dpp(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    return v;
}
// inclusive running maximum of non-negative values, likewise
__device__ __forceinline__ int tsg_wave_incl_max_dpp(int v) {
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
    return v;
}
// inclusive scan inside groups of 16 lanes
template <typename T>
__device__ __forceinline__ T tsg_group16_incl_scan(T v) {
    const int r = __lane_id() & 15;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        T w = __shfl_up(v, o, 16);
        if (r >= o) v += w;
    }
    return v;
}
// Tile columns of a wave's bitmap window, ascending, into list[0..): words
// [0, nw) of bm, the first at tile column w0; returns their number.  64 words
// with many tiles (more than 4 a word) are written one pair of words per
// step, each bit a lane, so that a store instruction covers consecutive
// entries; with few, each lane writes the bits of its own word (all of them
// in a few lines anyway).  Step-1 fill against a per-lane loop over several
// words: ER 65521 438 -> 39 us (72% of the tile columns), 27p 128^3 217 -> 167
// us, R-MAT scale 16 180 -> 67 us.  Every lane of the wave must be active.
__device__ __forceinline__ int emit_window(const unsigned *bm, int nw, int w0, int lane, int *__restrict__ list) {
    int done = 0;
    for (int k0 = 0; k0 < nw; k0 += 64) {
        const unsigned x = k0 + lane < nw ? bm[k0 + lane] : 0u;
        const int c = __popc(x), incl = tsg_wave_incl_scan_dpp(c);
        const int tot = __builtin_amdgcn_readlane(incl, 63);
        const int pos = done + incl - c;
        if (tot > 256) {
            unsigned long long nz = __ballot(x != 0u);
            while (nz) {
                const int j0 = __ffsll((long long)nz) - 1;
                nz &= nz - 1;
                const int j1 = nz ? __ffsll((long long)nz) - 1 : j0;
                const bool both = nz != 0;
                nz &= nz - 1;  // 0 stays 0
                const int j = lane < 32 ? j0 : j1;
                const unsigned wd = lane < 32 ? (unsigned)__builtin_amdgcn_readlane((int)x, j0)
                                              : (unsigned)__builtin_amdgcn_readlane((int)x, j1);
                const int p = lane < 32 ? __builtin_amdgcn_readlane(pos, j0) : __builtin_amdgcn_readlane(pos, j1);
                const int b = lane & 31;
                if ((lane < 32 || both) && (wd >> b) & 1u)
                    list[p + __popc(wd & ((1u << b) - 1u))] = w0 + 32 * (k0 + j) + b;
            }
        } else {
            unsigned y = x;
            for (int q = pos; y; q++) {
                list[q] = w0 + 32 * (k0 + lane) + __ffs(y) - 1;
                y &= y - 1;
            }
        }
        done += tot;
    }
    return done;
}
// The 16 row lengths of a tile, one byte each, from its row offsets: next
// offset minus offset, byte by byte.  Offsets ascend, so no borrow crosses a
// byte; the last byte's minuend is the entry count (mod 256).
__device__ __forceinline__ uint4 tile_row_lens(uint4 p, int tnnz) {
    return make_uint4(((p.x >> 8) | (p.y << 24)) - p.x, ((p.y >> 8) | (p.z << 24)) - p.y,
                      ((p.z >> 8) | (p.w << 24)) - p.z, ((p.w >> 8) | ((unsigned)tnnz << 24)) - p.w);
}
// Bytes as 16-bit pairs: v[2q] = rows 4q and 4q+2, v[2q+1] = rows 4q+1, 4q+3.
__device__ __forceinline__ void tile_widen_lens(uint4 l, unsigned v[8]) {
    const unsigned w[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        v[2 * q] = w[q] & 0x00ff00ffu;
        v[2 * q + 1] = (w[q] >> 8) & 0x00ff00ffu;
    }
}

// v's entry for row r (0..15)
__device__ __forceinline__ int tile_row_of(const unsigned v[8], int r) {
    unsigned x = 0;
#pragma unroll
    for (int q = 0; q < 8; q++)
        if (2 * (r >> 2) + (r & 1) == q) x = v[q];
    return (int)((r & 2) ? x >> 16 : x & 0xffffu);
}
// Bytes of w that are at most j, as 0x80 bits (unsigned, per byte).
__device__ __forceinline__ unsigned bytes_le(unsigned w, unsigned j) {
    const unsigned H = 0x80808080u, x = j * 0x01010101u;
    const unsigned t = (x | H) - (w & ~H);  // per byte, no borrow out
    return ((x & ~w) | (~(x ^ w) & t)) & H;
}
// Value of lane q of this lane's group of 16 lanes (q a constant after
// unrolling): a DPP row broadcast, a VALU move with no LDS traffic, where
// __shfl would issue a ds_bpermute.  Every lane of the group must be active.
// (bound_ctrl set, though no lane lacks a source: without it the move is not
// folded into the instruction that uses it.)
#define TSG_RB_CASE(Q) case Q: return __builtin_amdgcn_update_dpp((T)0, v, 0x150 + Q, 0xF, 0xF, true);
template <typename T>
__device__ __forceinline__ T tsg_row16_bcast(T v, int q) {
    switch (q) {
        TSG_RB_CASE(0) TSG_RB_CASE(1) TSG_RB_CASE(2) TSG_RB_CASE(3)
        TSG_RB_CASE(4) TSG_RB_CASE(5) TSG_RB_CASE(6) TSG_RB_CASE(7)
        TSG_RB_CASE(8) TSG_RB_CASE(9) TSG_RB_CASE(10) TSG_RB_CASE(11)
        TSG_RB_CASE(12) TSG_RB_CASE(13) TSG_RB_CASE(14) default: break;
    }
    return __builtin_amdgcn_update_dpp((T)0, v, 0x150 + 15, 0xF, 0xF, true);
}
#undef TSG_RB_CASE
template <typename T>
__device__ __forceinline__ T tsg_group16_sum(T v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
    return v;
}

// Blocks are dispatched round-robin over the 8 XCDs of an MI355X; remap so
// that each XCD (and its L2) works on one contiguous range of block ids.
__device__ __forceinline__ unsigned tsg_xcd_block(unsigned bid, unsigned nblocks) {
    const unsigned nx = 8;
    const unsigned per = nblocks / nx;      // full rounds
    const unsigned rem = nblocks % nx;
    const unsigned xcd = bid % nx, k = bid / nx;
    // XCD x owns per (+1 if x < rem) consecutive logical ids
    const unsigned base = xcd * per + (xcd < rem ? xcd : rem);
    return (k < per + (xcd < rem ? 1u : 0u)) ? base + k : bid;
}

static inline unsigned tsg_div_up(long long a, long long b) { return (unsigned)((a + b - 1) / b); }
// Grid of `blocks` blocks of `threads`: a launch takes fewer than 2^32 threads
// along x, so more go in rows of 2^31 along y.  Blocks are numbered by
// tsg_block(); the last row may have some past the end.
static inline dim3 tsg_grid(long long blocks, int threads) {
    const long long row = (1LL << 31) / threads;
    return blocks <= row ? dim3((unsigned)blocks) : dim3((unsigned)row, (unsigned)((blocks + row - 1) / row));
}
__device__ __forceinline__ unsigned tsg_block() { return blockIdx.y * gridDim.x + blockIdx.x; }
int tsg_validate_csr(tsg_ctx *ctx, const tsg_dcsr *a);
// sorted = 0: row pointers and column range only (repeated or unsorted
// columns allowed, as mmio_allinone leaves them).
int tsg_validate_csr_mode(tsg_ctx *ctx, const tsg_dcsr *a, int sorted);
