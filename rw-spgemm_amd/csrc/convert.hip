// convert.hip -- CSR <-> 16x16 tile conversions, CSC tile index, stable CSR
// transpose and the intermediate-product count, all on the device.
//
// csr2tile follows the output contract of csr2tile_row_major
// (src/csr2tile.h:196-259): tiles sorted by tile column inside each
// tile-row, per-tile exclusive nnz offsets, per-row u8 offsets inside a
// tile, MSB-first u16 row masks, values row-major inside a tile with
// ascending columns.  The reference builds it on the host with per-thread
// dense flag arrays of tilen entries; here one wave64 per tile-row collects
// the tile columns it touches in a windowed LDS bitmap, and one wave per run
// of those tiles builds their masks in LDS and permutes the entries.
#include <string.h>

#include "tsg_internal.h"

#define WAVES_PER_BLOCK 4
#define BM_WORDS 256  // LDS bitmap window per wave: 256 x 32 = 8192 tile columns
// Tile <-> CSR work split: waves per block, tiles of a tile-row per wave, and
// entries of a batch of at most 64 tiles that are permuted through LDS.
#define CV_WAVES 4
#define CV_SEG 1024
#define CV_CAP 448
#define CV_ROUNDS (CV_CAP / 64)

// First index in [lo, hi) with list[index] >= key (list ascending; any list
// ends in range).
__device__ __forceinline__ int first_ge(const int *__restrict__ list, int lo, int hi, int key) {
    while (lo < hi) {
        const int mid = (int)(((unsigned)lo + (unsigned)hi) >> 1);
        if (list[mid] < key) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// The same by a whole wave: 64 probes a step.
__device__ __forceinline__ int wave_first_ge(const int *__restrict__ list, int lo, int hi, int key) {
    const int lane = __lane_id();
    while (hi - lo > 64) {
        const int step = (int)(((unsigned)(hi - lo) + 63u) / 64u);
        const int p = min(lo + (int)min((long long)step * (lane + 1) - 1, (long long)(hi - lo - 1)), hi - 1);
        const int k = __popcll(__ballot(list[p] < key));  // probes ascend: a prefix of the lanes
        const int lo0 = lo;
        if (k > 0) lo = lo0 + (int)min((long long)step * k, (long long)(hi - lo0));
        if (k < 64) hi = lo0 + (int)min((long long)step * (k + 1) - 1, (long long)(hi - lo0 - 1));
    }
    const bool less = lo + lane < hi && list[lo + lane] < key;
    return lo + __popcll(__ballot(less));
}
// The same for 16 searches by a wave, lane's search = lane & 15, its four
// lanes probing a fifth apart.
__device__ __forceinline__ int rows16_first_ge(const int *__restrict__ list, int lo, int hi, int key) {
    const int lane = __lane_id(), g = lane >> 4, r = lane & 15;
    while (__ballot(lo < hi)) {
        const unsigned n = (unsigned)(hi - lo);  // 0 once done
        const int p = lo + (int)((n * (unsigned long long)(g + 1)) / 5u);  // the four ascend, all below hi if n > 0
        const bool less = n > 0 && list[p] < key;
        const int k = __popcll((__ballot(less) >> r) & 0x0001000100010001ull);
        const int lo0 = lo;
        if (n > 0) {
            if (k > 0) lo = lo0 + (int)((n * (unsigned long long)k) / 5u) + 1;
            if (k < 4) hi = lo0 + (int)((n * (unsigned long long)(k + 1)) / 5u);
        }
    }
    return lo;
}

// ---------------------------------------------------------------- input checks
// Input contract of the conversion: row pointers non-decreasing from 0 to
// nnz, columns in [0, n) and (when `sorted`) strictly increasing inside each
// row.  Any violation sets a flag instead of letting a later kernel index
// out of range.  The first nrow blocks check the row pointers, the others
// VAL_BLOCK entries each: a column not above its predecessor is allowed at a
// row's first entry only (the row starts of the block as bits in LDS).
// Entry parallel, so a hub row is not one lane's walk: R-MAT scale 18 5.07
// -> 0.05 ms, 27p 96^3 0.30 -> 0.035 ms.
#define VAL_BLOCK 4096
#define VAL_MARK_ROWS 16384  // rows starting in a block that are marked; more are searched
__global__ void __launch_bounds__(256)
k_validate_csr(const int *__restrict__ rowptr, const int *__restrict__ colidx, int m, int n, int nnz,
               int sorted, int nrow, int *__restrict__ bad) {
    if ((int)blockIdx.x < nrow) {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if (i > m) return;
        const int s = rowptr[i];
        if (i == 0 && s != 0) atomicOr(bad, 1);
        if (i == m) {
            if (s != nnz) atomicOr(bad, 1);
            return;
        }
        const int e = rowptr[i + 1];
        if (s < 0 || e < s || e > nnz) atomicOr(bad, 1);
        return;
    }
    const int end = min(nnz, max(rowptr[m], 0));  // nothing past what the rows claim is read
    const long long b0 = (long long)(blockIdx.x - nrow) * VAL_BLOCK;
    if (b0 >= end) return;
    const int e0 = (int)b0, ne = (int)min((long long)VAL_BLOCK, end - b0);
    __shared__ int s_lo[2];
    __shared__ unsigned s_start[VAL_BLOCK / 32];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (tid < VAL_BLOCK / 32) s_start[tid] = 0u;
    if (sorted && wave < 2) {  // rows starting in [e0, e0 + ne)
        const int i = wave_first_ge(rowptr, 0, m + 1, wave ? e0 + ne : e0);
        if (lane == 0) s_lo[wave] = i;
    }
    // a wave's entries: 64 consecutive ones per round
    int c[VAL_BLOCK / 256], p[VAL_BLOCK / 256];
#pragma unroll
    for (int k = 0; k < VAL_BLOCK / 256; k++) {
        const int x = (k * 4 + wave) * 64;
        c[k] = colidx[e0 + min(x + lane, ne - 1)];
        p[k] = colidx[max(e0 + min(x, ne - 1) - 1, 0)];  // wave-uniform
    }
    __syncthreads();
    bool marked = true;
    if (sorted) {
        const int lo = s_lo[0], hi = s_lo[1];
        marked = hi - lo <= VAL_MARK_ROWS;
        if (marked)
            for (int i = lo + tid; i < hi; i += 256) {
                const int x = rowptr[i] - e0;
                if (x >= 0 && x < ne) atomicOr(&s_start[x >> 5], 1u << (x & 31));
            }
        __syncthreads();
    }
    int f = 0;
#pragma unroll
    for (int k = 0; k < VAL_BLOCK / 256; k++) {
        const int x = (k * 4 + wave) * 64 + lane;
        int prev = __shfl_up(c[k], 1, 64);
        if (lane == 0) prev = p[k];
        if (x >= ne) continue;
        if (c[k] < 0 || c[k] >= n) f = 2;
        if (sorted && e0 + x > 0 && c[k] <= prev) {
            if (marked) {
                if (!((s_start[x >> 5] >> (x & 31)) & 1u)) f = 2;
            } else {
                const int i = first_ge(rowptr, s_lo[0], s_lo[1], e0 + x);
                if (i > m || rowptr[i] != e0 + x) f = 2;
            }
        }
    }
    if (f) atomicOr(bad, f);
}

static int launch_validate(tsg_ctx *ctx, const tsg_dcsr *a, int sorted, int *bad) {
    const unsigned nrow = tsg_div_up((long long)a->m + 1, 256), ncol = tsg_div_up(a->nnz, VAL_BLOCK);
    hipLaunchKernelGGL(k_validate_csr, dim3(nrow + ncol), dim3(256), 0, ctx->stream, a->rowptr, a->colidx, a->m, a->n,
                       a->nnz, sorted, (int)nrow, bad);
    TSG_LAUNCH_CHECK();
    return TSG_OK;
}

static int validate_status(long long bad, int sorted) {
    if (!bad) return TSG_OK;
    tsg_set_error(bad & 1 ? "CSR row pointers inconsistent with nnz"
                  : sorted ? "CSR columns out of range or not strictly increasing inside a row"
                           : "CSR columns out of range");
    return TSG_ERR_ARG;
}

int tsg_validate_csr_mode(tsg_ctx *ctx, const tsg_dcsr *a, int sorted) {
    void *scr;
    TSG_TRY(tsg_scratch(ctx, 64, &scr));
    TSG_HIP(hipMemsetAsync(scr, 0, 4, ctx->stream));
    TSG_TRY(launch_validate(ctx, a, sorted, (int *)scr));
    long long bad = 0;
    TSG_TRY(tsg_read_scalar_i64(ctx, scr, 0, &bad));
    return validate_status(bad, sorted);
}

int tsg_validate_csr(tsg_ctx *ctx, const tsg_dcsr *a) { return tsg_validate_csr_mode(ctx, a, 1); }

// ---------------------------------------------------------------- CSR -> tiles
// Counters of one conversion (zeroed beforehand): a flag for bad input, the
// tile-rows left to k_c2t_tiles_big, the runs of tiles past a tile-row's
// first CV_SEG.
struct C2tCount {
    int bad, nbig, nitems, pad;
};
#define C2T_BIG 4096  // entries of a tile-row above which a whole block collects its tiles

// Tiles of each tile-row: their number into cnt[I], their columns into
// list[rowptr[16I]..) (a tile has an entry, so they fit).  One wave per
// tile-row; a tile-row of more than C2T_BIG entries is put on the list of
// k_c2t_tiles_big.  Row pointers and columns are used only as far as they
// are in range: the input is checked in the same stream, not before.
__global__ void __launch_bounds__(64 * WAVES_PER_BLOCK)
k_c2t_tiles(const int *__restrict__ rowptr, const int *__restrict__ colidx, int m, int nnz, int tilem, int tilen,
            int *__restrict__ cnt, int *__restrict__ list, C2tCount *__restrict__ count, int *__restrict__ big,
            int maxbig, int2 *__restrict__ items, int maxitems) {
    __shared__ unsigned bm_all[WAVES_PER_BLOCK][BM_WORDS];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int I = blockIdx.x * WAVES_PER_BLOCK + wave;
    if (I >= tilem) return;
    unsigned *bm = bm_all[wave];
    const int r0 = I * TSG_TILE, rl = min(TSG_TILE, m - r0);
    const int rp = rowptr[r0 + min(lane, rl)], rpe = rowptr[r0 + min(lane + 1, rl)];
    if (__ballot(rp < 0 || rpe < rp || rpe > nnz)) {  // reported by the input check
        if (lane == 0) cnt[I] = 0;
        return;
    }
    const int e0 = __builtin_amdgcn_readlane(rp, 0), e1 = __builtin_amdgcn_readlane(rpe, 63);
    if (e1 - e0 > C2T_BIG) {
        if (lane == 0) {
            const int s = atomicAdd(&count->nbig, 1);
            if (s < maxbig) big[s] = I;
            cnt[I] = 0;
        }
        return;
    }
    int jmin = 0x7fffffff, jmax = -1;
    if (lane < rl && rpe > rp) {
        jmin = max(colidx[rp] >> 4, 0);
        jmax = min(colidx[rpe - 1] >> 4, tilen - 1);
    }
    jmin = tsg_wave_min(jmin);
    jmax = tsg_wave_max(jmax);
    int total = 0;
    for (int w0 = jmin; w0 <= jmax; w0 += 32 * BM_WORDS) {
        const int nw = min(BM_WORDS, ((jmax - w0) >> 5) + 1);
        for (int k = lane; k < nw; k += 64) bm[k] = 0u;
        tsg_wave_sync();
        for (int x = lane; x < e1 - e0; x += 256) {
            int d[4];
#pragma unroll
            for (int v = 0; v < 4; v++) d[v] = colidx[e0 + min(x + 64 * v, e1 - e0 - 1)];
#pragma unroll
            for (int v = 0; v < 4; v++) {  // a repeated last entry sets its bit again
                const int j = (d[v] >> 4) - w0;
                if (j >= 0 && j < 32 * nw) atomicOr(&bm[j >> 5], 1u << (j & 31));
            }
        }
        tsg_wave_sync();
        total += emit_window(bm, nw, w0, lane, list + e0 + total);
        tsg_wave_sync();
    }
    if (lane == 0) {
        cnt[I] = total;
        const int more = (total - 1) / CV_SEG;  // runs past the first
        if (total > CV_SEG) {
            const int s = atomicAdd(&count->nitems, more);
            for (int k = 0; k < more && s + k < maxitems; k++) items[s + k] = make_int2(I, k + 1);
        }
    }
}

// The same by a block of 16 waves per listed tile-row, with a window of
// 8192 words.
#define C2T_BIG_WORDS 8192
__global__ void __launch_bounds__(1024)
k_c2t_tiles_big(const int *__restrict__ rowptr, const int *__restrict__ colidx, int m, int tilen,
                int *__restrict__ cnt, int *__restrict__ list, C2tCount *__restrict__ count,
                const int *__restrict__ big, int maxbig, int2 *__restrict__ items, int maxitems) {
    __shared__ unsigned bm[C2T_BIG_WORDS];
    __shared__ int s_j[2], s_w[16];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nbig = min(count->nbig, maxbig);
    for (int q = blockIdx.x; q < nbig; q += gridDim.x) {
        const int I = big[q];
        const int r0 = I * TSG_TILE, rl = min(TSG_TILE, m - r0);
        const int e0 = rowptr[r0], e1 = rowptr[r0 + rl];
        if (wave == 0) {
            int jmin = 0x7fffffff, jmax = -1;
            if (lane < rl) {
                const int a = rowptr[r0 + lane], b = rowptr[r0 + lane + 1];
                if (b > a) {
                    jmin = max(colidx[a] >> 4, 0);
                    jmax = min(colidx[b - 1] >> 4, tilen - 1);
                }
            }
            jmin = tsg_wave_min(jmin);
            jmax = tsg_wave_max(jmax);
            if (lane == 0) {
                s_j[0] = jmin;
                s_j[1] = jmax;
            }
        }
        __syncthreads();
        const int jmin = s_j[0], jmax = s_j[1];
        int total = 0;
        for (int w0 = jmin; w0 <= jmax; w0 += 32 * C2T_BIG_WORDS) {
            const int nw = min(C2T_BIG_WORDS, ((jmax - w0) >> 5) + 1);
            for (int k = tid; k < nw; k += 1024) bm[k] = 0u;
            __syncthreads();
            const unsigned ne = (unsigned)(e1 - e0);
            for (unsigned x = tid; x < ne; x += 4096) {
                int d[4];
#pragma unroll
                for (int v = 0; v < 4; v++) d[v] = colidx[e0 + (int)min(x + 1024u * v, ne - 1u)];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int j = (d[v] >> 4) - w0;
                    if (j >= 0 && j < 32 * nw) {
                        const unsigned bit = 1u << (j & 31);
                        if (!(bm[j >> 5] & bit)) atomicOr(&bm[j >> 5], bit);
                    }
                }
            }
            __syncthreads();
            // each wave counts, then emits, a sixteenth of the words
            const int per = (nw + 15) / 16, k0 = min(nw, wave * per), k1 = min(nw, k0 + per);
            int c = 0;
            for (int k = k0 + lane; k < k1; k += 64) c += __popc(bm[k]);
            c = tsg_wave_sum(c);
            if (lane == 0) s_w[wave] = c;
            __syncthreads();
            int before = 0, all = 0;
            for (int w = 0; w < 16; w++) {
                before += w < wave ? s_w[w] : 0;
                all += s_w[w];
            }
            emit_window(bm + k0, k1 - k0, w0 + 32 * k0, lane, list + e0 + total + before);
            total += all;
            __syncthreads();
        }
        if (tid == 0) {
            cnt[I] = total;
            if (total > CV_SEG) {
                const int more = (total - 1) / CV_SEG;
                const int s = atomicAdd(&count->nitems, more);
                for (int k = 0; k < more && s + k < maxitems; k++) items[s + k] = make_int2(I, k + 1);
            }
        }
        __syncthreads();  // s_j
    }
}

// Masks, offsets, columns and values of the tiles, one wave per run of at
// most CV_SEG tiles of a tile-row (the first tilem waves the first runs, the
// others the item list), in batches of 64 tiles.  The entries of a batch are
// one range of each of the 16 rows (the columns ascend), and the entries of
// the tile-row before the batch are those before the ranges, so a run needs
// nothing from the runs before it.  Masks are OR-ed in LDS; an entry's place
// is its tile's and row's offset plus the mask bits before its own.  Batches
// of up to CV_CAP entries keep their entries in registers between the two
// and are permuted through LDS; denser ones are read twice and written in
// place, in runs of up to 16.  Bound by HBM: 12 bytes in and 9 out per entry
// plus 60 per tile.  One thread per matrix row (two walks of its entries,
// 64 lines per instruction, a hub row on one lane): 27p 96^3 1.38 ->
// 0.115 ms (4.4 TB/s), R-MAT scale 18 66.9 -> 0.55 ms.
__global__ void __launch_bounds__(64 * CV_WAVES)
k_c2t_fill(const int *__restrict__ rowptr, const int *__restrict__ colidx, const double *__restrict__ val, int m,
           int tilem, int nnz, int numtile, const int *__restrict__ tile_ptr, const int *__restrict__ list,
           const int2 *__restrict__ items, const C2tCount *__restrict__ count, int nblocks_rows,
           int *__restrict__ tile_colidx, int *__restrict__ tile_rowidx, int *__restrict__ tile_nnz,
           unsigned char *__restrict__ csr_ptr, unsigned short *__restrict__ mask, unsigned char *__restrict__ tcol,
           double *__restrict__ tval) {
    __shared__ double s_val[CV_WAVES][CV_CAP];
    __shared__ __align__(16) unsigned s_mask[CV_WAVES][64 * 8];  // two rows per word, even row low
    __shared__ uint4 s_ptr[CV_WAVES][64];
    __shared__ int s_J[CV_WAVES][64];
    __shared__ int s_off[CV_WAVES][16], s_src[CV_WAVES][16];
    __shared__ unsigned short s_toff[CV_WAVES][64];
    __shared__ unsigned char s_c8[CV_WAVES][CV_CAP];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15;
    unsigned *sm = s_mask[wave];
    int *sJ = s_J[wave], *so = s_off[wave], *ss = s_src[wave];
    if (blockIdx.x == 0 && threadIdx.x < 16) {  // the arrays' tails
        csr_ptr[16 * (long long)numtile + threadIdx.x] = 0;
        mask[16 * (long long)numtile + threadIdx.x] = 0;
        if (threadIdx.x == 0) tile_nnz[numtile] = nnz;
    }
    const bool listed = (int)blockIdx.x >= nblocks_rows;
    const int nwork = listed ? count->nitems : tilem;
    const int step = listed ? (int)(gridDim.x - nblocks_rows) * CV_WAVES : tilem;
    for (int w = (listed ? (int)blockIdx.x - nblocks_rows : (int)blockIdx.x) * CV_WAVES + wave; w < nwork; w += step) {
        const int I = listed ? items[w].x : w, sg = listed ? items[w].y : 0;
        const int t0 = tile_ptr[I], t1 = tile_ptr[I + 1], ta = t0 + sg * CV_SEG, te = min(t1, ta + CV_SEG);
        if (ta >= te) continue;
        // lanes r, r + 16, ...: row r's entries [rp, rpe) and where its next range starts
        const int rp = rowptr[min(16 * I + r, m)], rpe = rowptr[min(16 * I + r + 1, m)];
        const int e0 = __builtin_amdgcn_readlane(rp, 0);
        const int *tl = list + e0 - t0;  // tile columns by tile id
        int cur = sg == 0 ? rp : rows16_first_ge(colidx, rp, rpe, tl[ta] * 16);
        for (int tb = ta; tb < te; tb += 64) {
            const int nt = min(64, te - tb);
            const int J = tl[tb + min(lane, nt - 1)];
            // rows end with the tile-row's last tile; otherwise 64 tiles hold at most 1024 of a row's entries
            int end = rpe;
            if (tb + nt < t1)
                end = rows16_first_ge(colidx, cur, cur + min(rpe - cur, 1024), (__builtin_amdgcn_readlane(J, nt - 1) + 1) * 16);
            const int len = end - cur, incl = tsg_row16_incl_scan_dpp(len);
            const int total = __builtin_amdgcn_readlane(incl, 15);
            const int base = e0 + __builtin_amdgcn_readlane(tsg_row16_incl_scan_dpp(cur - rp), 15);
            if (lane < 16) {
                so[lane] = incl - len;
                ss[lane] = cur - (incl - len);
            }
            cur = end;
            sJ[lane] = lane < nt ? J : 0x7fffffff;
            for (int i = lane; i < 64 * 2; i += 64) reinterpret_cast<uint4 *>(sm)[i] = make_uint4(0u, 0u, 0u, 0u);
            tsg_wave_sync();
            // entry x of the batch: its row (the last whose range starts at or before x), then its tile
            auto row_of = [&](int x) {
                int q = 0;
#pragma unroll
                for (int st = 8; st > 0; st >>= 1)
                    if (so[q + st] <= x) q += st;
                return q;
            };
            auto tile_of = [&](int c) {
                int k = 0;
#pragma unroll
                for (int st = 32; st > 0; st >>= 1)
                    if (sJ[k + st] <= (c >> 4)) k += st;
                return k;
            };
            int code[CV_ROUNDS];  // column, then tile << 8 | in-tile column << 4 | row
            unsigned rows = 0;    // four bits per round
            static_assert(CV_ROUNDS <= 8, "rows of a lane's entries in one word");
            double v[CV_ROUNDS];
            if (total <= CV_CAP) {
#pragma unroll
                for (int i = 0; i < CV_ROUNDS; i++) {  // every lane loads in bounds
                    const int x = min(lane + 64 * i, total - 1), q = row_of(x), e = ss[q] + x;
                    v[i] = val[e];
                    code[i] = colidx[e];
                    rows |= (unsigned)q << (4 * i);
                }
#pragma unroll
                for (int i = 0; i < CV_ROUNDS; i++) {
                    const int q = (rows >> (4 * i)) & 15, c = code[i], k = tile_of(c);
                    code[i] = k << 8 | (c & 15) << 4 | q;
                    if (lane + 64 * i < total) atomicOr(&sm[k * 8 + (q >> 1)], (0x8000u >> (c & 15)) << (16 * (q & 1)));
                }
            } else {
                for (int x = lane; x < total; x += 64) {
                    const int q = row_of(x), c = colidx[ss[q] + x], k = tile_of(c);
                    atomicOr(&sm[k * 8 + (q >> 1)], (0x8000u >> (c & 15)) << (16 * (q & 1)));
                }
            }
            tsg_wave_sync();
            // lane = tile: row offsets, entries
            const uint4 ma = reinterpret_cast<const uint4 *>(sm)[2 * lane], mb = reinterpret_cast<const uint4 *>(sm)[2 * lane + 1];
            const unsigned mw[8] = {ma.x, ma.y, ma.z, ma.w, mb.x, mb.y, mb.z, mb.w};
            unsigned o[4];
            int sum = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                o[q] = 0;
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    o[q] |= (unsigned)sum << (8 * b);
                    sum += __popc((mw[2 * q + (b >> 1)] >> (16 * (b & 1))) & 0xffffu);
                }
            }
            const int toff = tsg_wave_incl_scan_dpp(sum) - sum;
            s_ptr[wave][lane] = make_uint4(o[0], o[1], o[2], o[3]);
            s_toff[wave][lane] = (unsigned short)toff;
            if (lane < nt) {
                const long long t = tb + lane;
                tile_colidx[t] = J;
                tile_rowidx[t] = I;
                tile_nnz[t] = base + toff;
                reinterpret_cast<uint4 *>(csr_ptr)[t] = make_uint4(o[0], o[1], o[2], o[3]);
                reinterpret_cast<uint4 *>(mask)[2 * t] = ma;
                reinterpret_cast<uint4 *>(mask)[2 * t + 1] = mb;
            }
            tsg_wave_sync();
            auto place = [&](int k, int q, int c) {
                const unsigned mr = (sm[k * 8 + (q >> 1)] >> (16 * (q & 1))) & 0xffffu;
                return (int)s_toff[wave][k] + reinterpret_cast<const unsigned char *>(&s_ptr[wave][k])[q] +
                       __popc(mr >> (16 - c));
            };
            if (total <= CV_CAP) {
#pragma unroll
                for (int i = 0; i < CV_ROUNDS; i++) {
                    if (lane + 64 * i >= total) continue;
                    const int q = code[i] & 15, c = (code[i] >> 4) & 15, pos = place(code[i] >> 8, q, c);
                    s_val[wave][pos] = v[i];
                    s_c8[wave][pos] = (unsigned char)c;
                }
                tsg_wave_sync();
                for (int x = lane; x < total; x += 64) {
                    tval[base + x] = s_val[wave][x];
                    tcol[base + x] = s_c8[wave][x];
                }
            } else {
                for (int x = lane; x < total; x += 64) {
                    const int q = row_of(x), e = ss[q] + x, c = colidx[e];
                    const int pos = base + place(tile_of(c), q, c & 15);
                    tval[pos] = val[e];
                    tcol[pos] = (unsigned char)(c & 15);
                }
            }
            tsg_wave_sync();  // the next batch rewrites the LDS arrays
        }
    }
}

extern "C" int tsg_csr2tile(tsg_ctx *ctx, const tsg_dcsr *a, tsg_dtiles *out) {
    memset(out, 0, sizeof(*out));
    if (!a || a->m < 0 || a->n < 0 || a->nnz < 0) { tsg_set_error("tsg_csr2tile: bad matrix"); return TSG_ERR_ARG; }
    tsg_dtiles &T = *out;
    T.m = a->m;
    T.n = a->n;
    T.nnz = a->nnz;
    T.tilem = (a->m + 15) / 16;
    T.tilen = (int)(((long long)a->n + 15) / 16);
    // counters, the tile-rows of more than C2T_BIG entries, the further runs
    // of tiles, the tile columns
    const int maxbig = a->nnz / C2T_BIG + 1, maxitems = a->nnz / CV_SEG + 1;
    const size_t o_big = 64, o_items = o_big + (((size_t)maxbig * 4 + 15) & ~(size_t)15);
    const size_t o_list = o_items + (((size_t)maxitems * 8 + 15) & ~(size_t)15);
    char *buf = nullptr;
    TSG_TRY(tsg_alloc_t(ctx, &T.tile_ptr, (size_t)T.tilem + 1));
    int st = tsg_alloc(ctx, (void **)&buf, o_list + ((size_t)a->nnz + 1) * 4);
    long long numtile = 0;
    if (st == TSG_OK) st = [&]() -> int {
        C2tCount *count = (C2tCount *)buf;
        int *big = (int *)(buf + o_big), *list = (int *)(buf + o_list);
        int2 *items = (int2 *)(buf + o_items);
        hipStream_t s = ctx->stream;
        TSG_HIP(hipMemsetAsync(count, 0, sizeof(C2tCount), s));
        TSG_TRY(launch_validate(ctx, a, 1, &count->bad));
        if (T.tilem > 0) {
            hipLaunchKernelGGL(k_c2t_tiles, dim3(tsg_div_up(T.tilem, WAVES_PER_BLOCK)), dim3(64 * WAVES_PER_BLOCK), 0, s,
                               a->rowptr, a->colidx, a->m, a->nnz, T.tilem, T.tilen, T.tile_ptr, list, count, big,
                               maxbig, items, maxitems);
            TSG_LAUNCH_CHECK();
            if (a->nnz > C2T_BIG) {
                hipLaunchKernelGGL(k_c2t_tiles_big, dim3((unsigned)std::min(maxbig, 512)), dim3(1024), 0, s, a->rowptr,
                                   a->colidx, a->m, T.tilen, T.tile_ptr, list, count, big, maxbig, items, maxitems);
                TSG_LAUNCH_CHECK();
            }
        }
        // a bad input's counts may add up to anything: its flag is looked at first
        const int sc = tsg_scan_i32(ctx, T.tile_ptr, T.tile_ptr, T.tilem, &numtile, &count->bad, 1);
        if (sc != TSG_OK && sc != TSG_ERR_OVERFLOW) return sc;
        TSG_TRY(validate_status(((volatile int *)(ctx->pinned + 1))[0], 1));
        TSG_TRY(sc);
        T.numtile = (int)numtile;
        TSG_TRY(tsg_alloc_t(ctx, &T.tile_colidx, (size_t)numtile + 1));
        TSG_TRY(tsg_alloc_t(ctx, &T.tile_rowidx, (size_t)numtile + 1));
        TSG_TRY(tsg_alloc_t(ctx, &T.tile_nnz, (size_t)numtile + 1));
        TSG_TRY(tsg_alloc_t(ctx, &T.csr_ptr, (size_t)numtile * 16 + 16));
        TSG_TRY(tsg_alloc_t(ctx, &T.mask, (size_t)numtile * 16 + 16));
        TSG_TRY(tsg_alloc_t(ctx, &T.csr_col, (size_t)a->nnz + 1));
        TSG_TRY(tsg_alloc_t(ctx, &T.val, (size_t)a->nnz + 1));
        const unsigned nb = tsg_div_up(T.tilem, CV_WAVES), extra = (unsigned)std::min(maxitems, 1024);
        hipLaunchKernelGGL(k_c2t_fill, dim3(nb + extra), dim3(64 * CV_WAVES), 0, s, a->rowptr, a->colidx, a->val, a->m,
                           T.tilem, a->nnz, T.numtile, T.tile_ptr, list, items, count, (int)nb, T.tile_colidx,
                           T.tile_rowidx, T.tile_nnz, T.csr_ptr, T.mask, T.csr_col, T.val);
        TSG_LAUNCH_CHECK();
        return TSG_OK;
    }();
    tsg_free(ctx, buf);
    if (st != TSG_OK) tsg_tiles_free(ctx, out);
    return st;
}

// ---------------------------------------------------------------- CSC tile index
__global__ void k_iota(int *v, long long n) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) v[i] = (int)i;
}
// keys[i] = src[i], idx[i] = i: the input of a sort by src.
__global__ void __launch_bounds__(256)
k_sort_input(const int *__restrict__ src, long long n, unsigned *__restrict__ keys, int *__restrict__ idx) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        keys[i] = (unsigned)src[i];
        idx[i] = (int)i;
    }
}
// ptr[j] = first position of a key >= j in the sorted keys, j = 0..ncol.  A
// search per pointer: counting the keys instead met one atomic per entry of
// a hub column on one address (R-MAT scale 18: 648 us against 13).
__global__ void __launch_bounds__(256)
k_ptr_of_sorted(const unsigned *__restrict__ keys, long long n, int ncol, int *__restrict__ ptr) {
    const long long j = (long long)blockIdx.x * 256 + threadIdx.x;
    if (j > ncol) return;
    long long lo = 0, hi = n;
    while (lo < hi) {
        const long long mid = (lo + hi) >> 1;
        if (keys[mid] < (unsigned)j) lo = mid + 1; else hi = mid;
    }
    ptr[j] = (int)lo;
}
__global__ void k_gather_i32(const int *__restrict__ src, const int *__restrict__ idx, long long n, int *__restrict__ dst) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[idx[i]];
}
__global__ void k_scatter_i32(const int *__restrict__ src, const int *__restrict__ idx, long long n, int *__restrict__ dst) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[idx[i]] = src[i];
}
__global__ void k_gather_entries(const int *__restrict__ src, const double *__restrict__ val, const int *__restrict__ idx,
                                 long long n, int *__restrict__ dst, double *__restrict__ oval) {
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        const int e = idx[i];
        dst[i] = src[e];
        oval[i] = val[e];
    }
}

static int bits_for(long long v) {
    int b = 1;
    while ((1ll << b) <= v) b++;
    return b;
}

extern "C" int tsg_tiles_build_csc(tsg_ctx *ctx, tsg_dtiles *t) {
    if (t->csc_ptr) return TSG_OK;
    const long long nt = t->numtile;
    TSG_TRY(tsg_alloc_t(ctx, &t->csc_ptr, (size_t)t->tilen + 1));
    TSG_TRY(tsg_alloc_t(ctx, &t->csc_rowidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &t->csc_tileid, (size_t)nt + 1));
    unsigned *keys = nullptr;
    if (nt > 0) {
        TSG_TRY(tsg_alloc_t(ctx, &keys, (size_t)nt));
        hipLaunchKernelGGL(k_sort_input, dim3(tsg_div_up(nt, 256)), dim3(256), 0, ctx->stream, t->tile_colidx, nt, keys,
                           t->csc_tileid);
        TSG_LAUNCH_CHECK();
        TSG_TRY(tsg_sort_pairs_u32(ctx, keys, t->csc_tileid, nt, bits_for(t->tilen)));
        hipLaunchKernelGGL(k_gather_i32, dim3(tsg_div_up(nt, 256)), dim3(256), 0, ctx->stream, t->tile_rowidx,
                           t->csc_tileid, nt, t->csc_rowidx);
        TSG_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_ptr_of_sorted, dim3(tsg_div_up((long long)t->tilen + 1, 256)), dim3(256), 0, ctx->stream,
                       (const unsigned *)keys, nt, t->tilen, t->csc_ptr);
    TSG_LAUNCH_CHECK();
    tsg_free(ctx, keys);
    return TSG_OK;
}

// ---------------------------------------------------------------- tile -> CSR
// Follows tile2csr (src/tile2csr.h:71-137): per-row counts from the tiles of
// the row's tile-row, exclusive scan, then entries copied tile by tile in
// ascending tile column (so columns come out sorted); explicit zeros kept.
// Row r of tile t spans [ptr[r], end) with end = tile nnz for the last row
// of the tile-row (rowlen-1) and ptr[r+1] otherwise (src/tile2csr.h:19-21),
// so only the offsets are needed, not the masks.
__device__ __forceinline__ int t2c_row_len(const int *tile_nnz, const unsigned char *csr_ptr, int t, int r,
                                           int rowlen) {
    const int s = csr_ptr[(long long)t * 16 + r];
    const int e = (r == rowlen - 1) ? tile_nnz[t + 1] - tile_nnz[t] : csr_ptr[(long long)t * 16 + r + 1];
    return e - s;
}

// A tile-row's entries are the same contiguous range in both formats, so the
// conversion is a permutation inside it and needs no scan over the rows:
// row 16I+r starts at the tile-row's first entry plus the entries of its
// rows before r.  Work is one wave per run of at most CV_SEG tiles of a
// tile-row (a hub tile-row's further runs go through an item list, each with
// its 16 rows' entries before it), in batches of at most 64 tiles and CV_CAP
// entries: the batch is loaded as one contiguous range, permuted through
// LDS, and written as 16 row runs.  Bound by HBM: 9 bytes in (plus the tile
// index) and 12 out per entry.  One thread per matrix row walking its tiles
// left 8-byte accesses to 64 different lines per instruction and a hub
// row's whole walk on one lane: 62M entries of a 27-point product (27d
// 79x83x81, A^2) 2.31 -> 0.55 ms for the call, 2.9 TB/s in k_t2c_emit; the
// row index of R-MAT scale 18 17.4 -> 0.37 ms (both kernels).
struct T2cItem {
    int I, seg;     // tiles [CV_SEG * seg, CV_SEG * (seg + 1)) of tile-row I
    int carry[16];  // entries of each row in the tile-row's tiles before them
};

// A tile's row offsets with those past the matrix's rows (rowlen < 16, the
// last tile-row) set to the tile's entry count, at most 240 there.
__device__ __forceinline__ uint4 t2c_offsets(uint4 p, int tnnz, int rowlen) {
    unsigned w[4] = {p.x, p.y, p.z, p.w};
    if (rowlen < 16) {
#pragma unroll
        for (int q = 0; q < 16; q++)
            if (q >= rowlen) w[q >> 2] = (w[q >> 2] & ~(0xffu << (8 * (q & 3)))) | ((unsigned)tnnz << (8 * (q & 3)));
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}
// 16 bytes from an address of any alignment (one load: the target allows
// unaligned global access).
__device__ __forceinline__ uint4 load16(const unsigned char *p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// Entries of each row over up to CV_SEG tiles [ta, te) by a wave starting at
// tile ta + lane with the given stride: v[2q] = rows 4q and 4q+2, v[2q+1] =
// rows 4q+1 and 4q+3 (at most 16 * CV_SEG per half), summed over the wave.
__device__ __forceinline__ void t2c_row_sums(const int *__restrict__ tile_nnz, const unsigned char *__restrict__ csr_ptr,
                                             int ta, int te, int stride, int rowlen, unsigned v[8]) {
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = 0u;
#pragma unroll 4
    for (int t = ta; t < te; t += stride) {
        unsigned x[8];
        const int tn = tile_nnz[t + 1] - tile_nnz[t];
        tile_widen_lens(tile_row_lens(t2c_offsets(load16(csr_ptr + 16 * (long long)t), tn, rowlen), tn), x);
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] += x[q];
    }
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = (unsigned)__builtin_amdgcn_readlane(tsg_wave_incl_scan_dpp((int)v[q]), 63);
}
// Row pointers; one wave per tile-row of up to CV_SEG tiles, a tile per lane,
// the block's four waves together for a longer one.  *nitems (zeroed
// beforehand) counts the further runs (the first maxitems are listed); host
// (pinned) gets the entries and the tiles of the matrix or view.
__global__ void __launch_bounds__(64 * CV_WAVES)
k_t2c_rowptr(int m, int tilem, const int *__restrict__ tile_ptr, const int *__restrict__ tile_nnz,
             const unsigned char *__restrict__ csr_ptr, int *__restrict__ rowptr, T2cItem *__restrict__ items,
             int *__restrict__ nitems, int maxitems, long long *__restrict__ host) {
    __shared__ int s_sum[CV_WAVES][16];
    __shared__ int s_slot;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int nb0 = tile_nnz[tile_ptr[0]];
    const int I = blockIdx.x * CV_WAVES + wave;
    unsigned v[8];
    if (I < tilem) {
        const int t0 = tile_ptr[I], t1 = tile_ptr[I + 1];
        if (t1 - t0 <= CV_SEG) {
            const int rowlen = min(16, m - 16 * I);
            t2c_row_sums(tile_nnz, csr_ptr, t0 + lane, t1, 64, rowlen, v);
            const int c = tile_row_of(v, lane & 15), incl = tsg_row16_incl_scan_dpp(c);
            if (lane < rowlen) rowptr[16 * I + lane] = tile_nnz[t0] - nb0 + incl - c;
        }
        if (I == tilem - 1 && lane == 0) {
            const int nnz = tile_nnz[t1] - nb0;
            rowptr[m] = nnz;
            host[0] = nnz;
            host[1] = t1 - tile_ptr[0];
        }
    }
    for (int w = 0; w < CV_WAVES; w++) {
        const int Iw = blockIdx.x * CV_WAVES + w;
        if (Iw >= tilem) break;
        const int t0 = tile_ptr[Iw], t1 = tile_ptr[Iw + 1];
        if (t1 - t0 <= CV_SEG) continue;  // block-uniform
        const int rowlen = min(16, m - 16 * Iw), nseg = (t1 - t0 + CV_SEG - 1) / CV_SEG;
        if (tid == 0) s_slot = atomicAdd(nitems, nseg - 1);
        __syncthreads();
        const int slot = s_slot;
        int carry = 0;  // threads 0..15: the row's entries so far
        for (int sg = 0; sg < nseg; sg++) {
            if (sg > 0 && tid < 16 && slot + sg <= maxitems) {
                items[slot + sg - 1].carry[tid] = carry;
                if (tid == 0) {
                    items[slot + sg - 1].I = Iw;
                    items[slot + sg - 1].seg = sg;
                }
            }
            t2c_row_sums(tile_nnz, csr_ptr, t0 + sg * CV_SEG + tid, min(t1, t0 + (sg + 1) * CV_SEG), 64 * CV_WAVES,
                         rowlen, v);
            if (lane < 16) s_sum[wave][lane] = tile_row_of(v, lane);
            __syncthreads();
            if (tid < 16)
                for (int w2 = 0; w2 < CV_WAVES; w2++) carry += s_sum[w2][tid];
            __syncthreads();
        }
        if (tid < 16) {
            const int incl = tsg_group16_incl_scan(carry);
            if (tid < rowlen) rowptr[16 * Iw + tid] = tile_nnz[t0] - nb0 + incl - carry;
        }
        __syncthreads();  // s_slot
    }
}

// Entries: the first tilem waves take each tile-row's first run, the others
// the item list.  One lane per entry: its tile from a mark at each tile's
// first entry (running maximum over the lanes), its row from the tile's row
// offsets, its place in the batch from the (tile, row)'s entries before it.
__global__ void __launch_bounds__(64 * CV_WAVES)
k_t2c_emit(int m, int tilem, const int *__restrict__ tile_ptr, const int *__restrict__ tile_colidx,
           const int *__restrict__ tile_nnz, const unsigned char *__restrict__ csr_ptr,
           const unsigned char *__restrict__ tcol, const double *__restrict__ tval, const int *__restrict__ rowptr,
           const T2cItem *__restrict__ items, const int *__restrict__ nitems, int nblocks_rows, int jbase,
           int *__restrict__ col, double *__restrict__ val) {
    static_assert(CV_CAP % 64 == 0 && CV_CAP >= 256, "whole rounds; a full tile fits");
    // per wave: the batch's values, columns and rows in output order (the
    // row bytes first hold the tile marks), each tile's row offsets, and each
    // (tile, row)'s first output position (row 64: the rows' ends)
    __shared__ double s_val[CV_WAVES][CV_CAP];
    __shared__ int s_col[CV_WAVES][CV_CAP];
    __shared__ __align__(16) unsigned char s_row[CV_WAVES][CV_CAP];
    __shared__ uint4 s_p16[CV_WAVES][64];
    __shared__ __align__(16) unsigned short s_pre[CV_WAVES][65 * 16];
    __shared__ int s_dst[CV_WAVES][16];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15;
    double *sv = s_val[wave];
    int *sc = s_col[wave], *sd = s_dst[wave];
    unsigned char *sr = s_row[wave];
    unsigned short *sp = s_pre[wave];
    const bool listed = (int)blockIdx.x >= nblocks_rows;
    const int nwork = listed ? *nitems : tilem;
    const int step = listed ? (int)(gridDim.x - nblocks_rows) * CV_WAVES : tilem;
    for (int w = (listed ? (int)blockIdx.x - nblocks_rows : (int)blockIdx.x) * CV_WAVES + wave; w < nwork; w += step) {
        const int I = listed ? items[w].I : w, sg = listed ? items[w].seg : 0;
        const int rowlen = min(16, m - 16 * I);
        const int t1 = tile_ptr[I + 1], ta = tile_ptr[I] + sg * CV_SEG, te = min(t1, ta + CV_SEG);
        // lanes r, r + 16, ...: where row r's next run starts in the output
        int gout = r < rowlen ? rowptr[16 * I + r] : 0;
        if (listed) gout += items[w].carry[r];
        for (int tb = ta; tb < te;) {
            const int t = min(tb + lane, te - 1);
            const int n0 = tile_nnz[t], n1 = tile_nnz[t + 1];
            const uint4 p16 = t2c_offsets(load16(csr_ptr + 16 * (long long)t), n1 - n0, rowlen);
            const int J16 = (tile_colidx[t] - jbase) * 16;
            const int start = __builtin_amdgcn_readfirstlane(n0);
            // the batch: the leading tiles whose entries fit (a tile holds at most 256)
            const int nt = __popcll(__ballot(tb + lane < te && n1 - start <= CV_CAP));
            const int total = __builtin_amdgcn_readlane(n1, nt - 1) - start;
            if (total == 0) {
                tb += nt;
                continue;
            }
            double v[CV_ROUNDS];
            unsigned char c8[CV_ROUNDS];
#pragma unroll
            for (int i = 0; i < CV_ROUNDS; i++) {  // every lane loads in bounds
                const int x = min(lane + 64 * i, total - 1);
                v[i] = tval[start + x];
                c8[i] = tcol[start + x];
            }
            // tile marks (k + 1 at each nonempty tile's first entry), row offsets
            for (int i = lane; i < CV_CAP / 4; i += 64) reinterpret_cast<unsigned *>(sr)[i] = 0u;
            s_p16[wave][lane] = p16;
            tsg_wave_sync();
            if (lane < nt && n1 > n0) sr[n0 - start] = (unsigned char)(lane + 1);
            // entries of each row in the tiles before the lane's; the rows' runs
            unsigned len[8], tot[8];
            tile_widen_lens(tile_row_lens(p16, n1 - n0), len);
            unsigned run = 0;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                if (lane >= nt) len[q] = 0u;
                const unsigned incl = (unsigned)tsg_wave_incl_scan_dpp((int)len[q]);
                tot[q] = (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
                len[q] = incl - len[q];  // from here on: before the lane's tile
            }
            unsigned *spw = reinterpret_cast<unsigned *>(sp);
#pragma unroll
            for (int q = 0; q < 4; q++) {  // rows 4q..4q+3 in order
                const unsigned r0 = run, r1 = r0 + (tot[2 * q] & 0xffffu), r2 = r1 + (tot[2 * q + 1] & 0xffffu);
                const unsigned r3 = r2 + (tot[2 * q] >> 16);
                run = r3 + (tot[2 * q + 1] >> 16);
                const unsigned e = len[2 * q] + (r0 | (r2 << 16)), o = len[2 * q + 1] + (r1 | (r3 << 16));
                spw[lane * 8 + 2 * q] = (e & 0xffffu) | (o << 16);
                spw[lane * 8 + 2 * q + 1] = (e >> 16) | (o & 0xffff0000u);
                if (lane == 0) {
                    spw[64 * 8 + 2 * q] = r1 | (r2 << 16);
                    spw[64 * 8 + 2 * q + 1] = r3 | (run << 16);
                }
            }
            tsg_wave_sync();
            const int rend = sp[64 * 16 + r], rbeg = r ? sp[64 * 16 + r - 1] : 0;
            if (lane < 16) sd[lane] = gout - rbeg;
            gout += rend - rbeg;
            int k[CV_ROUNDS], last = 0;
#pragma unroll
            for (int i = 0; i < CV_ROUNDS; i++) {
                k[i] = max(last, tsg_wave_incl_max_dpp((int)sr[lane + 64 * i]));
                last = __builtin_amdgcn_readlane(k[i], 63);
            }
            tsg_wave_sync();  // the marks are read; their bytes take the rows
#pragma unroll
            for (int i = 0; i < CV_ROUNDS; i++) {
                const int x = lane + 64 * i;
                const int kk = k[i] - 1;
                const int j = x - (__shfl(n0, kk, 64) - start), Jk = __shfl(J16, kk, 64);
                if (x < total) {
                    const uint4 pk = s_p16[wave][kk];
                    // the last row starting at or before entry j
                    const int rr = __popc(bytes_le(pk.x, j)) + __popc(bytes_le(pk.y, j)) + __popc(bytes_le(pk.z, j)) +
                             __popc(bytes_le(pk.w, j)) - 1;
                    const int pos = sp[kk * 16 + rr] + j - reinterpret_cast<const unsigned char *>(&s_p16[wave][kk])[rr];
                    sv[pos] = v[i];
                    sc[pos] = Jk + c8[i];
                    sr[pos] = (unsigned char)rr;
                }
            }
            tsg_wave_sync();
            for (int o = lane; o < total; o += 64) {
                const int d = sd[sr[o]] + o;
                col[d] = sc[o];
                val[d] = sv[o];
            }
            tsg_wave_sync();  // the next batch rewrites the LDS arrays
            tb += nt;
        }
    }
}

extern "C" int tsg_tile2csr(tsg_ctx *ctx, const tsg_dtiles *t, tsg_dcsr *out) {
    return tsg_tile2csr_view(ctx, t, 0, out);
}

// buf: the further runs' count, then the runs (the caller frees it)
static int tile2csr_run(tsg_ctx *ctx, const tsg_dtiles *t, int jbase, tsg_dcsr *out, char **buf) {
    TSG_TRY(tsg_alloc_t(ctx, &out->rowptr, (size_t)t->m + 1));
    if (t->m <= 0) {
        TSG_HIP(hipMemsetAsync(out->rowptr, 0, 4, ctx->stream));
        TSG_TRY(tsg_alloc_t(ctx, &out->colidx, 1));
        TSG_TRY(tsg_alloc_t(ctx, &out->val, 1));
        return TSG_OK;
    }
    const int tilem = (int)tsg_div_up(t->m, 16);
    const unsigned nb = tsg_div_up(tilem, CV_WAVES);
    long long maxitems = 0, nnz = 0;
    for (long long tiles = std::max(t->numtile, 0);;) {
        maxitems = tiles / CV_SEG + 1;  // further runs: at most one per CV_SEG tiles
        TSG_TRY(tsg_alloc(ctx, (void **)buf, 64 + (size_t)maxitems * sizeof(T2cItem)));
        TSG_HIP(hipMemsetAsync(*buf, 0, 4, ctx->stream));
        hipLaunchKernelGGL(k_t2c_rowptr, dim3(nb), dim3(64 * CV_WAVES), 0, ctx->stream, t->m, tilem, t->tile_ptr,
                           t->tile_nnz, t->csr_ptr, out->rowptr, (T2cItem *)(*buf + 64), (int *)*buf, (int)maxitems,
                           ctx->pinned);
        TSG_LAUNCH_CHECK();
        TSG_HIP(hipStreamSynchronize(ctx->stream));
        nnz = ((volatile long long *)ctx->pinned)[0];
        const long long have = ((volatile long long *)ctx->pinned)[1];
        if (have <= tiles) break;
        tiles = have;  // a view whose numtile is not its own: once more, with room for every run
        tsg_free(ctx, *buf);
        *buf = nullptr;
    }
    const T2cItem *items = (const T2cItem *)(*buf + 64);
    const int *nitems = (const int *)*buf;
    out->nnz = (int)nnz;
    TSG_TRY(tsg_alloc_t(ctx, &out->colidx, (size_t)nnz + 1));
    TSG_TRY(tsg_alloc_t(ctx, &out->val, (size_t)nnz + 1));
    if (nnz > 0) {
        const unsigned extra = (unsigned)std::min<long long>(maxitems, 1024);
        hipLaunchKernelGGL(k_t2c_emit, dim3(nb + extra), dim3(64 * CV_WAVES), 0, ctx->stream, t->m, tilem, t->tile_ptr,
                           t->tile_colidx, t->tile_nnz, t->csr_ptr, t->csr_col, t->val, out->rowptr, items, nitems,
                           (int)nb, jbase, out->colidx, out->val);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

// t may be a view of a tile-row range of a larger tile matrix (tile_ptr
// pointing into the parent's, every other array the parent's, indices
// absolute); output columns are taken relative to tile column jbase.
int tsg_tile2csr_view(tsg_ctx *ctx, const tsg_dtiles *t, int jbase, tsg_dcsr *out) {
    memset(out, 0, sizeof(*out));
    out->m = t->m;
    out->n = t->n;
    char *buf = nullptr;
    const int st = tile2csr_run(ctx, t, jbase, out, &buf);
    tsg_free(ctx, buf);
    if (st != TSG_OK) tsg_dcsr_free(ctx, out);  // what it got before the error
    return st;
}

// ------------------------------------------------------------------ checksums, sampled rows
// splitmix64's finalizer: a bijective 64-bit mix.
__device__ __forceinline__ unsigned long long csum_mix(unsigned long long x) {
    x ^= x >> 30;
    x *= 0xbf58476d1ce4e5b9ull;
    x ^= x >> 27;
    x *= 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// One thread per row of the view: the row's entries (as tile2csr emits
// them) and its share of every tile of the tile-row (row mask and row
// offset; row 0 adds the tile's nonzero count).  Sums are order-free, so
// they add up over chunks.  acc[0] tiles, acc[1] entries, acc[2] nonzeros,
// acc[3] tiles counted, acc[4] entries with row and column swapped (equal
// to acc[1] exactly when C is bit-symmetric).
__global__ void __launch_bounds__(256)
k_checksum(int m, const int *__restrict__ tile_ptr, const int *__restrict__ tile_colidx,
           const int *__restrict__ tile_nnz, const unsigned char *__restrict__ csr_ptr,
           const unsigned short *__restrict__ mask, const unsigned char *__restrict__ tcol,
           const double *__restrict__ tval, long long row_base, int jbase, unsigned long long *__restrict__ acc) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    unsigned long long ht = 0, he = 0, hx = 0, nz = 0, nt = 0;
    if (i < m) {
        const int I = i >> 4, r = i & 15;
        const int rowlen = min(16, m - I * 16);
        const long long row = row_base + i, Ig = (row_base >> 4) + I;
        for (int t = tile_ptr[I]; t < tile_ptr[I + 1]; t++) {
            const long long J = tile_colidx[t] - jbase;
            const unsigned long long tk = csum_mix(((unsigned long long)Ig << 32) ^ (unsigned long long)J);
            ht += csum_mix(tk ^ ((unsigned long long)(r + 1) << 40) ^
                           ((unsigned long long)mask[(long long)t * 16 + r] << 8) ^ csr_ptr[(long long)t * 16 + r]);
            if (r == 0) {
                ht += csum_mix(tk + (unsigned long long)(tile_nnz[t + 1] - tile_nnz[t]));
                nt++;
            }
            const int k = t2c_row_len(tile_nnz, csr_ptr, t, r, rowlen);
            const int s = tile_nnz[t] + csr_ptr[(long long)t * 16 + r];
            for (int j = 0; j < k; j++) {
                const unsigned long long col = (unsigned long long)(J * 16 + tcol[s + j]);
                const unsigned long long vb = (unsigned long long)__double_as_longlong(tval[s + j]);
                he += csum_mix(csum_mix(((unsigned long long)row << 32) ^ col) ^ vb);
                hx += csum_mix(csum_mix((col << 32) ^ (unsigned long long)row) ^ vb);
            }
            nz += k > 0 ? k : 0;
        }
    }
    ht = tsg_wave_sum(ht);
    he = tsg_wave_sum(he);
    hx = tsg_wave_sum(hx);
    nz = tsg_wave_sum(nz);
    nt = tsg_wave_sum(nt);
    if (__lane_id() == 0) {
        atomicAdd(&acc[0], ht);
        atomicAdd(&acc[1], he);
        atomicAdd(&acc[2], nz);
        atomicAdd(&acc[3], nt);
        atomicAdd(&acc[4], hx);
    }
}

extern "C" int tsg_tiles_checksum(tsg_ctx *ctx, const tsg_dtiles *c, long long row_base, int jbase,
                                  tsg_csum *out) {
    memset(out, 0, sizeof(*out));
    if (row_base < 0 || (row_base & 15)) {
        tsg_set_error("tsg_tiles_checksum: row_base must be a non-negative multiple of 16");
        return TSG_ERR_ARG;
    }
    if (c->m <= 0) return TSG_OK;
    unsigned long long *acc;
    TSG_TRY(tsg_alloc_t(ctx, &acc, 5));
    int st = TSG_OK;
    if (hipMemsetAsync(acc, 0, 40, ctx->stream) != hipSuccess) {
        tsg_set_error("tsg_tiles_checksum: memset failed");
        st = TSG_ERR_HIP;
    }
    if (st == TSG_OK) {
        hipLaunchKernelGGL(k_checksum, dim3(tsg_div_up(c->m, 256)), dim3(256), 0, ctx->stream, c->m, c->tile_ptr,
                           c->tile_colidx, c->tile_nnz, c->csr_ptr, c->mask, c->csr_col, c->val, row_base, jbase,
                           acc);
        if (hipGetLastError() != hipSuccess) {
            tsg_set_error("tsg_tiles_checksum: launch failed");
            st = TSG_ERR_HIP;
        }
    }
    unsigned long long h[5] = {0, 0, 0, 0, 0};
    if (st == TSG_OK) st = tsg_d2h(ctx, h, acc, 40);
    if (st == TSG_OK && hipStreamSynchronize(ctx->stream) != hipSuccess) {
        tsg_set_error("tsg_tiles_checksum: synchronize failed");
        st = TSG_ERR_HIP;
    }
    tsg_free(ctx, acc);
    TSG_TRY(st);
    out->tiles = h[0];
    out->entries = h[1];
    out->nnz = (long long)h[2];
    out->numtile = (long long)h[3];
    out->entries_t = h[4];
    return TSG_OK;
}

// Selected rows of a view (row ids local to the view, any order) as CSR.
template <int PASS>
__global__ void __launch_bounds__(256)
k_rows_sel(int m, int nsel, const int *__restrict__ sel, const int *__restrict__ tile_ptr,
           const int *__restrict__ tile_colidx, const int *__restrict__ tile_nnz,
           const unsigned char *__restrict__ csr_ptr, const unsigned char *__restrict__ tcol,
           const double *__restrict__ tval, int *__restrict__ cnt_or_ptr, int *__restrict__ col,
           double *__restrict__ val, int jbase) {
    const int x = blockIdx.x * 256 + threadIdx.x;
    if (x >= nsel) return;
    const int i = sel[x];
    const int I = i >> 4, r = i & 15;
    const int rowlen = min(16, m - I * 16);
    const int t0 = tile_ptr[I], t1 = tile_ptr[I + 1];
    if (PASS == 0) {
        int c = 0;
        for (int t = t0; t < t1; t++) c += t2c_row_len(tile_nnz, csr_ptr, t, r, rowlen);
        cnt_or_ptr[x] = c;
    } else {
        int out = cnt_or_ptr[x];
        for (int t = t0; t < t1; t++) {
            const int k = t2c_row_len(tile_nnz, csr_ptr, t, r, rowlen);
            if (k <= 0) continue;
            const int s = tile_nnz[t] + csr_ptr[(long long)t * 16 + r];
            const int J16 = (tile_colidx[t] - jbase) * 16;
            for (int j = 0; j < k; j++) {
                col[out + j] = J16 + tcol[s + j];
                val[out + j] = tval[s + j];
            }
            out += k;
        }
    }
}

extern "C" int tsg_tiles_rows(tsg_ctx *ctx, const tsg_dtiles *c, int jbase, const int *rows, int nrows,
                              tsg_hcsr *out) {
    memset(out, 0, sizeof(*out));
    if (nrows < 0 || (nrows > 0 && !rows)) { tsg_set_error("tsg_tiles_rows: bad row list"); return TSG_ERR_ARG; }
    for (int x = 0; x < nrows; x++)
        if (rows[x] < 0 || rows[x] >= c->m) {
            tsg_set_error("tsg_tiles_rows: row %d outside [0, %d)", rows[x], c->m);
            return TSG_ERR_ARG;
        }
    out->m = nrows;
    out->n = c->n;
    out->rowptr = (int *)malloc(4 * ((size_t)nrows + 1));
    if (!out->rowptr) { tsg_set_error("tsg_tiles_rows: host allocation failed"); return TSG_ERR_NOMEM; }
    out->rowptr[0] = 0;
    if (nrows == 0) {
        out->colidx = (int *)malloc(4);
        out->val = (double *)malloc(8);
        return TSG_OK;
    }
    int *dsel = nullptr, *dptr = nullptr, *dcol = nullptr;
    double *dval = nullptr;
    long long nnz = 0;
    const dim3 grid(tsg_div_up(nrows, 256));
    int st = tsg_alloc_t(ctx, &dsel, (size_t)nrows);
    if (st == TSG_OK) st = tsg_alloc_t(ctx, &dptr, (size_t)nrows + 1);
    if (st == TSG_OK) st = tsg_h2d(ctx, dsel, rows, 4 * (size_t)nrows);
    if (st == TSG_OK) {
        hipLaunchKernelGGL(k_rows_sel<0>, grid, dim3(256), 0, ctx->stream, c->m, nrows, dsel, c->tile_ptr,
                           c->tile_colidx, c->tile_nnz, c->csr_ptr, c->csr_col, c->val, dptr, (int *)nullptr,
                           (double *)nullptr, jbase);
        if (hipGetLastError() != hipSuccess) { tsg_set_error("tsg_tiles_rows: launch failed"); st = TSG_ERR_HIP; }
    }
    if (st == TSG_OK) st = tsg_scan_i32(ctx, dptr, dptr, nrows, &nnz);
    if (st == TSG_OK) st = tsg_alloc_t(ctx, &dcol, (size_t)nnz + 1);
    if (st == TSG_OK) st = tsg_alloc_t(ctx, &dval, (size_t)nnz + 1);
    if (st == TSG_OK && nnz > 0) {
        hipLaunchKernelGGL(k_rows_sel<1>, grid, dim3(256), 0, ctx->stream, c->m, nrows, dsel, c->tile_ptr,
                           c->tile_colidx, c->tile_nnz, c->csr_ptr, c->csr_col, c->val, dptr, dcol, dval, jbase);
        if (hipGetLastError() != hipSuccess) { tsg_set_error("tsg_tiles_rows: launch failed"); st = TSG_ERR_HIP; }
    }
    if (st == TSG_OK) {
        out->nnz = (int)nnz;
        out->colidx = (int *)malloc(4 * (size_t)(nnz ? nnz : 1));
        out->val = (double *)malloc(8 * (size_t)(nnz ? nnz : 1));
        if (!out->colidx || !out->val) { tsg_set_error("tsg_tiles_rows: host allocation failed"); st = TSG_ERR_NOMEM; }
    }
    if (st == TSG_OK) st = tsg_d2h(ctx, out->rowptr, dptr, 4 * ((size_t)nrows + 1));
    if (st == TSG_OK && nnz > 0) st = tsg_d2h(ctx, out->colidx, dcol, 4 * (size_t)nnz);
    if (st == TSG_OK && nnz > 0) st = tsg_d2h(ctx, out->val, dval, 8 * (size_t)nnz);
    if (st == TSG_OK && hipStreamSynchronize(ctx->stream) != hipSuccess) {
        tsg_set_error("tsg_tiles_rows: synchronize failed");
        st = TSG_ERR_HIP;
    }
    tsg_free(ctx, dval);
    tsg_free(ctx, dcol);
    tsg_free(ctx, dptr);
    tsg_free(ctx, dsel);
    if (st != TSG_OK) tsg_hcsr_free(out);
    return st;
}

extern "C" int tsg_tiles_build_rowindex(tsg_ctx *ctx, tsg_dtiles *t) {
    if (t->rowx_ptr) return TSG_OK;
    tsg_dcsr d;
    TSG_TRY(tsg_tile2csr_view(ctx, t, 0, &d));
    t->rowx_ptr = d.rowptr;
    t->rowx_col = d.colidx;
    t->rowx_val = d.val;
    return TSG_OK;
}

extern "C" void tsg_tiles_free(tsg_ctx *ctx, tsg_dtiles *t) {
    if (!t) return;
    void *ps[] = {t->tile_ptr, t->tile_colidx, t->tile_rowidx, t->tile_nnz, t->csr_ptr, t->csr_col,
                  t->val, t->mask, t->csc_ptr, t->csc_rowidx, t->csc_tileid, t->rowx_ptr, t->rowx_col,
                  t->rowx_val};
    for (void *p : ps) tsg_free(ctx, p);
    memset(t, 0, sizeof(*t));
}

template <typename T>
static int dl(tsg_ctx *ctx, T **dst, const T *src, size_t n) {
    *dst = nullptr;
    if (!src) return TSG_OK;
    *dst = (T *)malloc((n ? n : 1) * sizeof(T));
    if (!*dst) { tsg_set_error("host allocation failed"); return TSG_ERR_NOMEM; }
    if (n) TSG_HIP(hipMemcpyAsync(*dst, src, n * sizeof(T), hipMemcpyDeviceToHost, ctx->stream));
    return TSG_OK;
}

extern "C" int tsg_tiles_download(tsg_ctx *ctx, const tsg_dtiles *d, tsg_htiles *h) {
    memset(h, 0, sizeof(*h));
    h->m = d->m; h->n = d->n; h->tilem = d->tilem; h->tilen = d->tilen;
    h->numtile = d->numtile; h->nnz = d->nnz;
    size_t nt = (size_t)d->numtile;
    TSG_TRY(dl(ctx, &h->tile_ptr, d->tile_ptr, (size_t)d->tilem + 1));
    TSG_TRY(dl(ctx, &h->tile_colidx, d->tile_colidx, nt));
    TSG_TRY(dl(ctx, &h->tile_rowidx, d->tile_rowidx, nt));
    TSG_TRY(dl(ctx, &h->tile_nnz, d->tile_nnz, nt + 1));
    TSG_TRY(dl(ctx, &h->csr_ptr, d->csr_ptr, nt * 16));
    TSG_TRY(dl(ctx, &h->csr_col, d->csr_col, (size_t)d->nnz));
    TSG_TRY(dl(ctx, &h->val, d->val, (size_t)d->nnz));
    TSG_TRY(dl(ctx, &h->mask, d->mask, nt * 16));
    TSG_TRY(dl(ctx, &h->csc_ptr, d->csc_ptr, (size_t)d->tilen + 1));
    TSG_TRY(dl(ctx, &h->csc_rowidx, d->csc_rowidx, nt));
    TSG_TRY(dl(ctx, &h->csc_tileid, d->csc_tileid, nt));
    TSG_HIP(hipStreamSynchronize(ctx->stream));
    return TSG_OK;
}

extern "C" void tsg_htiles_free(tsg_htiles *h) {
    if (!h) return;
    void *ps[] = {h->tile_ptr, h->tile_colidx, h->tile_rowidx, h->tile_nnz, h->csr_ptr, h->csr_col,
                  h->val, h->mask, h->csc_ptr, h->csc_rowidx, h->csc_tileid};
    for (void *p : ps) free(p);
    memset(h, 0, sizeof(*h));
}

// ---------------------------------------------------------------- transpose
// The row of every entry, VAL_BLOCK entries per block: each row start of the
// block marks its entry in LDS and the marks' running maximum is the row.
// Entry parallel, so a hub row is not one lane's loop (R-MAT scale 18: 848 ->
// 32 us).
__global__ void __launch_bounds__(256)
k_row_of_entry(const int *__restrict__ rowptr, int m, int nnz, int *__restrict__ rowid) {
    __shared__ int s_row[VAL_BLOCK];  // row + 1 at a row's first entry
    __shared__ int s_lo[2], s_max[4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int e0 = blockIdx.x * VAL_BLOCK, ne = min(VAL_BLOCK, nnz - e0);
    for (int i = tid; i < VAL_BLOCK; i += 256) s_row[i] = 0;
    if (wave < 2) {
        const int i = wave_first_ge(rowptr, 0, m + 1, wave ? e0 + ne : e0);
        if (lane == 0) s_lo[wave] = i;
    }
    __syncthreads();
    const int lo = s_lo[0], hi = s_lo[1];  // rows starting in the block
    if (hi - lo > VAL_MARK_ROWS) {         // mostly empty rows: a search per entry
        for (int x = tid; x < ne; x += 256) rowid[e0 + x] = first_ge(rowptr, 0, m + 1, e0 + x + 1) - 1;
        return;  // block-uniform
    }
    // of rows starting at one entry the last has it
    for (int i = lo + tid; i < hi; i += 256) atomicMax(&s_row[rowptr[i] - e0], i + 1);
    __syncthreads();
    int mx = 0;
    for (int k = 0; k < VAL_BLOCK / 256; k++) mx = max(mx, s_row[wave * (VAL_BLOCK / 4) + 64 * k + lane]);
    mx = tsg_wave_max(mx);
    if (lane == 0) s_max[wave] = mx;
    __syncthreads();
    int last = lo;  // row lo - 1 holds the entries before the block's first row start
    for (int w = 0; w < wave; w++) last = max(last, s_max[w]);
    for (int k = 0; k < VAL_BLOCK / 256; k++) {
        const int x = wave * (VAL_BLOCK / 4) + 64 * k + lane;
        const int r = max(last, tsg_wave_incl_max_dpp(s_row[x]));
        last = __builtin_amdgcn_readlane(r, 63);
        if (x < ne) rowid[e0 + x] = r - 1;
    }
}

// Stable CSR -> CSC (src/utils.h:158-195): a stable sort of the entries by
// column keeps rows ascending inside every column.
extern "C" int tsg_dcsr_transpose(tsg_ctx *ctx, const tsg_dcsr *a, tsg_dcsr *at) {
    memset(at, 0, sizeof(*at));
    TSG_TRY(tsg_validate_csr(ctx, a));
    at->m = a->n;
    at->n = a->m;
    at->nnz = a->nnz;
    const long long nnz = a->nnz;
    TSG_TRY(tsg_alloc_t(ctx, &at->rowptr, (size_t)a->n + 1));
    TSG_TRY(tsg_alloc_t(ctx, &at->colidx, (size_t)nnz + 1));
    TSG_TRY(tsg_alloc_t(ctx, &at->val, (size_t)nnz + 1));
    unsigned *keys = nullptr;
    if (nnz > 0) {
        int *perm, *rowid;
        TSG_TRY(tsg_alloc_t(ctx, &keys, (size_t)nnz));
        TSG_TRY(tsg_alloc_t(ctx, &perm, (size_t)nnz));
        TSG_TRY(tsg_alloc_t(ctx, &rowid, (size_t)nnz));
        const unsigned g = tsg_div_up(nnz, 256);
        hipLaunchKernelGGL(k_sort_input, dim3(g), dim3(256), 0, ctx->stream, a->colidx, nnz, keys, perm);
        hipLaunchKernelGGL(k_row_of_entry, dim3(tsg_div_up(nnz, VAL_BLOCK)), dim3(256), 0, ctx->stream, a->rowptr, a->m,
                           a->nnz, rowid);
        TSG_LAUNCH_CHECK();
        TSG_TRY(tsg_sort_pairs_u32(ctx, keys, perm, nnz, bits_for(a->n)));
        hipLaunchKernelGGL(k_gather_entries, dim3(g), dim3(256), 0, ctx->stream, rowid, a->val, perm, nnz, at->colidx,
                           at->val);
        TSG_LAUNCH_CHECK();
        tsg_free(ctx, perm);
        tsg_free(ctx, rowid);
    }
    hipLaunchKernelGGL(k_ptr_of_sorted, dim3(tsg_div_up((long long)a->n + 1, 256)), dim3(256), 0, ctx->stream,
                       (const unsigned *)keys, nnz, a->n, at->rowptr);
    TSG_LAUNCH_CHECK();
    tsg_free(ctx, keys);
    return TSG_OK;
}

// ---------------------------------------------------------------- nnzCub
__global__ void __launch_bounds__(256)
k_nnzcub(const int *__restrict__ colA, long long nnzA, const int *__restrict__ rowptrB,
         unsigned long long *__restrict__ out) {
    unsigned long long s = 0;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < nnzA; e += (long long)gridDim.x * 256) {
        const int k = colA[e];
        s += (unsigned long long)(rowptrB[k + 1] - rowptrB[k]);
    }
    s = tsg_wave_sum(s);
    if ((threadIdx.x & 63) == 0) atomicAdd(out, s);
}

extern "C" int tsg_dcsr_nnzcub(tsg_ctx *ctx, const tsg_dcsr *a, const tsg_dcsr *b, unsigned long long *out) {
    if (a->n != b->m) { tsg_set_error("nnzcub: inner dimensions differ (%d vs %d)", a->n, b->m); return TSG_ERR_ARG; }
    TSG_TRY(tsg_validate_csr(ctx, a));
    TSG_TRY(tsg_validate_csr(ctx, b));
    void *scr;
    TSG_TRY(tsg_scratch(ctx, 64, &scr));
    TSG_HIP(hipMemsetAsync(scr, 0, 8, ctx->stream));
    if (a->nnz > 0) {
        unsigned nb = (unsigned)std::min<long long>(tsg_div_up(a->nnz, 256), 8192);
        hipLaunchKernelGGL(k_nnzcub, dim3(nb), dim3(256), 0, ctx->stream, a->colidx, (long long)a->nnz, b->rowptr,
                           (unsigned long long *)scr);
        TSG_LAUNCH_CHECK();
    }
    long long t;
    TSG_TRY(tsg_read_scalar_i64(ctx, scr, 1, &t));
    *out = (unsigned long long)t;
    return TSG_OK;
}

// ---------------------------------------------------------------- host-layer utilities
extern "C" int tsg_dmalloc(tsg_ctx *ctx, void **p, size_t bytes) { return tsg_alloc(ctx, p, bytes); }
extern "C" void tsg_dfree(tsg_ctx *ctx, void *p) { tsg_free(ctx, p); }
extern "C" int tsg_h2d(tsg_ctx *ctx, void *d, const void *h, size_t bytes) {
    if (bytes) TSG_HIP(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, ctx->stream));
    TSG_HIP(hipStreamSynchronize(ctx->stream));
    return TSG_OK;
}
extern "C" int tsg_d2h(tsg_ctx *ctx, void *h, const void *d, size_t bytes) {
    if (bytes) TSG_HIP(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, ctx->stream));
    TSG_HIP(hipStreamSynchronize(ctx->stream));
    return TSG_OK;
}
extern "C" int tsg_d_iota(tsg_ctx *ctx, int *d, long long n) {
    if (n > 0) {
        hipLaunchKernelGGL(k_iota, dim3(tsg_div_up(n, 256)), dim3(256), 0, ctx->stream, d, n);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

// (row << 4) | col in-tile bytes, the A-operand column layout of
// csr2tile_row_major (src/csr2tile.h:185).  One thread per (tile, row).
__global__ void __launch_bounds__(256)
k_pack_cols(long long nrows16, const int *__restrict__ tile_nnz, const unsigned char *__restrict__ ptr16,
            const unsigned char *__restrict__ col, unsigned char *__restrict__ out) {
    const long long x = (long long)blockIdx.x * 256 + threadIdx.x;
    if (x >= nrows16) return;
    const long long t = x >> 4;
    const int r = (int)(x & 15);
    const int tn = tile_nnz[t + 1] - tile_nnz[t];
    const int s = ptr16[x], e = r == 15 ? tn : ptr16[x + 1];
    for (int j = s; j < e; j++) out[tile_nnz[t] + j] = (unsigned char)((r << 4) | col[tile_nnz[t] + j]);
}

extern "C" int tsg_tiles_packed_cols(tsg_ctx *ctx, const tsg_dtiles *t, unsigned char *d_out) {
    const long long n16 = (long long)t->numtile * 16;
    if (n16 > 0) {
        hipLaunchKernelGGL(k_pack_cols, dim3(tsg_div_up(n16, 256)), dim3(256), 0, ctx->stream, n16, t->tile_nnz,
                           t->csr_ptr, t->csr_col, d_out);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

// Tile data re-ordered into CSC tile order (the B-operand layout of
// csr2tile_col_major, src/csr2tile.h:327-477).
__global__ void __launch_bounds__(256)
k_csc_meta(int nt, const int *__restrict__ cscid, const int *__restrict__ tile_nnz, const unsigned char *__restrict__ ptr16,
           const unsigned short *__restrict__ mask, unsigned char *__restrict__ optr16, unsigned short *__restrict__ omask,
           int *__restrict__ ocnt) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= nt) return;
    const int s = cscid[p];
    *reinterpret_cast<uint4 *>(optr16 + (long long)p * 16) = *reinterpret_cast<const uint4 *>(ptr16 + (long long)s * 16);
    const uint4 *ms = reinterpret_cast<const uint4 *>(mask + (long long)s * 16);
    uint4 *md = reinterpret_cast<uint4 *>(omask + (long long)p * 16);
    md[0] = ms[0];
    md[1] = ms[1];
    ocnt[p] = tile_nnz[s + 1] - tile_nnz[s];
}
__global__ void __launch_bounds__(256)
k_csc_data(int nt, const int *__restrict__ cscid, const int *__restrict__ tile_nnz, const int *__restrict__ onnz,
           const unsigned char *__restrict__ col, const double *__restrict__ val, unsigned char *__restrict__ ocol,
           double *__restrict__ oval) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= nt) return;
    const int s = cscid[p];
    const int src = tile_nnz[s], dst = onnz[p], n = onnz[p + 1] - dst;
    for (int j = 0; j < n; j++) {
        ocol[dst + j] = col[src + j];
        oval[dst + j] = val[src + j];
    }
}

extern "C" int tsg_tiles_csc_order(tsg_ctx *ctx, tsg_dtiles *t, tsg_dtiles *o) {
    memset(o, 0, sizeof(*o));
    TSG_TRY(tsg_tiles_build_csc(ctx, t));
    *o = *t;
    const long long nt = t->numtile;
    o->tile_ptr = o->tile_colidx = o->tile_rowidx = o->tile_nnz = nullptr;
    o->csr_ptr = o->csr_col = nullptr;
    o->val = nullptr;
    o->mask = nullptr;
    o->csc_ptr = o->csc_rowidx = o->csc_tileid = nullptr;
    o->rowx_ptr = o->rowx_col = nullptr;
    o->rowx_val = nullptr;
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_ptr, (size_t)t->tilem + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_colidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_rowidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csc_ptr, (size_t)t->tilen + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csc_rowidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csc_tileid, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_nnz, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csr_ptr, (size_t)nt * 16 + 16));
    TSG_TRY(tsg_alloc_t(ctx, &o->mask, (size_t)nt * 16 + 16));
    TSG_TRY(tsg_alloc_t(ctx, &o->csr_col, (size_t)t->nnz + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->val, (size_t)t->nnz + 1));
    hipStream_t s = ctx->stream;
    TSG_HIP(hipMemcpyAsync(o->tile_ptr, t->tile_ptr, ((size_t)t->tilem + 1) * 4, hipMemcpyDeviceToDevice, s));
    TSG_HIP(hipMemcpyAsync(o->csc_ptr, t->csc_ptr, ((size_t)t->tilen + 1) * 4, hipMemcpyDeviceToDevice, s));
    if (nt > 0) {
        TSG_HIP(hipMemcpyAsync(o->tile_colidx, t->tile_colidx, nt * 4, hipMemcpyDeviceToDevice, s));
        TSG_HIP(hipMemcpyAsync(o->tile_rowidx, t->tile_rowidx, nt * 4, hipMemcpyDeviceToDevice, s));
        TSG_HIP(hipMemcpyAsync(o->csc_rowidx, t->csc_rowidx, nt * 4, hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(k_iota, dim3(tsg_div_up(nt, 256)), dim3(256), 0, s, o->csc_tileid, nt);
        hipLaunchKernelGGL(k_csc_meta, dim3(tsg_div_up(nt, 256)), dim3(256), 0, s, (int)nt, t->csc_tileid, t->tile_nnz,
                           t->csr_ptr, t->mask, o->csr_ptr, o->mask, o->tile_nnz);
        TSG_LAUNCH_CHECK();
    }
    TSG_TRY(tsg_scan_i32(ctx, o->tile_nnz, o->tile_nnz, nt, nullptr));
    if (nt > 0) {
        hipLaunchKernelGGL(k_csc_data, dim3(tsg_div_up(nt, 256)), dim3(256), 0, s, (int)nt, t->csc_tileid, t->tile_nnz,
                           o->tile_nnz, t->csr_col, t->val, o->csr_col, o->val);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

// Inverse of tsg_tiles_csc_order: tile data given in CSC tile order (the B
// layout csr2tile_col_major hands to the reference's tilespgemm) is moved to
// row-major tile order, and csc_tileid maps each CSC position to its
// row-major tile.  One thread per tile column walks its CSC entries and
// binary-searches each tile in its tile-row's (sorted) column list.
__global__ void __launch_bounds__(256)
k_csc_to_rm(int tilen, const int *__restrict__ csc_ptr, const int *__restrict__ csc_row,
            const int *__restrict__ tile_ptr, const int *__restrict__ tile_col, const int *__restrict__ nnz_csc,
            int *__restrict__ rm, int *__restrict__ cnt_rm, int *__restrict__ bad) {
    const int J = blockIdx.x * 256 + threadIdx.x;
    if (J >= tilen) return;
    for (int p = csc_ptr[J]; p < csc_ptr[J + 1]; p++) {
        const int K = csc_row[p];
        const int s = tile_ptr[K], len = tile_ptr[K + 1] - s;
        int lo = 0, hi = len - 1, f = -1;
        while (lo <= hi) {
            const int mid = (lo + hi) >> 1, v = tile_col[s + mid];
            if (v == J) { f = mid; break; }
            if (v < J) lo = mid + 1; else hi = mid - 1;
        }
        if (f < 0) { atomicOr(bad, 1); rm[p] = 0; continue; }
        rm[p] = s + f;
        cnt_rm[s + f] = nnz_csc[p + 1] - nnz_csc[p];
    }
}
__global__ void __launch_bounds__(256)
k_scatter_meta(int nt, const int *__restrict__ rm, const unsigned char *__restrict__ ptr16,
               const unsigned short *__restrict__ mask, unsigned char *__restrict__ optr16,
               unsigned short *__restrict__ omask) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= nt) return;
    const long long d = rm[p];
    *reinterpret_cast<uint4 *>(optr16 + d * 16) = *reinterpret_cast<const uint4 *>(ptr16 + (long long)p * 16);
    const uint4 *ms = reinterpret_cast<const uint4 *>(mask + (long long)p * 16);
    uint4 *md = reinterpret_cast<uint4 *>(omask + d * 16);
    md[0] = ms[0];
    md[1] = ms[1];
}
__global__ void __launch_bounds__(256)
k_scatter_data(int nt, const int *__restrict__ rm, const int *__restrict__ nnz_csc, const int *__restrict__ nnz_rm,
               const unsigned char *__restrict__ col, const double *__restrict__ val, unsigned char *__restrict__ ocol,
               double *__restrict__ oval) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= nt) return;
    const int src = nnz_csc[p], n = nnz_csc[p + 1] - src, dst = nnz_rm[rm[p]];
    for (int j = 0; j < n; j++) {
        if (ocol) ocol[dst + j] = col[src + j];
        oval[dst + j] = val[src + j];
    }
}

extern "C" int tsg_tiles_from_csc_order(tsg_ctx *ctx, const tsg_dtiles *in, tsg_dtiles *o) {
    memset(o, 0, sizeof(*o));
    if (!in->csc_ptr || !in->csc_rowidx || !in->tile_ptr || !in->tile_colidx) {
        tsg_set_error("tsg_tiles_from_csc_order: needs the row-major and the CSC tile index");
        return TSG_ERR_ARG;
    }
    const long long nt = in->numtile;
    o->m = in->m; o->n = in->n; o->tilem = in->tilem; o->tilen = in->tilen;
    o->numtile = in->numtile; o->nnz = in->nnz;
    hipStream_t s = ctx->stream;
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_ptr, (size_t)in->tilem + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_colidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_rowidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csc_ptr, (size_t)in->tilen + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csc_rowidx, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csc_tileid, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->tile_nnz, (size_t)nt + 1));
    TSG_TRY(tsg_alloc_t(ctx, &o->csr_ptr, (size_t)nt * 16 + 16));
    TSG_TRY(tsg_alloc_t(ctx, &o->mask, (size_t)nt * 16 + 16));
    TSG_TRY(tsg_alloc_t(ctx, &o->val, (size_t)in->nnz + 1));
    if (in->csr_col) TSG_TRY(tsg_alloc_t(ctx, &o->csr_col, (size_t)in->nnz + 1));
    TSG_HIP(hipMemcpyAsync(o->tile_ptr, in->tile_ptr, ((size_t)in->tilem + 1) * 4, hipMemcpyDeviceToDevice, s));
    TSG_HIP(hipMemcpyAsync(o->csc_ptr, in->csc_ptr, ((size_t)in->tilen + 1) * 4, hipMemcpyDeviceToDevice, s));
    void *scr;
    TSG_TRY(tsg_scratch(ctx, 64, &scr));
    TSG_HIP(hipMemsetAsync(scr, 0, 4, s));
    if (nt > 0) {
        TSG_HIP(hipMemcpyAsync(o->tile_colidx, in->tile_colidx, nt * 4, hipMemcpyDeviceToDevice, s));
        TSG_HIP(hipMemcpyAsync(o->csc_rowidx, in->csc_rowidx, nt * 4, hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(k_csc_to_rm, dim3(tsg_div_up(in->tilen, 256)), dim3(256), 0, s, in->tilen, in->csc_ptr,
                           in->csc_rowidx, in->tile_ptr, in->tile_colidx, in->tile_nnz, o->csc_tileid, o->tile_nnz,
                           (int *)scr);
        TSG_LAUNCH_CHECK();
    }
    long long bad = 0;
    TSG_TRY(tsg_read_scalar_i64(ctx, scr, 0, &bad));
    if (bad) { tsg_set_error("CSC tile index does not match the row-major tile index"); return TSG_ERR_ARG; }
    TSG_TRY(tsg_scan_i32(ctx, o->tile_nnz, o->tile_nnz, nt, nullptr));
    if (nt > 0) {
        // tile row of every row-major tile
        hipLaunchKernelGGL(k_scatter_i32, dim3(tsg_div_up(nt, 256)), dim3(256), 0, s, in->csc_rowidx, o->csc_tileid, nt,
                           o->tile_rowidx);
        hipLaunchKernelGGL(k_scatter_meta, dim3(tsg_div_up(nt, 256)), dim3(256), 0, s, (int)nt, o->csc_tileid,
                           in->csr_ptr, in->mask, o->csr_ptr, o->mask);
        hipLaunchKernelGGL(k_scatter_data, dim3(tsg_div_up(nt, 256)), dim3(256), 0, s, (int)nt, o->csc_tileid,
                           in->tile_nnz, o->tile_nnz, in->csr_col, in->val, o->csr_col, o->val);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}
