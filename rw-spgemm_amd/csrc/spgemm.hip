// spgemm.hip -- the TileSpGEMM pipeline on gfx950 (wave64, LDS, FP64 FMA).
//
// Step 1 (tile-level symbolic, src/tilespgemm-cuda.h:257-369 and the nsparse
//   hash path src/spgemm_nsparse_kernel.h:138-1511): for each A tile-row I the
//   set of C tile columns  U_{K in A(I,:)} B(K,:)  -- one wave per tile-row,
//   the (K, J) candidates flattened across the 64 lanes and OR-ed into a
//   windowed LDS bitmap; count pass, device scan, then a fill pass emitting
//   the sorted tile columns.  Covers every tilen (no SPA/hash split).
// Step 2 (16x16 bitmask symbolic, src/tilespgemm-cuda.h:371-755):
//   k_step2_rows, one block per C tile-row, visits every (A tile, B tile)
//   pair of the row once (no intersection search) and ORs the pair's
//   boolean product rows into the C tile masks held in LDS; popcounts give
//   the u8 row offsets and tile nnz; a tile-row with more C tiles than LDS
//   holds is cut into segments.  With row indices, hypersparse and hub
//   tile-rows go entry by entry instead (k_step2_elem, C tiles in a hash;
//   k_step2_dense, the tile-row's columns as bits).  k_step2_tiles (one C tile
//   per 16-lane group, pairs from a sorted-list intersection, 64-bit ballots
//   to keep them in K order) takes all of C on request (force_tile_parallel).
// Step 3 (numeric, src/tilespgemm-cuda.h:1505-2608): k_step3_lines, one block
//   per C tile-row, adds B rows line by line (both row indices needed);
//   tile-rows it does not take, and all without them, go by k_step3_rows if
//   they fit it: one block per C tile-row accumulates the row's C values in
//   LDS in their final order; each C row belongs to one wave, which takes its tasks in
//   ascending K.  A tile K with several entries has A tile K and B tile-row
//   K staged into LDS (software pipelined) and the (B tile, A row) tasks
//   that meet nonempty B rows run compacted per wave; a single-entry A tile
//   is handled by its row's wave from registers.  The rest, hypersparse and
//   hub rows mostly: k_step3_flat and k_step3_heavy with both row indices,
//   k_step3_elem with B's alone, else k_step3 (one C tile per
//   16-lane group, lane r owns tile row r, dense or compact LDS row
//   accumulator).  No floating-point atomics: every C entry receives its
//   products in ascending inner index k, the order of the serial SPA
//   reference, so results are deterministic and bit-identical to it.  (The
//   reference uses FP64 atomicAdd, src/tilespgemm-cuda.h:1670.)
#include <string.h>

#include <mutex>
#include <type_traits>

#include "tsg_internal.h"

#define S1_WAVES 4
#define S23_WAVES 4
#define TILES_PER_WAVE 4
#define S2_KINDS 4  // step-2 kernels (step2_kind)

extern "C" void tsg_tune_default(tsg_tune *t) {
    memset(t, 0, sizeof(*t));
    t->dense_acc_min_nnz = 64;
    t->s1_window_words = 0;
}

// ------------------------------------------------------------------ B tile-row bitmaps
// For step 1: the tile columns of B tile-row K as a bitmap of nw 32-bit
// words from absolute word F (bit b of word w <-> tile column 32 (F + w) + b),
// kept at bits + off when it is at most about twice the size of the row's
// column list (nw <= 2 * tiles + 2); desc[K] = {off, F, nw, 0} with nw = 0
// for a row that is empty or not kept.  off = 2 * Bptr[K] + 2 * K bounds
// every row's room without a scan.  Two launches (graph-capturable, every
// word of a kept row written once, no memset): k_brow_desc, one lane per
// tile-row, then k_brow_fill, one lane per B tile, so a hub tile-row's
// words are spread over as many waves as it has tiles.  With longest (and B's
// row pointers), longest[K] = entries of the longest row of tile-row K.
// Tile-row K's descriptor (and longest[K]); returns whether it is kept.
__device__ __forceinline__ bool brow_desc(const int *__restrict__ Bptr, const int *__restrict__ Bcol, int K, int4 *desc,
                                          const int *__restrict__ Browp, int m, int *longest) {
    const int b0 = Bptr[K], n = Bptr[K + 1] - b0;
    int F = 0, nw = 0;
    if (n > 0) {
        F = Bcol[b0] >> 5;
        nw = (Bcol[b0 + n - 1] >> 5) - F + 1;
        if (nw > 2 * n + 2) nw = 0;
    }
    desc[K] = make_int4(2 * b0 + 2 * K, F, nw, 0);
    if (longest) {
        int p = Browp[16 * K], mx = 0;
        if (16 * K + 16 <= m) {
            int q[16];
#pragma unroll
            for (int r = 0; r < 16; r++) q[r] = Browp[16 * K + 1 + r];
#pragma unroll
            for (int r = 0; r < 16; r++) mx = max(mx, q[r] - (r ? q[r - 1] : p));
        } else {
            for (int r = 16 * K + 1; r <= m; r++) {
                mx = max(mx, Browp[r] - p);
                p = Browp[r];
            }
        }
        longest[K] = mx;
    }
    return nw > 0;
}
__global__ void __launch_bounds__(256)
k_brow_desc(const int *__restrict__ Bptr, const int *__restrict__ Bcol, int tilem, int4 *__restrict__ desc,
            int *__restrict__ any, const int *__restrict__ Browp, int m, int *__restrict__ longest) {
    const int K = blockIdx.x * 256 + threadIdx.x;
    const bool kept = K < tilem && brow_desc(Bptr, Bcol, K, desc, Browp, m, longest);
    // any (may be NULL, zeroed beforehand): set when some row is kept; the
    // same value from every writer, and no store once it reads 1
    if (any && __ballot(kept) && (threadIdx.x & 63) == 0 && *(volatile int *)any == 0) *(volatile int *)any = 1;
}

// A run is the tiles of one kept row in one bitmap word (consecutive in the
// row-major tile order).  Its last tile's lane writes the word (the run's
// bits OR-ed across lanes, plus the run's tiles before the wave's first,
// at most 31) and zeroes the empty words up to the row's next run.
// t: the lane's tile, whole waves (desc is not restrict: k_brow_one writes it)
__device__ __forceinline__ void brow_fill(const int *__restrict__ Brow, const int *__restrict__ Bcol, long long numtile,
                                          const int4 *desc, unsigned *__restrict__ bits, long long t) {
    const int lane = threadIdx.x & 63;
    const long long t0 = t - lane;  // the wave's first tile
    if (t0 >= numtile) return;
    const bool valid = t < numtile;
    int K = -1, w = -1, col = 0;
    int4 d = make_int4(0, 0, 0, 0);
    if (valid) {
        K = Brow[t];
        d = desc[K];
        col = Bcol[t];
        if (d.z > 0) w = (col >> 5) - d.y;
    }
    const bool kept = valid && d.z > 0;
    // the next tile's row and word (lane 63: loaded)
    int Kn = __shfl_down(K, 1, 64), wn = __shfl_down(w, 1, 64), cn = __shfl_down(col, 1, 64);
    if (lane == 63) {
        Kn = -1;
        if (t + 1 < numtile) {
            Kn = Brow[t + 1];
            cn = Bcol[t + 1];
            wn = Kn == K ? (cn >> 5) - d.y : -1;
        }
    }
    const bool last = kept && !(Kn == K && wn == w);
    // inclusive OR over the run's lanes up to this one
    unsigned v = kept ? 1u << (col & 31) : 0u;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned vv = __shfl_up(v, o, 64);
        const int kk = __shfl_up(K, o, 64), ww = __shfl_up(w, o, 64);
        if (lane >= o && kk == K && ww == w) v |= vv;
    }
    // lane 0's run, read with every lane active (a shuffle inside the branch
    // below would not see lane 0 unless it is a run's last lane too)
    const int K0 = __shfl(K, 0, 64), w0 = __shfl(w, 0, 64);
    if (last) {
        if (K0 == K && w0 == w)  // the run began before this wave
            for (long long u = t0 - 1; u >= 0 && Brow[u] == K; u--) {
                const int c = Bcol[u];
                if ((c >> 5) - d.y != w) break;
                v |= 1u << (c & 31);
            }
        unsigned *row = bits + d.x;
        row[w] = v;
        const int wend = Kn == K ? wn : d.z;  // the row's next run, or its end
        for (int g = w + 1; g < wend; g++) row[g] = 0u;
    }
}

__global__ void __launch_bounds__(256)
k_brow_fill(const int *__restrict__ Brow, const int *__restrict__ Bcol, long long numtile,
            const int4 *__restrict__ desc, unsigned *__restrict__ bits, const int *__restrict__ any) {
    if (any && *any == 0) return;  // no row kept (k_brow_desc's flag, when given)
    brow_fill(Brow, Bcol, numtile, desc, bits, (long long)blockIdx.x * 256 + threadIdx.x);
}

// Both for a small B in one block, which also clears the SCR_WORDS words of scr
// (may be NULL) and sets any: a launch takes about 4 us of a small product, more than
// its kernels' work.  5-point 64^2 A^2 in 8 launches instead of 13 (this one, k_row_stats_one,
// the class maxima by k_row_class's last block): 84 -> 77 us.
// ER 1000 (4 per row, 2,500 tiles) 103 -> 99 us, but with 3,900 tiles 110 -> 114.
#define BROW_ONE 2560  // tiles of a B that one block takes
#define BROW_ONE_ROWS 1024  // and tile-rows
#define SCR_WORDS 32
__global__ void __launch_bounds__(1024)
k_brow_one(const int *__restrict__ Bptr, const int *__restrict__ Brow, const int *__restrict__ Bcol, int tilem,
           int numtile, int4 *desc, unsigned *__restrict__ bits, int *scr, int *any, const int *__restrict__ Browp, int m,
           int *__restrict__ longest) {
    __shared__ int s_any;
    if (threadIdx.x == 0) s_any = 0;
    if (scr && threadIdx.x < SCR_WORDS && scr + threadIdx.x != any) scr[threadIdx.x] = 0;
    __syncthreads();
    bool kept = false;
    for (int K = threadIdx.x; K < tilem; K += 1024) kept |= brow_desc(Bptr, Bcol, K, desc, Browp, m, longest);
    if (__ballot(kept) && (threadIdx.x & 63) == 0) s_any = 1;
    __syncthreads();  // the block's descriptors are written
    if (any && threadIdx.x == 0) *any = s_any;
    if (!s_any) return;
    for (int t = threadIdx.x; t - (int)(threadIdx.x & 63) < numtile; t += 1024) brow_fill(Brow, Bcol, numtile, desc, bits, t);
}

// ------------------------------------------------------------------ step 1
// Bdesc / Bbits (may be NULL): B tile-rows kept as bitmaps (k_brow_desc,
// k_brow_fill).  Their candidates are not enumerated: each lane ORs the
// bitmap words over its own window words, with no search and no LDS
// atomics.  Bany (may be NULL) is k_brow_desc's flag: when no row was kept,
// the descriptors are not read at all.
template <bool FILL, int BMW>
__global__ void __launch_bounds__(64 * S1_WAVES)
k_step1(const int *__restrict__ Aptr, const int *__restrict__ Acol, int tilem,
        const int *__restrict__ Bptr, const int *__restrict__ Bcol, const int4 *__restrict__ Bdesc,
        const unsigned *__restrict__ Bbits, const int *__restrict__ Bany, int *__restrict__ Cptr_or_cnt,
        int *__restrict__ Ccol, int *__restrict__ Crow, unsigned *__restrict__ bmstore, int *__restrict__ rowspan) {
    // rowspan (may be NULL): count pass, each row's C tile-column span; fill
    // pass, S2_KINDS counters to clear for k_seg2_fill
    if (FILL && rowspan && blockIdx.x == 0 && threadIdx.x < S2_KINDS) rowspan[threadIdx.x] = 0;
    __shared__ unsigned s_bm[S1_WAVES][BMW];
    __shared__ int s_pre[S1_WAVES][64];
    __shared__ int s_b0[S1_WAVES][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int I = blockIdx.x * S1_WAVES + wave;
    if (I >= tilem) return;
    unsigned *bm = s_bm[wave];
    int *pre = s_pre[wave], *pb0 = s_b0[wave];
    const int a0 = Aptr[I], a1 = Aptr[I + 1];
    if (Bany && *Bany == 0) Bdesc = nullptr;  // wave-uniform

    // range of candidate tile columns: B rows are sorted
    int jmin = 0x7fffffff, jmax = -1;
    for (int p = a0 + lane; p < a1; p += 64) {
        const int K = Acol[p];
        const int b0 = Bptr[K], b1 = Bptr[K + 1];
        if (b1 > b0) {
            jmin = min(jmin, Bcol[b0]);
            jmax = max(jmax, Bcol[b1 - 1]);
        }
    }
    jmin = tsg_wave_min(jmin);
    jmax = tsg_wave_max(jmax);
    // windows start on a word boundary of absolute tile columns (the words
    // of B's tile-row bitmaps)
    const int jb = jmin & ~31;

    // a row spanning 2..64 windows (a periodic grid's boundary rows) first
    // finds the windows its candidates hit and visits only those
    constexpr int WSH = __builtin_ctz(32 * BMW);  // log2 of the columns per window
    unsigned long long wmask = ~0ull;
    if (jmax >= jmin && ((jmax - jb) >> WSH) >= 1 && ((jmax - jb) >> WSH) < 64) {
        unsigned wlo = 0u, whi = 0u;
        for (int c0 = a0; c0 < a1; c0 += 64) {
            const int p = c0 + lane;
            int b0 = 0, len = 0;
            if (p < a1) {
                const int K = Acol[p];
                b0 = Bptr[K];
                len = Bptr[K + 1] - b0;
                if (Bdesc) {
                    const int4 d = Bdesc[K];
                    if (d.z > 0) {  // a kept row marks the windows its words span
                        len = 0;
                        const int i0 = (max(d.y << 5, jb) - jb) >> WSH;
                        const int i1 = (min(((d.y + d.z) << 5) - 1, jmax) - jb) >> WSH;
                        const unsigned long long m = (i1 >= 63 ? ~0ull : (2ull << i1) - 1) & ~((1ull << i0) - 1);
                        wlo |= (unsigned)m;
                        whi |= (unsigned)(m >> 32);
                    }
                }
            }
            const int incl = tsg_wave_incl_scan(len);
            const int tot = __shfl(incl, 63, 64);
            pre[lane] = incl - len;
            pb0[lane] = b0;
            tsg_wave_sync();
            for (int c = lane; c < tot; c += 64) {
                int lo = 0;
#pragma unroll
                for (int st = 32; st > 0; st >>= 1)
                    if (pre[lo + st] <= c) lo += st;
                const int wi = (Bcol[pb0[lo] + (c - pre[lo])] - jb) >> WSH;
                if (wi < 32) wlo |= 1u << wi; else whi |= 1u << (wi - 32);
            }
            tsg_wave_sync();
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            wlo |= __shfl_xor(wlo, o, 64);
            whi |= __shfl_xor(whi, o, 64);
        }
        wmask = ((unsigned long long)whi << 32) | wlo;
    }

    int total = 0;
    const int base = FILL ? Cptr_or_cnt[I] : 0;
    // a row whose candidates fit one window keeps the count pass's bitmap
    // (bmstore, BMW words per tile-row) so the fill pass reads it back
    const bool kept = bmstore != nullptr && jmax >= jmin && jmax - jb < 32 * BMW;
    unsigned *keep = kept ? bmstore + (long long)I * BMW : nullptr;
    constexpr int V = BMW / 64;            // window words per lane: lane + 64 v
    constexpr int U = BMW == 128 ? 8 : BMW == 256 ? 2 : 1;  // kept B tile-rows whose words are loaded together
    for (int w0 = jb; w0 <= jmax; w0 += 32 * BMW) {
        const int wi = (w0 - jb) >> WSH;
        if (wi < 64 && !((wmask >> wi) & 1ull)) continue;  // no candidate in this window
        const int nw = min(BMW, ((jmax - w0) >> 5) + 1);
        if (FILL && kept) {
            for (int k = lane; k < nw; k += 64) bm[k] = keep[k];
            tsg_wave_sync();
        } else {
            for (int k = lane; k < nw; k += 64) bm[k] = 0u;
            tsg_wave_sync();
            const int W0 = w0 >> 5;  // absolute word of the window's first word
            for (int c0 = a0; c0 < a1; c0 += 64) {
                const int p = c0 + lane;
                int b0 = 0, len = 0;
                int4 d = make_int4(0, 0, 0, 0);
                if (p < a1) {
                    const int K = Acol[p];
                    b0 = Bptr[K];
                    len = Bptr[K + 1] - b0;
                    if (Bdesc) {
                        d = Bdesc[K];
                        if (d.z > 0) len = 0;
                    }
                }
                // kept B tile-rows: window words [lo, hi) of each, U rows' loads
                // in flight; a lane ORs only its own words (lane + 64 v), so
                // no atomics, and LDS order within the wave keeps these
                // before the candidate atomics below
                unsigned long long dm = __ballot(d.z > 0);
                while (dm) {
                    unsigned t[U][V];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        int lo = 0, hi = 0, base = 0;
                        if (dm) {
                            const int j = __ffsll((long long)dm) - 1;
                            dm &= dm - 1;
                            const int dF = __builtin_amdgcn_readlane(d.y, j);
                            const int dn = __builtin_amdgcn_readlane(d.z, j);
                            lo = max(W0, dF) - W0;
                            hi = min(W0 + nw, dF + dn) - W0;
                            base = __builtin_amdgcn_readlane(d.x, j) + W0 - dF;
                        }
#pragma unroll
                        for (int v = 0; v < V; v++) {
                            const int k = 64 * v + lane;
                            t[u][v] = 0u;
                            if (64 * v + 64 > lo && 64 * v < hi && k >= lo && k < hi) t[u][v] = Bbits[base + k];
                        }
                    }
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        unsigned x = 0u;
#pragma unroll
                        for (int u = 0; u < U; u++) x |= t[u][v];
                        if (x) bm[64 * v + lane] |= x;
                    }
                }
                const int incl = tsg_wave_incl_scan(len);
                const int tot = __shfl(incl, 63, 64);
                pre[lane] = incl - len;
                pb0[lane] = b0;
                tsg_wave_sync();
                // 4 B tile columns per lane are loaded before their bits are set
                if (tot >= 64 * 32) {
                    // long B tile-rows (32+ tiles on average): the 64 lanes sweep
                    // one B tile-row at a time, no candidate search
                    const int na = min(64, a1 - c0);
                    for (int j = 0; j < na; j++) {
                        const int bj = pb0[j], lj = (j + 1 < na ? pre[j + 1] : tot) - pre[j];
                        for (int c = lane; c < lj; c += 256) {
                            int d[4];
#pragma unroll
                            for (int v = 0; v < 4; v++) d[v] = c + 64 * v < lj ? Bcol[bj + c + 64 * v] - w0 : -1;
#pragma unroll
                            for (int v = 0; v < 4; v++)
                                if (d[v] >= 0 && d[v] < 32 * BMW) atomicOr(&bm[d[v] >> 5], 1u << (d[v] & 31));
                        }
                    }
                } else {
                    for (int c = lane; c < tot; c += 256) {
                        int d[4];
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const int cc = c + 64 * v;
                            d[v] = -1;
                            if (cc < tot) {
                                int lo = 0;
#pragma unroll
                                for (int st = 32; st > 0; st >>= 1)
                                    if (pre[lo + st] <= cc) lo += st;
                                d[v] = Bcol[pb0[lo] + (cc - pre[lo])] - w0;
                            }
                        }
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            if (d[v] >= 0 && d[v] < 32 * BMW) atomicOr(&bm[d[v] >> 5], 1u << (d[v] & 31));
                    }
                }
                tsg_wave_sync();
            }
            if (!FILL && kept)
                for (int k = lane; k < nw; k += 64) keep[k] = bm[k];
        }
        if (!FILL) {
            int cnt = 0;
            for (int k = lane; k < nw; k += 64) cnt += __popc(bm[k]);
            total += tsg_wave_sum(cnt);
        } else {
            total += emit_window(bm, nw, w0, lane, Ccol + base + total);
        }
        tsg_wave_sync();
    }
    if (FILL)
        for (int k = lane; k < total; k += 64) Crow[base + k] = I;
    if (!FILL && lane == 0) {
        Cptr_or_cnt[I] = total;
        // the candidates are exactly C's tiles, so this is the row's C tile-column span
        if (rowspan) rowspan[I] = total > 0 ? jmax - jmin + 1 : 0;
    }
}

// ------------------------------------------------------------------ pairs
// Operands of steps 2 and 3.  B's tile data is in row-major tile order;
// its CSC index (Bcscptr/Bcscrow/Bcscid) lists each tile column's tiles by
// ascending tile row.
struct TileOperands {
    const int *Aptr, *Acol, *Annz;
    const unsigned char *Aptr16;
    const unsigned short *Amask;
    const double *Aval;
    const int *Bptr, *Bcol;
    const int *Bcscptr, *Bcscrow, *Bcscid, *Bnnz;
    const unsigned char *Bptr16;
    const unsigned short *Bmask;
    const double *Bval;
    // A's element row index (may be NULL): rows' entries in ascending k
    const int *Arowp, *Acolx;
    const double *Avalx;
};

// Index p in [0, len) with list[p] == key, or -1 (list ascending).
__device__ __forceinline__ int find_sorted(const int *__restrict__ list, int len, int key) {
    int lo = 0, hi = len - 1;
    while (lo <= hi) {
        const int mid = (lo + hi) >> 1;
        const int v = list[mid];
        if (v == key) return mid;
        if (v < key) lo = mid + 1; else hi = mid - 1;
    }
    return -1;
}

#define PAIR_LDS_MAX 64  // both tile lists staged in LDS when each is this short

// Calls body(ta, tb) for every matched pair (A tile ta, B tile tb) of C tile
// (I, J), in ascending inner tile index K, uniformly across the 16 lanes of
// the calling group (g = group in the wave, r = lane in the group).  The
// keys of the shorter list are binary-searched in the longer one, 16 per
// round; a 64-bit ballot keeps the matches in key order.  Short lists are
// first copied to the group's LDS slots (sa/sb) so the searches hit LDS.
template <typename Body>
__device__ __forceinline__ void for_each_pair(const TileOperands &op, int I, int J, int g, int r, int *sa, int *sb,
                                              Body body) {
    const int a0 = op.Aptr[I], la = op.Aptr[I + 1] - a0;
    const int b0 = op.Bcscptr[J], lb = op.Bcscptr[J + 1] - b0;
    if (la == 0 || lb == 0) return;
    const bool a_short = la <= lb;
    const int ls = a_short ? la : lb, ll = a_short ? lb : la;
    const int *S = a_short ? op.Acol + a0 : op.Bcscrow + b0;
    const int *L = a_short ? op.Bcscrow + b0 : op.Acol + a0;
    const bool staged = la <= PAIR_LDS_MAX && lb <= PAIR_LDS_MAX;
    if (staged) {
        for (int x = r; x < ls; x += 16) sa[x] = S[x];
        for (int x = r; x < ll; x += 16) sb[x] = L[x];
        tsg_wave_sync();
        S = sa;
        L = sb;
    }
    const int src_base = g * 16;
    for (int base = 0; base < ls; base += 16) {
        const int idx = base + r;
        int pos = -1;
        if (idx < ls) pos = find_sorted(L, ll, S[idx]);
        const unsigned long long bal = __ballot(pos >= 0);
        unsigned m16 = (unsigned)(bal >> src_base) & 0xffffu;
        while (m16) {
            const int j = __ffs(m16) - 1;
            m16 &= m16 - 1;
            const int sidx = base + j;
            const int lpos = __shfl(pos, src_base + j, 64);
            const int apos = a_short ? sidx : lpos;
            const int bpos = a_short ? lpos : sidx;
            body(a0 + apos, op.Bcscid[b0 + bpos]);
        }
    }
    if (staged) tsg_wave_sync();
}

// ------------------------------------------------------------------ segments
// A segment is a range [s0, s1) of the C tiles of one tile-row I, stored
// as int4 {I, s0, s1, index in the tile-row}; its C tiles cover the tile
// columns [Ccol[c0+s0], Ccol[c0+s1-1]], and only the B tiles inside that
// column range meet them.

// Step-2 segments: tile-rows are cut so that a segment fits a block's LDS.
#define G2_UMAX 512       // C tiles of one segment of the tile-pair and hash kernels
#define G2_MAP_MAX 16384  // widest tile-row span with a direct column map (bytes of LDS)
#define G2D_WIN 4096      // tile columns of one window of the dense kernel (128 KiB of bits)
#define G2D_SMALL 1024    // widest tile-row span that takes it with small blocks

// Step-2 kernel of a tile-row with u > 0 C tiles over `span` tile columns,
// whose A tile-row has `ents` entries in `tiles` tiles:
//   0  tile pairs (k_step2_rows)
//   1  element-wise, C tiles in a hash (k_step2_elem)
//   2  element-wise, the tile-row's columns as bits in LDS, one small block
//      per tile-row (k_step2_dense)
//   3  the same in windows of G2D_WIN tile columns, one large block each
// Element-wise needs B's row index (elem), and the dense form A's too (rx).
// Hypersparse tile-rows (at most 4 entries per A tile, or all with `all`)
// go element-wise: one step per product instead of one per tile pair.  The
// dense form costs its window's 32 bytes a tile column whatever is in it and
// one LDS atomic a product, and a second window walks the A rows again with
// two searches in every B row; the hash costs a probe chain a product and
// such a walk per 512 tiles.  Erdos-Renyi A^2, hash against dense: 65536 rows
// with 43 / 53 / 63% of the span filled 408 / 483 / 632 against 413 / 486 /
// 535 us, 16384 rows with 29 / 50% 165 / 162 against 182 / 157 us; 131072
// rows (two windows) with 39 / 54 / 67 / 86% 1138 / 1487 / 1830 / 2423
// against 1240 / 1537 / 1820 / 2326 us.  So half of one window, three fifths
// of several.  Tile-pair rows of more than one segment take it too (each
// pair a loop over 16 rows, the segments a walk each): the 72 hub tile-rows
// of R-MAT scale 16 A*A^T, 24% of its products, were 5.5 ms of step 2's 17.1;
// all of it is 2.1 ms now.  So do those of many A tiles, whose pairs one block
// visits: above 128 tiles (R-MAT A^2, 6 edges a vertex, scale 12 546 -> 471 us,
// scale 13 1190 -> 880; scale 13 A*A^T, 14 edges, 2170 -> 1820).  From 65 tiles, a
// launch more for a part of few tile-rows costs what it saves (R-MAT scale 11, 16
// edges, 481 -> 538).
__device__ __forceinline__ int step2_kind(int u, int span, long long ents, int tiles, int elem, int all, int rx) {
    if (!elem) return 0;
    const bool el = all || ents <= 4ll * tiles;
    const bool many = tiles > 128 && ents <= 64ll * tiles;
    if (rx && (el || many || u > G2_UMAX) && (span <= G2D_WIN ? 2ll * u >= span : 5ll * u >= 3ll * span))
        return span <= G2D_SMALL ? 2 : 3;
    return el ? 1 : 0;
}
// Segments of such a tile-row.  Kind 3: windows of equal width of at most
// G2D_WIN tile columns, and one more per G2D_ENTS entries of the A tile-row
// (a hub tile-row's products would keep one CU busy long after the others: R-MAT
// scale 16 2.4 ms with 16384, 2.15 with 4096, 2.2 with 1024),
// at most as many as the hash kernel would take, so that a list of one per
// tile-row and G2_UMAX tiles holds every kind's.
#define G2D_ENTS 4096
__device__ __forceinline__ int step2_segments(int kind, int u, int span, long long ents) {
    if (kind == 2) return 1;
    const int n = (u + G2_UMAX - 1) / G2_UMAX;
    if (kind < 2) return n;
    return max((span + G2D_WIN - 1) / G2D_WIN, (int)min((long long)n, ents / G2D_ENTS + 1));
}

// The step-2 segments of every kind, kind k from items[base.k] on in no
// particular order (neighbouring tile-rows stay near each other); ctr[k]
// (zeroed beforehand) counts them.  One atomic per wave and kind present.
__global__ void __launch_bounds__(256)
k_seg2_fill(const int *__restrict__ Cptr, const int *__restrict__ Ccol, const int *__restrict__ Aptr,
            const int *__restrict__ Annz, int tilem, int elem, int all, int rx, int4 base, int *__restrict__ ctr,
            int4 *__restrict__ items) {
    const int I = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
    int c0 = 0, u = 0, span = 0, kind = -1, n = 0;
    if (I < tilem) {
        c0 = Cptr[I];
        u = Cptr[I + 1] - c0;
        if (u > 0) {
            const int a0 = Aptr[I], a1 = Aptr[I + 1];
            span = Ccol[c0 + u - 1] - Ccol[c0] + 1;
            kind = step2_kind(u, span, (long long)Annz[a1] - Annz[a0], a1 - a0, elem, all, rx);
            n = step2_segments(kind, u, span, (long long)Annz[a1] - Annz[a0]);
        }
    }
    int pos = 0;
#pragma unroll
    for (int k = 0; k < S2_KINDS; k++) {
        if (!__ballot(kind == k)) continue;
        const int mine = kind == k ? n : 0, incl = tsg_wave_incl_scan_dpp(mine);
        int b = 0;
        if (lane == 63) b = atomicAdd(&ctr[k], incl);
        b = __builtin_amdgcn_readlane(b, 63) + (k == 0 ? base.x : k == 1 ? base.y : k == 2 ? base.z : base.w);
        if (kind == k) pos = b + incl - mine;
    }
    if (kind < 0) return;
    if (kind < 2) {
        for (int j = 0; j < n; j++)
            items[pos + j] = make_int4(I, j * G2_UMAX, min(u, (j + 1) * G2_UMAX), j);
    } else {
        int s0 = 0;
        const int jlo = Ccol[c0], win = (span + n - 1) / n;
        for (int j = 0; j < n; j++) {  // first tile at or past each window's end
            int lo = s0, hi = u;
            if (j + 1 < n) {
                const int key = jlo + (j + 1) * win;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (Ccol[c0 + mid] < key) lo = mid + 1; else hi = mid;
                }
            } else {
                lo = u;
            }
            items[pos + j] = make_int4(I, s0, lo, j);
            s0 = lo;
        }
    }
}

// Step-3 element segments: tile s belongs to segment floor(p(s) / H), p(s) =
// C nonzeros of the row before tile s and H = max_nnz - 255; a tile holds at
// most 256 nonzeros, so ids grow by at most one per tile, every id up to the
// last is present, and a segment holds at most H + 255 = max_nnz nonzeros.
// Counts of the tile-rows with rowcls == want; k_seg1_fill writes them.
__global__ void __launch_bounds__(256)
k_seg1_count(const int *__restrict__ Cptr, const int *__restrict__ Cnnz, int tilem,
             const unsigned char *__restrict__ rowcls, int want, int max_nnz, int *__restrict__ cnt) {
    const int I = blockIdx.x * 256 + threadIdx.x;
    if (I >= tilem) return;
    const int c0 = Cptr[I], u = Cptr[I + 1] - c0;
    cnt[I] = u > 0 && rowcls[I] == want ? (Cnnz[c0 + u - 1] - Cnnz[c0]) / (max_nnz - 255) + 1 : 0;
}

// Upper bound on the step-2 segments of a C with tilem tile-rows and numtile
// tiles: one per tile-row and one per G2_UMAX tiles (a dense window past a
// row's first stands for at least G2D_WIN / 2 tiles or for G2_UMAX).
static long long seg2_bound(long long tilem, long long numtile) { return tilem + numtile / G2_UMAX + 1; }
static_assert(G2D_WIN / 2 >= G2_UMAX, "dense windows within the segment bound");

// First index in [lo, hi) with list[index] >= key (list ascending).
__device__ __forceinline__ int lower_bound_i(const int *__restrict__ list, int lo, int hi, int key) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (list[mid] < key) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Step-3 element segments, one thread per segment (a hub tile-row has thousands, each
// found by a binary search; one thread per row left the whole launch
// waiting on the longest row): segment j's row is the last row whose first
// segment is at or before j (off[] is the scanned per-row count, off[tilem]
// the total), its bounds the first tiles at or past its ends.
__global__ void __launch_bounds__(256)
k_seg1_fill(const int *__restrict__ Cptr, const int *__restrict__ Cnnz, int tilem, const int *__restrict__ off,
            int max_nnz, int4 *__restrict__ items) {
    const long long j = (long long)blockIdx.x * 256 + threadIdx.x;
    if (j >= off[tilem]) return;
    int lo = 0, hi = tilem - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= j) lo = mid; else hi = mid - 1;
    }
    const int I = lo, jj = (int)(j - off[I]), n = off[I + 1] - off[I];
    const int c0 = Cptr[I], u = Cptr[I + 1] - c0;
    const int H = max_nnz - 255, base = Cnnz[c0];
    const int s0 = jj == 0 ? 0 : lower_bound_i(Cnnz, c0, c0 + u - 1, base + jj * H) - c0;
    const int s1 = jj + 1 == n ? u : lower_bound_i(Cnnz, c0, c0 + u - 1, base + (jj + 1) * H) - c0;
    items[j] = make_int4(I, s0, s1, jj);
}

// ------------------------------------------------------------------ step 2
// Row-wise (Gustavson) bitmask symbolic: one 256-thread block per segment
// of a C tile-row.  Every (A tile (I,K), B tile (K,J)) pair of the row
// with J in the segment's column range -- the pairs step 1 enumerated --
// is visited exactly once, flattened over the threads; no intersection
// search is needed.  Row r of the pair's product pattern, OR over k in
// Amask[r] of Bmask[k], is OR-ed into C tile J's row mask held in LDS (OR
// is order-free, so LDS atomics are exact).  A tiles with a single entry
// (r, k) contribute B row k to C row r alone; their pairs are enumerated
// before the others' so that a wave's lanes take one kind of pair.
#define G2_THREADS 256
#define G2_PCHUNK 256  // A tiles per enumeration round
#define G2_MSTRIDE 9      // LDS words per C tile mask set / per thread B mask copy (8 used)

// Sizes of steps 2 and 3 from the step-1 count pass's per-row tile counts
// and spans (atomics on out[0..8), zeroed beforehand):
//   [0] most C tiles of a tile-pair tile-row (capped at the segment size)
//   [1] widest tile-column span of a tile-row
//   [2] widest span of at most G2_MAP_MAX of a tile-pair tile-row
//   [3 + k] step-2 segments of kind k
//   [7] widest span of a kind-2 tile-row
// A few large blocks stride over the rows, so that the atomics (one cache
// line, serialised) are few.
#define ROW_STATS_BLOCKS 64
#define ROW_STATS 8
__device__ __forceinline__ void row_stats_add(int v[ROW_STATS], int I, int u, const int *__restrict__ span,
                                              const int *__restrict__ Aptr, const int *__restrict__ Annz, int elem, int all,
                                              int rx) {
    if (u <= 0) return;
    const int s1 = span[I], a0 = Aptr[I], a1 = Aptr[I + 1];
    const long long ents = (long long)Annz[a1] - Annz[a0];
    const int kind = step2_kind(u, s1, ents, a1 - a0, elem, all, rx);
    v[1] = max(v[1], s1);
    if (kind == 0) {
        v[0] = max(v[0], min(u, G2_UMAX));
        if (s1 <= G2_MAP_MAX) v[2] = max(v[2], s1);
    }
#pragma unroll
    for (int k = 0; k < S2_KINDS; k++) v[3 + k] += kind == k ? step2_segments(kind, u, s1, ents) : 0;
    if (kind == 2) v[7] = max(v[7], s1);
}
// The block's (1024 threads) sum or maximum of word i, in the threads i < ROW_STATS.
__device__ __forceinline__ int row_stats_fold(int v[ROW_STATS], int s_r[16][ROW_STATS]) {
#pragma unroll
    for (int i = 0; i < ROW_STATS; i++) {
        v[i] = i >= 3 && i < 7 ? tsg_wave_sum(v[i]) : tsg_wave_max(v[i]);
        if ((threadIdx.x & 63) == 0) s_r[threadIdx.x >> 6][i] = v[i];
    }
    __syncthreads();
    int x = 0;
    if (threadIdx.x < ROW_STATS) {
        const int i = threadIdx.x;
        x = s_r[0][i];
        for (int w = 1; w < 16; w++) x = i >= 3 && i < 7 ? x + s_r[w][i] : max(x, s_r[w][i]);
    }
    return x;
}
__global__ void __launch_bounds__(1024)
k_row_stats(const int *__restrict__ cnt, const int *__restrict__ span, const int *__restrict__ Aptr,
            const int *__restrict__ Annz, int tilem, int elem, int all, int rx, int *__restrict__ out) {
    __shared__ int s_r[16][ROW_STATS];
    int v[ROW_STATS];
#pragma unroll
    for (int i = 0; i < ROW_STATS; i++) v[i] = 0;
    for (int I = blockIdx.x * 1024 + threadIdx.x; I < tilem; I += gridDim.x * 1024)
        row_stats_add(v, I, cnt[I], span, Aptr, Annz, elem, all, rx);
    const int x = row_stats_fold(v, s_r);
    if (threadIdx.x < ROW_STATS) {
        if (threadIdx.x >= 3 && threadIdx.x < 7) atomicAdd(&out[threadIdx.x], x);
        else atomicMax(&out[threadIdx.x], x);
    }
}
// The same for few tile-rows, one a thread, with the scan of the counts, in
// place (ptr[tilem] = total); the total and the statistics go to pinned memory.
// (With four a thread it lost 2 to 10 us against two launches at 3,100 to 3,750
// tile-rows.)
#define ROW_STATS_ONE 1024
__global__ void __launch_bounds__(1024)
k_row_stats_one(int *ptr, const int *__restrict__ span, const int *__restrict__ Aptr, const int *__restrict__ Annz,
                int tilem, int elem, int all, int rx, long long *__restrict__ host) {
    __shared__ int s_r[16][ROW_STATS];
    __shared__ long long s_w[16];
    const int I = threadIdx.x, c = I < tilem ? ptr[I] : 0;
    int v[ROW_STATS];
#pragma unroll
    for (int i = 0; i < ROW_STATS; i++) v[i] = 0;
    row_stats_add(v, I, c, span, Aptr, Annz, elem, all, rx);
    const long long incl = tsg_wave_incl_scan((long long)c);
    if ((I & 63) == 63) s_w[I >> 6] = incl;
    const int x = row_stats_fold(v, s_r);  // (a barrier within)
    long long at = incl - c;
    for (int w = 0; w < (I >> 6); w++) at += s_w[w];
    if (I < ROW_STATS) reinterpret_cast<int *>(host + 1)[I] = x;
    if (I < tilem) ptr[I] = (int)at;
    if (I == 1023) {
        host[0] = at + c;
        ptr[tilem] = at + c > 0x7fffffffLL ? 0x7fffffff : (int)(at + c);
    }
}

static_assert(G2_PCHUNK == G2_THREADS, "one A tile of a chunk per thread");
__global__ void __launch_bounds__(G2_THREADS)
k_step2_rows(TileOperands op, const int4 *__restrict__ segs, int nseg, const int *__restrict__ Cptr, const int *__restrict__ Ccol, unsigned short *__restrict__ Cmask, unsigned char *__restrict__ Cptr16,
             int *__restrict__ Cnnz, int umax, int mapbytes) {
    // dynamic LDS, sized by the largest segment: the segment's C tile masks
    // (two 16-bit rows per word, even row high; G2_MSTRIDE words per tile so
    // that the lanes' tiles fall in distinct banks), its tile columns, and
    // when every segment has at most 256 tiles, mapbytes bytes for a direct
    // map tile column -> slot, used by the segments spanning at most
    // mapbytes tile columns (the others search the tile columns)
    extern __shared__ __align__(16) unsigned char g2_smem[];
    unsigned *s_m = reinterpret_cast<unsigned *>(g2_smem);
    int *s_ccol = reinterpret_cast<int *>(g2_smem + 4 * G2_MSTRIDE * (size_t)umax);
    unsigned char *s_map = g2_smem + (4 * G2_MSTRIDE + 4) * (size_t)umax;
    // per enumeration position (single-entry A tiles first): first pair,
    // first B tile, A tile (offset in the chunk), single entry (row |
    // column << 4, or 255)
    __shared__ int s_pre[G2_PCHUNK];
    __shared__ int s_b0[G2_PCHUNK];
    __shared__ unsigned char s_pid[G2_PCHUNK];
    __shared__ unsigned char s_rk[G2_PCHUNK];
    __shared__ int s_wsg[G2_THREADS / 64];
    __shared__ int s_tot;
    // B masks of each thread's pair, word-major (word i = rows 2i (low half)
    // and 2i+1), so that a wave's lanes read and write consecutive banks
    __shared__ unsigned s_bst[8][G2_THREADS];
    const int tid = threadIdx.x;
    // one block per segment, each XCD a contiguous range; without a list
    // (segs NULL) every tile-row is one segment
    const unsigned blk = tsg_block();
    if (blk >= (unsigned)nseg) return;  // block-uniform
    const int w = (int)tsg_xcd_block(blk, (unsigned)nseg);
    int4 sg = make_int4(w, 0, 0, 0);
    if (segs) {
        sg = segs[w];
    } else {
        sg.z = Cptr[w + 1] - Cptr[w];
        if (sg.z == 0) return;  // block-uniform
    }
    const int I = sg.x;
    const int c0 = Cptr[I] + sg.y, u = sg.z - sg.y;
    const bool whole = sg.y == 0 && sg.z == Cptr[I + 1] - Cptr[I];
    const int jlo = Ccol[c0], jhi = Ccol[c0 + u - 1];
    const bool usemap = jhi - jlo < mapbytes;
    for (int i = tid; i < u; i += G2_THREADS) {
        const int J = Ccol[c0 + i];
        s_ccol[i] = J;
        if (usemap) s_map[J - jlo] = (unsigned char)i;
    }
    for (int i = tid; i < u * G2_MSTRIDE; i += G2_THREADS) s_m[i] = 0u;
    const int a0 = op.Aptr[I], a1 = op.Aptr[I + 1];
    __shared__ int s_wsum[G2_THREADS / 64];
    for (int pc = a0; pc < a1; pc += G2_PCHUNK) {
        const int np = min(G2_PCHUNK, a1 - pc);
        int len = 0, b0 = 0, rk = 255;
        if (tid < np) {
            const uint4 *am4 = reinterpret_cast<const uint4 *>(op.Amask + (long long)(pc + tid) * 16);
            const uint4 aA = am4[0], aB = am4[1];
            const unsigned aw[8] = {aA.x, aA.y, aA.z, aA.w, aB.x, aB.y, aB.z, aB.w};
            int nz = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                nz += __popc(aw[i]);
                if (aw[i]) {
                    const int bit = 31 - __clz(aw[i]);  // row 2i in the low half, 2i+1 in the high
                    rk = (2 * i + (bit >> 4)) | ((15 - (bit & 15)) << 4);
                }
            }
            if (nz != 1) rk = 255;
            const int K = op.Acol[pc + tid];
            b0 = op.Bptr[K];
            int b1 = op.Bptr[K + 1];
            if (!whole) {  // B tiles of row K inside the segment's columns
                b0 = lower_bound_i(op.Bcol, b0, b1, jlo);
                b1 = lower_bound_i(op.Bcol, b0, b1, jhi + 1);
            }
            len = b1 - b0;
        }
        // enumeration positions: single-entry A tiles first, in thread order
        {
            const bool sgl = tid < np && rk != 255, dns = tid < np && rk == 255;
            const unsigned long long sb = __ballot(sgl), db = __ballot(dns);
            const unsigned long long lt = (1ull << (tid & 63)) - 1ull;
            if ((tid & 63) == 0) {
                s_wsg[tid >> 6] = __popcll(sb);
                s_wsum[tid >> 6] = __popcll(db);
            }
            __syncthreads();
            int ns = 0, sbef = 0, dbef = 0;
            for (int w2 = 0; w2 < G2_THREADS / 64; w2++) {
                ns += s_wsg[w2];
                if (w2 < (tid >> 6)) {
                    sbef += s_wsg[w2];
                    dbef += s_wsum[w2];
                }
            }
            const int pos = sgl ? sbef + __popcll(sb & lt) : ns + dbef + __popcll(db & lt);
            if (tid < np) {
                s_pre[pos] = len;
                s_b0[pos] = b0;
                s_pid[pos] = (unsigned char)tid;
                s_rk[pos] = (unsigned char)rk;
            }
            __syncthreads();
            len = tid < np ? s_pre[tid] : 0;
        }
        // block-wide exclusive scan of len in position order
        const int incl = tsg_wave_incl_scan(len);
        if ((tid & 63) == 63) s_wsum[tid >> 6] = incl;
        __syncthreads();
        int woff = 0;
        for (int w2 = 0; w2 < (tid >> 6); w2++) woff += s_wsum[w2];
        s_pre[tid] = woff + incl - len;
        if (tid == G2_THREADS - 1) s_tot = woff + incl;
        __syncthreads();
        const int total = s_tot;
        // two pairs per round, so that both pairs' B tile loads are in flight
#pragma unroll 2
        for (int x = tid; x < total; x += G2_THREADS) {
            int p = 0;
#pragma unroll
            for (int st = G2_PCHUNK / 2; st > 0; st >>= 1)
                if (p + st < G2_PCHUNK && s_pre[p + st] <= x) p += st;
            const int q = s_b0[p] + (x - s_pre[p]);
            const int J = op.Bcol[q];  // J is in the segment's step-1 list
            int slot;
            if (usemap) {
                slot = s_map[J - jlo];
            } else {
                int lo = 0, hi = u - 1;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (s_ccol[mid] < J) lo = mid + 1; else hi = mid;
                }
                slot = lo;
            }
            const int rk1 = s_rk[p];
            if (rk1 != 255) {  // single entry (r, k): B row k into C row r
                const int r = rk1 & 15;
                const unsigned m = op.Bmask[(long long)q * 16 + (rk1 >> 4)];
                atomicOr(&s_m[slot * G2_MSTRIDE + (r >> 1)], m << ((r & 1) ? 0 : 16));
                continue;
            }
            const uint4 *bm4 = reinterpret_cast<const uint4 *>(op.Bmask + (long long)q * 16);
            const uint4 bA = bm4[0], bB = bm4[1];
            s_bst[0][tid] = bA.x;
            s_bst[1][tid] = bA.y;
            s_bst[2][tid] = bA.z;
            s_bst[3][tid] = bA.w;
            s_bst[4][tid] = bB.x;
            s_bst[5][tid] = bB.y;
            s_bst[6][tid] = bB.z;
            s_bst[7][tid] = bB.w;
            const uint4 *am4 = reinterpret_cast<const uint4 *>(op.Amask + (long long)(pc + s_pid[p]) * 16);
            const uint4 aA = am4[0], aB = am4[1];
            const unsigned aw[8] = {aA.x, aA.y, aA.z, aA.w, aB.x, aB.y, aB.z, aB.w};
#pragma unroll
            for (int r = 0; r < 16; r++) {
                unsigned am = (aw[r >> 1] >> ((r & 1) * 16)) & 0xffffu;  // little-endian: row 2w low half
                if (!am) continue;
                unsigned acc = 0;  // even k in the low half, odd in the high
                // a word of two B rows a step (one row a step: banded 39989, nearly full
                // tiles, 36 us of kernel against 27; three entries a row the same)
                while (am) {
                    const int i = (__clz((int)am) - 16) >> 1, sh = 14 - 2 * i;
                    const unsigned sel = am >> sh, x = sel >> 1 | (sel & 1u) << 16;
                    acc |= s_bst[i][tid] & ((x << 16) - x);  // x * 0xffff
                    am &= (1u << sh) - 1u;
                }
                acc |= acc >> 16;
                atomicOr(&s_m[slot * G2_MSTRIDE + (r >> 1)], (r & 1) ? acc & 0xffffu : acc << 16);
            }
        }
        __syncthreads();
    }
    // per C tile: popcounts, u8 row offsets, tile nnz
    for (int s = tid; s < u; s += G2_THREADS) {
        unsigned w8[8];
#pragma unroll
        for (int k = 0; k < 8; k++) w8[k] = s_m[s * G2_MSTRIDE + k];
        unsigned mk[8], pt[4];
        int sum = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const unsigned hi = w8[k] >> 16, lo = w8[k] & 0xffffu;  // rows 2k, 2k+1
            mk[k] = hi | (lo << 16);                               // little-endian u16 pair
        }
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            unsigned o = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int r = q4 * 4 + b;
                const unsigned row = (r & 1) ? (w8[r >> 1] & 0xffffu) : (w8[r >> 1] >> 16);
                o |= (unsigned)sum << (8 * b);
                sum += __popc(row);
            }
            pt[q4] = o;
        }
        const long long t = c0 + s;
        uint4 *cm4 = reinterpret_cast<uint4 *>(Cmask + t * 16);
        cm4[0] = make_uint4(mk[0], mk[1], mk[2], mk[3]);
        cm4[1] = make_uint4(mk[4], mk[5], mk[6], mk[7]);
        *reinterpret_cast<uint4 *>(Cptr16 + t * 16) = make_uint4(pt[0], pt[1], pt[2], pt[3]);
        Cnnz[t] = sum;
    }
}

// Element-wise bitmask symbolic for hypersparse tile-rows (B carries its
// row index): one 256-thread block per segment; each thread takes whole A
// tiles of the tile-row and, for each of their entries (r, k), ORs the
// columns of B row k that fall in the segment's range into the row-r mask
// of their C tile (slot found through an LDS hash of the segment's tile
// columns).  Work is one step per intermediate product instead of one per
// (A tile, B tile) pair; OR is order-free, so LDS atomics are exact.
#define G2E_HASH 1024  // >= 2 * G2_UMAX
static_assert(G2_UMAX <= 512, "C tile index in 9 bits of a step-2 hash slot");

__device__ __forceinline__ unsigned col_hash10(int J) { return ((unsigned)J * 2654435761u) >> 22; }

__global__ void __launch_bounds__(G2_THREADS)
k_step2_elem(TileOperands op, const int *__restrict__ Browp, const int *__restrict__ Bcolx,
             const int4 *__restrict__ segs, int nseg, const int *__restrict__ Cptr, const int *__restrict__ Ccol,
             unsigned short *__restrict__ Cmask, unsigned char *__restrict__ Cptr16, int *__restrict__ Cnnz) {
    __shared__ unsigned s_m[G2_UMAX * 8];  // two 16-bit rows per word, even row high
    // hash of the segment's tile columns: slot (J - jlo + 1) << 9 | C tile
    // index (J - jlo + 1 < 2^23 as B has at most 2^27 - 32 columns when this
    // kernel runs, index < G2_UMAX = 512); 0 = empty
    __shared__ unsigned s_hkey[G2E_HASH];
    const int tid = threadIdx.x;
    const unsigned blk = tsg_block();
    if (blk >= (unsigned)nseg) return;  // block-uniform
    const int4 sg = segs[tsg_xcd_block(blk, (unsigned)nseg)];
    const int I = sg.x;
    const int c0 = Cptr[I] + sg.y, u = sg.z - sg.y;
    for (int i = tid; i < u * 8; i += G2_THREADS) s_m[i] = 0u;
    for (int i = tid; i < G2E_HASH; i += G2_THREADS) s_hkey[i] = 0u;
    __syncthreads();
    const int jlo = Ccol[c0];
    for (int i = tid; i < u; i += G2_THREADS) {
        const int J = Ccol[c0 + i];
        unsigned h = col_hash10(J);
        const unsigned ent = (unsigned)(J - jlo + 1) << 9 | (unsigned)i;
        while (atomicCAS(&s_hkey[h], 0u, ent) != 0u) h = (h + 1) & (G2E_HASH - 1);  // u <= G2E_HASH / 2
    }
    __syncthreads();
    const int col_lo = Ccol[c0] * 16, col_hi = Ccol[c0 + u - 1] * 16 + 16;
    const int a0 = op.Aptr[I], a1 = op.Aptr[I + 1];
    __shared__ int s_tex[G2_THREADS + 1];  // entries before each tile of the chunk
    for (int tc = a0; tc < a1; tc += G2_THREADS) {
        // one chunk of A tiles: their entries numbered block-wide, one
        // entry per thread per step (balanced whatever the tile densities)
        const int t = tc + tid;
        int cnt = 0;
        if (t < a1) {
            const uint4 *am4 = reinterpret_cast<const uint4 *>(op.Amask + (long long)t * 16);
            const uint4 aA = am4[0], aB = am4[1];
            cnt = __popc(aA.x) + __popc(aA.y) + __popc(aA.z) + __popc(aA.w) + __popc(aB.x) + __popc(aB.y) +
                  __popc(aB.z) + __popc(aB.w);
        }
        __shared__ int s_w[G2_THREADS / 64];
        const int incl = tsg_wave_incl_scan(cnt);
        if ((tid & 63) == 63) s_w[tid >> 6] = incl;
        __syncthreads();
        int woff = 0;
        for (int q = 0; q < (tid >> 6); q++) woff += s_w[q];
        s_tex[tid] = woff + incl - cnt;
        if (tid == G2_THREADS - 1) s_tex[G2_THREADS] = woff + incl;
        __syncthreads();
        const int total = s_tex[G2_THREADS];
        for (int x = tid; x < total; x += G2_THREADS) {
            int ow = 0;  // tile of entry x: last with s_tex <= x
#pragma unroll
            for (int st = G2_THREADS / 2; st > 0; st >>= 1)
                if (ow + st < G2_THREADS && s_tex[ow + st] <= x) ow += st;
            const int tt = tc + ow;
            int j = x - s_tex[ow];
            // the tile's 16 row masks in one load; the row holding its j-th entry
            const uint4 *am4 = reinterpret_cast<const uint4 *>(op.Amask + (long long)tt * 16);
            const uint4 mA = am4[0], mB = am4[1];
            const unsigned mw[8] = {mA.x, mA.y, mA.z, mA.w, mB.x, mB.y, mB.z, mB.w};
            int r = 0;
            unsigned am = mw[0] & 0xffffu;
#pragma unroll
            for (int rr = 0; rr < 16; rr++) {
                const unsigned mr = (mw[rr >> 1] >> ((rr & 1) * 16)) & 0xffffu;
                if (rr == r && r < 15 && j >= __popc(mr)) {
                    j -= __popc(mr);
                    r++;
                }
            }
            am = (mw[r >> 1] >> ((r & 1) * 16)) & 0xffffu;
            for (int q = 0; q < j; q++) am &= ~(1u << (31 - __clz(am)));
            const int k = op.Acol[tt] * 16 + 15 - (31 - __clz(am));
            const int e1 = Browp[k + 1];
            bool more = true;
            // B row k's entries in the segment's column range, 4 loads at a time
            // the tile-row's first segment starts at B row k's first entry
            const int eb = sg.y == 0 ? Browp[k] : lower_bound_i(Bcolx, Browp[k], e1, col_lo);
            for (int e = eb; more && e < e1; e += 4) {
                int cols[4];
#pragma unroll
                for (int v = 0; v < 4; v++) cols[v] = e + v < e1 ? Bcolx[e + v] : 0x7fffffff;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int col = cols[v];
                    if (col >= col_hi) more = false;
                    if (!more) continue;
                    const int J = col >> 4;
                    unsigned h = col_hash10(J);  // J is in the segment's tile list
                    const unsigned key = (unsigned)(J - jlo + 1);
                    int probe = 0;
                    unsigned ent;
                    while (((ent = s_hkey[h]) >> 9) != key && ++probe < G2E_HASH) h = (h + 1) & (G2E_HASH - 1);
                    if (probe == G2E_HASH) continue;  // not reached for a consistent C structure
                    const unsigned bit = 1u << (15 - (col & 15));
                    atomicOr(&s_m[(int)(ent & 511u) * 8 + (r >> 1)], bit << ((r & 1) ? 0 : 16));
                }
            }
        }
        __syncthreads();  // s_tex is rewritten by the next chunk
    }
    __syncthreads();
    for (int sl = tid; sl < u; sl += G2_THREADS) {
        unsigned w8[8];
#pragma unroll
        for (int k = 0; k < 8; k++) w8[k] = s_m[sl * 8 + k];
        unsigned mk[8], pt[4];
        int sum = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) mk[k] = (w8[k] >> 16) | ((w8[k] & 0xffffu) << 16);
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            unsigned o = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int r = q4 * 4 + b;
                const unsigned row = (r & 1) ? (w8[r >> 1] & 0xffffu) : (w8[r >> 1] >> 16);
                o |= (unsigned)sum << (8 * b);
                sum += __popc(row);
            }
            pt[q4] = o;
        }
        const long long t = c0 + sl;
        uint4 *cm4 = reinterpret_cast<uint4 *>(Cmask + t * 16);
        cm4[0] = make_uint4(mk[0], mk[1], mk[2], mk[3]);
        cm4[1] = make_uint4(mk[4], mk[5], mk[6], mk[7]);
        *reinterpret_cast<uint4 *>(Cptr16 + t * 16) = make_uint4(pt[0], pt[1], pt[2], pt[3]);
        Cnnz[t] = sum;
    }
}

// Row offsets, entry count and masks of a C tile from its 16 row masks.
__device__ __forceinline__ void step2_store(const unsigned mk[8], long long t, unsigned short *__restrict__ Cmask,
                                            unsigned char *__restrict__ Cptr16, int *__restrict__ Cnnz) {
    unsigned pt[4];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        pt[q] = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            pt[q] |= (unsigned)sum << (8 * b);
            sum += __popc((mk[2 * q + (b >> 1)] >> (16 * (b & 1))) & 0xffffu);
        }
    }
    uint4 *cm4 = reinterpret_cast<uint4 *>(Cmask + t * 16);
    cm4[0] = make_uint4(mk[0], mk[1], mk[2], mk[3]);
    cm4[1] = make_uint4(mk[4], mk[5], mk[6], mk[7]);
    *reinterpret_cast<uint4 *>(Cptr16 + t * 16) = make_uint4(pt[0], pt[1], pt[2], pt[3]);
    Cnnz[t] = sum;
}

// Element-wise bitmask symbolic with the window's 16 rows as bits in LDS (a
// u16 per row and tile column): one block per segment, at most one LDS atomic
// OR per intermediate product and no lookup.  A wave takes up to 64 entries
// of the tile-row's A rows at a time.  B rows of G2D_LONG or more entries in
// the window are taken by the whole wave one after another; the products of
// the others are numbered through and taken one per lane, the entry of each
// found from a mark at its first product (running maximum over the lanes).
// Bound by HBM for short rows (ER 65521 A^2 1.17 GB in 0.285 ms, three quarters
// of it the 52 bytes per tile written), for hub rows by VALU (busy half of the
// time) and LDS (a third) behind the block's chain of loads, with the last
// blocks alone on the chip (R-MAT scale 16: CUs busy 62%).  Against the hash kernel (a probe chain per
// product, the tile-row cut every 512 tiles) and tile pairs: ER 65521 A^2 0.53
// -> 0.285 ms, R-MAT scale 16 A*A^T 17.1 -> 2.15 ms (580 G products/s).  Without
// the read before the atomic, the long rows' own path and the split of hub
// tile-rows the latter took 5.5 ms.
#define G2D_LONG 256                      // entries of a B row that a wave takes by itself
#define G2D_ROUNDS 8                      // products per lane and batch
#define G2D_BATCH (64 * G2D_ROUNDS)
#define G2D_WAVE_LDS (64 * 8 + G2D_BATCH) // bytes per wave
// LDS of a block of `threads` for windows of up to `width` tile columns.
static size_t g2d_lds(int width, int threads) {
    return 32 * (size_t)((width + 2) & ~1) + (size_t)(threads / 64) * G2D_WAVE_LDS;
}
__global__ void __launch_bounds__(1024)
k_step2_dense(const int *__restrict__ Arowp, const int *__restrict__ Acolx, int m, const int *__restrict__ Browp,
              const int *__restrict__ Bcolx, const int4 *__restrict__ segs, int nseg, const int *__restrict__ Cptr,
              const int *__restrict__ Ccol, unsigned short *__restrict__ Cmask, unsigned char *__restrict__ Cptr16,
              int *__restrict__ Cnnz, int width) {
    extern __shared__ __align__(16) unsigned char g2d_smem[];
    __shared__ int s_rp[17];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, nthr = blockDim.x, nwave = nthr >> 6;
    unsigned *bm = reinterpret_cast<unsigned *>(g2d_smem);
    unsigned char *ws = g2d_smem + 32 * (size_t)((width + 2) & ~1) + (size_t)wave * G2D_WAVE_LDS;
    int *s_delta = reinterpret_cast<int *>(ws), *s_row = s_delta + 64;
    unsigned char *s_mark = ws + 64 * 8;
    for (int w = blockIdx.x; w < nseg; w += gridDim.x) {
        const int4 sg = segs[w];
        const int I = sg.x, cb = Cptr[I], c0 = cb + sg.y, u = sg.z - sg.y;
        if (u == 0) continue;  // block-uniform: a window without tiles
        // the window starts at an even tile column, so that a word's half and
        // bit follow from the column alone: bit (column & 31) ^ 15
        const int j0 = Ccol[c0] & ~1, j1 = Ccol[c0 + u - 1];
        const int stride = (j1 - j0 + 2) & ~1;  // u16 per row
        const bool whole = cb + sg.y == cb && c0 + u == Cptr[I + 1];
        for (int i = tid; i < 2 * stride; i += nthr) reinterpret_cast<uint4 *>(bm)[i] = make_uint4(0u, 0u, 0u, 0u);
        if (tid < 17) s_rp[tid] = Arowp[min(16 * I + tid, m)];
        __syncthreads();
        const int x0 = s_rp[0], nx = s_rp[16] - x0;
        const int per = min(64, max(1, (nx + nwave - 1) / nwave));
        for (int c = wave * per; c < nx; c += nwave * per) {
            int b0 = 0, len = 0, row = 0;
            if (lane < per && c + lane < nx) {
                const int x = x0 + c + lane, k = Acolx[x];
                b0 = Browp[k];
                int b1 = Browp[k + 1];
                if (!whole) {  // B row k's entries in the window's columns
                    b0 = lower_bound_i(Bcolx, b0, b1, j0 * 16);
                    b1 = lower_bound_i(Bcolx, b0, b1, j1 * 16 + 16);
                }
                len = b1 - b0;
#pragma unroll
                for (int st = 8; st > 0; st >>= 1)
                    if (s_rp[row + st] <= x) row += st;
            }
            const int rw = (row * stride - j0) / 2;  // word of column 0 in the row
            // sets the bits of a lane's columns; those already set (most, in
            // a hub tile-row) cost a read, which lanes of one word share
            auto set = [&](const int (&col)[G2D_ROUNDS], const int (&rwi)[G2D_ROUNDS], int n) {
                unsigned have[G2D_ROUNDS];
#pragma unroll
                for (int i = 0; i < G2D_ROUNDS; i++) have[i] = bm[rwi[i] + (col[i] >> 5)];
#pragma unroll
                for (int i = 0; i < G2D_ROUNDS; i++) {
                    const unsigned bit = 1u << ((col[i] & 31) ^ 15);
                    if (64 * i + lane < n && !(have[i] & bit)) atomicOr(&bm[rwi[i] + (col[i] >> 5)], bit);
                }
            };
            // long B rows one at a time by the whole wave
            unsigned long long lm = __ballot(len >= G2D_LONG);
            while (lm) {
                const int j = __ffsll((long long)lm) - 1;
                lm &= lm - 1;
                const int n = __builtin_amdgcn_readlane(len, j), rwj = __builtin_amdgcn_readlane(rw, j);
                const int *bc = Bcolx + __builtin_amdgcn_readlane(b0, j);
                int rwi[G2D_ROUNDS];
#pragma unroll
                for (int i = 0; i < G2D_ROUNDS; i++) rwi[i] = rwj;
                for (int e = 0; e < n; e += G2D_BATCH) {
                    int col[G2D_ROUNDS];
#pragma unroll
                    for (int i = 0; i < G2D_ROUNDS; i++) col[i] = bc[min(e + 64 * i + lane, n - 1)];
                    set(col, rwi, n - e);
                }
            }
            if (len >= G2D_LONG) len = 0;
            const int incl = tsg_wave_incl_scan_dpp(len), pre = incl - len;
            const int total = __builtin_amdgcn_readlane(incl, 63);
            s_delta[lane] = b0 - pre;
            s_row[lane] = rw;
            int last = 0;
            for (int base = 0; base < total; base += G2D_BATCH) {
                reinterpret_cast<uint2 *>(s_mark)[lane] = make_uint2(0u, 0u);
                tsg_wave_sync();
                if (len > 0 && pre >= base && pre < base + G2D_BATCH) s_mark[pre - base] = (unsigned char)(lane + 1);
                tsg_wave_sync();
                int rwi[G2D_ROUNDS], col[G2D_ROUNDS];
#pragma unroll
                for (int i = 0; i < G2D_ROUNDS; i++) {
                    int q = s_mark[64 * i + lane];
                    if (__ballot(q != 0)) {
                        q = max(last, tsg_wave_incl_max_dpp(q));
                        last = __builtin_amdgcn_readlane(q, 63);
                    } else {  // all of one B row
                        q = last;
                    }
                    col[i] = s_delta[q - 1];
                    rwi[i] = s_row[q - 1];
                }
#pragma unroll
                for (int i = 0; i < G2D_ROUNDS; i++)  // every lane loads in bounds
                    col[i] = Bcolx[col[i] + min(base + 64 * i + lane, total - 1)];
                set(col, rwi, total - base);
                tsg_wave_sync();
            }
        }
        __syncthreads();
        const unsigned short *bm16 = reinterpret_cast<const unsigned short *>(bm);
        for (int t = tid; t < u; t += nthr) {
            const int at = Ccol[c0 + t] - j0;
            unsigned mk[8];
#pragma unroll
            for (int q = 0; q < 8; q++)
                mk[q] = bm16[2 * q * stride + at] | (unsigned)bm16[(2 * q + 1) * stride + at] << 16;
            step2_store(mk, c0 + t, Cmask, Cptr16, Cnnz);
        }
        __syncthreads();  // the next segment clears the bits
    }
}

// Tile-parallel step 2 (force_tile_parallel): one C tile per 16-lane group,
// pairs from the sorted-list intersection.
// Tile-parallel grids cover 16 work-items per C tile, which exceeds the
// 2^32 work-items of a launch beyond 2^28 tiles: such kernels run at most
// TP_MAX_BLOCKS blocks, each looping over virtual blocks.
#define TP_MAX_BLOCKS (1u << 20)

static inline unsigned tp_grid(long long vblocks) {
    return (unsigned)std::min<long long>(std::max<long long>(vblocks, 1), TP_MAX_BLOCKS);
}

__device__ __forceinline__ void step2_tile_body(const TileOperands &op, const int *__restrict__ Crow,
                                                const int *__restrict__ Ccol,
                                                int numtileC, unsigned short *__restrict__ Cmask,
                                                unsigned char *__restrict__ Cptr16, int *__restrict__ Cnnz,
                                                long long vblk, unsigned short *s_bm,
                                                int (*s_la)[PAIR_LDS_MAX], int (*s_lb)[PAIR_LDS_MAX]);

__global__ void __launch_bounds__(64 * S23_WAVES)
k_step2_tiles(TileOperands op, const int *__restrict__ Crow, const int *__restrict__ Ccol, int numtileC, unsigned short *__restrict__ Cmask,
              unsigned char *__restrict__ Cptr16, int *__restrict__ Cnnz) {
    __shared__ unsigned short s_bm[S23_WAVES][64];
    __shared__ int s_la[S23_WAVES][TILES_PER_WAVE][PAIR_LDS_MAX];
    __shared__ int s_lb[S23_WAVES][TILES_PER_WAVE][PAIR_LDS_MAX];
    const int wave = threadIdx.x >> 6;
    const long long nvb = ((long long)numtileC + S23_WAVES * TILES_PER_WAVE - 1) / (S23_WAVES * TILES_PER_WAVE);
    for (long long vb = tsg_xcd_block(blockIdx.x, gridDim.x); vb < nvb; vb += gridDim.x)
        step2_tile_body(op, Crow, Ccol, numtileC, Cmask, Cptr16, Cnnz, vb, s_bm[wave], s_la[wave],
                        s_lb[wave]);
}

__device__ __forceinline__ void step2_tile_body(const TileOperands &op, const int *__restrict__ Crow,
                                                const int *__restrict__ Ccol,
                                                int numtileC, unsigned short *__restrict__ Cmask,
                                                unsigned char *__restrict__ Cptr16, int *__restrict__ Cnnz,
                                                long long vblk, unsigned short *s_bmw,
                                                int (*s_law)[PAIR_LDS_MAX], int (*s_lbw)[PAIR_LDS_MAX]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r = lane & 15;
    const long long t = (vblk * S23_WAVES + wave) * TILES_PER_WAVE + g;
    if (t >= numtileC) return;  // whole groups exit together
    const int I = Crow[t], J = Ccol[t];
    unsigned short *bmg = &s_bmw[g * 16];
    unsigned orow = 0;
    for_each_pair(op, I, J, g, r, s_law[g], s_lbw[g], [&](int ta, int tb) {
        bmg[r] = op.Bmask[(long long)tb * 16 + r];
        tsg_wave_sync();
        unsigned am = op.Amask[(long long)ta * 16 + r];
        while (am) {
            const int b = 31 - __clz(am);
            am &= ~(1u << b);
            orow |= bmg[15 - b];
        }
        tsg_wave_sync();
    });
    const int cnt = __popc(orow);
    const int incl = tsg_group16_incl_scan(cnt);
    const int tot = __shfl(incl, g * 16 + 15, 64);
    Cmask[t * 16 + r] = (unsigned short)orow;
    Cptr16[t * 16 + r] = (unsigned char)(incl - cnt);
    if (r == 0) Cnnz[t] = tot;
}

// Tile counts per accumulator class (statistics only): one atomic per block.
__global__ void __launch_bounds__(256)
k_bins(const int *__restrict__ cnt, long long n, int dense_min, unsigned long long *__restrict__ bins) {
    __shared__ unsigned s[3];
    if (threadIdx.x < 3) s[threadIdx.x] = 0;
    __syncthreads();
    unsigned c0 = 0, c1 = 0, c2 = 0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int v = cnt[i];
        c0 += v == 0;
        c1 += v > 0 && v < dense_min;
        c2 += v >= dense_min;
    }
    c0 = tsg_wave_sum(c0);
    c1 = tsg_wave_sum(c1);
    c2 = tsg_wave_sum(c2);
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&s[0], c0);
        atomicAdd(&s[1], c1);
        atomicAdd(&s[2], c2);
    }
    __syncthreads();
    if (threadIdx.x < 3) atomicAdd(&bins[threadIdx.x], (unsigned long long)s[threadIdx.x]);
}

// ------------------------------------------------------------------ step 3
// Tile-rows whose C tiles and nonzeros fit the row-wise kernel's LDS
// accumulator go through k_step3_rows; the others through the
// tile-parallel k_step3 below (any size, no LDS limit on the row).
#define G3_THREADS 256
// Caps of the row-wise kernel (the LDS layout is sized at launch from the
// actual maxima of the rows that fit, at most ~60 KB per block).
#define G3_UMAX 256     // C tiles per tile-row (u8 slot ids)
#define G3_NNZMAX 3072  // C nonzeros per tile-row (LDS accumulator)
#define G3_QB 32        // B tiles per B tile-row (staging thread roles)
#define G3_BNNZ 512     // B values per B tile-row (two per thread)


#define ACC_STRIDE 17  // doubles per lane row (padding against bank conflicts)

__device__ __forceinline__ void step3_tile_body(const TileOperands &op, const int *__restrict__ Crow,
                                                const int *__restrict__ Ccol, int numtileC,
                                                const unsigned short *__restrict__ Cmask,
                                                const unsigned char *__restrict__ Cptr16,
                                                const int *__restrict__ Cnnz, unsigned char *__restrict__ Ccol8,
                                                double *__restrict__ Cval, int dense_min, int all_rows,
                                                const unsigned char *__restrict__ rowcls, long long vblk,
                                                double *s_accw, unsigned short *s_bmw, unsigned char *s_bpw,
                                                int (*s_law)[PAIR_LDS_MAX], int (*s_lbw)[PAIR_LDS_MAX]);

__global__ void __launch_bounds__(64 * S23_WAVES)
k_step3(TileOperands op, const int *__restrict__ Cptr, const int *__restrict__ Crow, const int *__restrict__ Ccol,
        int numtileC, const unsigned short *__restrict__ Cmask, const unsigned char *__restrict__ Cptr16,
        const int *__restrict__ Cnnz, unsigned char *__restrict__ Ccol8, double *__restrict__ Cval,
        int dense_min, int all_rows, const unsigned char *__restrict__ rowcls) {
    __shared__ double s_acc[S23_WAVES][64 * ACC_STRIDE];
    __shared__ unsigned short s_bm[S23_WAVES][64];
    __shared__ unsigned char s_bp[S23_WAVES][64];
    __shared__ int s_la[S23_WAVES][TILES_PER_WAVE][PAIR_LDS_MAX];
    __shared__ int s_lb[S23_WAVES][TILES_PER_WAVE][PAIR_LDS_MAX];
    const int wave = threadIdx.x >> 6;
    const long long nvb = ((long long)numtileC + S23_WAVES * TILES_PER_WAVE - 1) / (S23_WAVES * TILES_PER_WAVE);
    for (long long vb = tsg_xcd_block(blockIdx.x, gridDim.x); vb < nvb; vb += gridDim.x)
        step3_tile_body(op, Crow, Ccol, numtileC, Cmask, Cptr16, Cnnz, Ccol8, Cval, dense_min, all_rows, rowcls, vb,
                        s_acc[wave], s_bm[wave], s_bp[wave], s_la[wave], s_lb[wave]);
}

__device__ __forceinline__ void step3_tile_body(const TileOperands &op, const int *__restrict__ Crow,
                                                const int *__restrict__ Ccol, int numtileC,
                                                const unsigned short *__restrict__ Cmask,
                                                const unsigned char *__restrict__ Cptr16,
                                                const int *__restrict__ Cnnz, unsigned char *__restrict__ Ccol8,
                                                double *__restrict__ Cval, int dense_min, int all_rows,
                                                const unsigned char *__restrict__ rowcls, long long vblk,
                                                double *s_accw, unsigned short *s_bmw, unsigned char *s_bpw,
                                                int (*s_law)[PAIR_LDS_MAX], int (*s_lbw)[PAIR_LDS_MAX]) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = lane >> 4, r = lane & 15;
    const long long t = (vblk * S23_WAVES + wave) * TILES_PER_WAVE + g;
    if (t >= numtileC) return;
    const int coff = Cnnz[t], cn = Cnnz[t + 1] - coff;
    if (cn == 0) return;  // structurally empty tile (step-1 phantom)
    if (!all_rows && rowcls[Crow[t]] != 0) return;  // done by k_step3_rows or k_step3_lines
    const unsigned cm = Cmask[t * 16 + r];
    const int cp = Cptr16[t * 16 + r];
    const int rowlen = __popc(cm);
    const bool dense = cn >= dense_min;
    double *accg = &s_accw[g * 16 * ACC_STRIDE];  // 272 doubles per group
    double *accr = accg + r * ACC_STRIDE;          // dense: lane-private row
    if (dense) {
#pragma unroll
        for (int c = 0; c < 16; c++) accr[c] = 0.0;
    } else {
        for (int j = 0; j < rowlen; j++) accg[cp + j] = 0.0;
    }
    unsigned short *bmg = &s_bmw[g * 16];
    unsigned char *bpg = &s_bpw[g * 16];
    const int I = Crow[t], J = Ccol[t];
    for_each_pair(op, I, J, g, r, s_law[g], s_lbw[g], [&](int ta, int tb) {
        bmg[r] = op.Bmask[(long long)tb * 16 + r];
        bpg[r] = op.Bptr16[(long long)tb * 16 + r];
        tsg_wave_sync();
        const double *bval = op.Bval + op.Bnnz[tb];
        unsigned am = op.Amask[(long long)ta * 16 + r];
        const double *aval = op.Aval + op.Annz[ta] + op.Aptr16[(long long)ta * 16 + r];
        int ia = 0;
        while (am) {
            const int b = 31 - __clz(am);  // highest bit = smallest column k
            am &= ~(1u << b);
            const int k = 15 - b;
            const double a = aval[ia++];
            unsigned bm = bmg[k];
            const double *brow = bval + bpg[k];
            int jb = 0;
            while (bm) {
                const int bb = 31 - __clz(bm);
                bm &= ~(1u << bb);
                const double bv = brow[jb++];
                double *slot = dense ? &accr[15 - bb] : &accg[cp + __popc(cm >> (bb + 1))];
                *slot = __builtin_fma(a, bv, *slot);
            }
        }
        tsg_wave_sync();
    });
    // write out row r of the tile, ascending columns
    double *outv = Cval + coff + cp;
    unsigned char *outc = Ccol8 + coff + cp;
    unsigned x = cm;
    for (int j = 0; j < rowlen; j++) {
        const int bb = 31 - __clz(x);
        x &= ~(1u << bb);
        const int c = 15 - bb;
        outv[j] = dense ? accr[c] : accg[cp + j];
        outc[j] = (unsigned char)c;
    }
}

// ------------------------------------------------------------------ step 3, element-wise
// Segments of tile-rows the row-wise tile kernel cannot hold (too many C
// tiles, A tiles or B tiles, typically hypersparse rows where most tiles
// carry one or two nonzeros): element-level Gustavson with B's row index.
// One 256-thread block per segment (a run of C tiles holding <= G3E_NNZ
// nonzeros, accumulated in LDS in final order and located through an LDS
// hash of the segment's C entries); 16 groups of 16 lanes, group r owns C
// row 16I+r.  The group walks A row 16I+r in ascending k (A tiles in
// ascending K, bits in ascending column) and, for each a_ik, its lanes
// scatter the entries of B row k that fall in the segment's column range:
// distinct C entries per step, steps in ascending k, so each C entry again
// sums its products in the serial SPA order, without atomics.  Segments of
// 1536 nonzeros balance the re-walks of A rows per tile-row against the
// block's LDS (accumulator, hash, column bytes), which sets the blocks per
// CU in gfx950's 1,280-byte LDS granules.
#define G3E_NNZ 1536

// LDS hash of the segment's C entries: key (column - col_lo) * 16 + row,
// stored + 1 (0 = empty), value = the entry's position in the segment,
// linear probing.  2560 slots (load factor at most 0.6): six blocks per CU
// packed (25.6 KB of LDS), five unpacked (30.7 KB).
#define G3E_EHASH 2560
#define G3E_PF 4  // C tiles per thread whose metadata is loaded per round
// home slot of a key in a table of HS slots (multiply-shift range
// reduction) and the next slot
template <unsigned HS>
__device__ __forceinline__ unsigned ent_slot(unsigned key) {
    return (unsigned)(((unsigned long long)(key * 2654435761u) * HS) >> 32);
}
template <unsigned HS>
__device__ __forceinline__ unsigned ent_next(unsigned h) { return h + 1 == HS ? 0u : h + 1; }
// PK: when every tile-row spans fewer than 8192 tile columns the key (+1) is
// below 2^21 and one 32-bit slot holds key << 11 | position (positions are
// below G3E_NNZ <= 2048); without the separate position array the block's
// LDS fits six blocks per CU.
#define G3E_PK_SPAN 8192
static_assert(G3E_NNZ <= 2048, "positions take 11 bits of a packed hash slot");

// For an A without its row index (its rows' entries are decoded from its
// tiles); with it, k_step3_flat takes these tile-rows.
template <bool PK>
__global__ void __launch_bounds__(256, PK ? 6 : 5)
k_step3_elem(TileOperands op, const int *__restrict__ Browp, const int *__restrict__ Bcolx,
             const double *__restrict__ Bvalx, int m, const int4 *__restrict__ segs, const int *__restrict__ nseg,
             const int *__restrict__ Cptr, const int *__restrict__ Ccol, const unsigned short *__restrict__ Cmask,
             const unsigned char *__restrict__ Cptr16, const int *__restrict__ Cnnz, unsigned char *__restrict__ Ccol8,
             double *__restrict__ Cval) {
    __shared__ double s_acc[G3E_NNZ];
    constexpr unsigned HS = G3E_EHASH;
    __shared__ unsigned s_ekey[HS];
    __shared__ unsigned short s_epos[PK ? 1 : HS];
    __shared__ unsigned char s_ecol[G3E_NNZ];  // in-tile column of each entry, final order
    const int tid = threadIdx.x;
    // the grid is an upper bound: the first *nseg blocks (spread evenly over
    // the XCDs) take the segments, each XCD a contiguous range
    const int ns = *nseg;
    const unsigned blk = tsg_block();
    if (blk >= (unsigned)ns) return;  // block-uniform
    const int w = (int)tsg_xcd_block(blk, (unsigned)ns);
    const int4 sg = segs[w];
    const int I = sg.x;
    const int c0 = Cptr[I] + sg.y, u = sg.z - sg.y;
    const int nbase = Cnnz[c0], nseg_nnz = Cnnz[c0 + u] - nbase;
    const int col_lo = Ccol[c0] * 16, col_hi = Ccol[c0 + u - 1] * 16 + 16;
    for (int i = tid; i < nseg_nnz; i += 256) s_acc[i] = 0.0;
    for (int i = tid; i < (int)HS; i += 256) s_ekey[i] = 0u;
    __syncthreads();
    // every C entry of the segment into the hash, and its in-tile column
    // into s_ecol (one C tile per thread; structurally empty tiles skipped).
    // The metadata of up to G3E_PF of a thread's tiles is loaded in one
    // round before their entries are inserted.
    for (int i0 = 0; i0 < u; i0 += 256 * G3E_PF) {
        int pos0[G3E_PF], nt[G3E_PF];
        unsigned j16[G3E_PF];
        uint4 mA[G3E_PF], mB[G3E_PF];
#pragma unroll
        for (int v = 0; v < G3E_PF; v++) {
            const int i = i0 + v * 256 + tid;
            nt[v] = 0;
            if (i < u) {
                const long long t = c0 + i;
                pos0[v] = Cnnz[t] - nbase;
                nt[v] = Cnnz[t + 1] - Cnnz[t];
                const uint4 *cm4 = reinterpret_cast<const uint4 *>(Cmask + t * 16);
                mA[v] = cm4[0];
                mB[v] = cm4[1];
                j16[v] = (unsigned)(Ccol[t] * 16 - col_lo);
            }
        }
#pragma unroll
        for (int v = 0; v < G3E_PF; v++) {
            if (nt[v] == 0) continue;
            const unsigned mw[8] = {mA[v].x, mA[v].y, mA[v].z, mA[v].w, mB[v].x, mB[v].y, mB[v].z, mB[v].w};
            int pos = pos0[v];
            for (int rr = 0; rr < 16; rr++) {  // rows in order: positions follow
                unsigned cm = (mw[rr >> 1] >> ((rr & 1) * 16)) & 0xffffu;
                while (cm) {
                    const int bb = 31 - __clz(cm);
                    cm &= ~(1u << bb);
                    const unsigned key = (((j16[v] + 15 - bb) << 4) | (unsigned)rr) + 1u;
                    unsigned h = ent_slot<HS>(key);
                    if (PK) {
                        const unsigned ent = key << 11 | (unsigned)pos;
                        while (atomicCAS(&s_ekey[h], 0u, ent) != 0u) h = ent_next<HS>(h);
                    } else {
                        while (atomicCAS(&s_ekey[h], 0u, key) != 0u) h = ent_next<HS>(h);  // nnz < HS
                        s_epos[h] = (unsigned short)pos;
                    }
                    s_ecol[pos] = (unsigned char)(15 - bb);
                    pos++;
                }
            }
        }
    }
    __syncthreads();
    const int r = tid >> 4, l = tid & 15;
    const int row = 16 * I + r;
    const int gb = tid & 48;  // first lane of this group in its wave
    __shared__ int s_gex[16][16];             // per group: entries before each lane's tile
    __shared__ unsigned short s_gam[16][16];  // per group: each lane's tile row mask
    // adds a * b into C entry (row 16I+r, col), located through the hash
    // (the entry is in C's structure; the probe bound is not reached for a
    // consistent C)
    auto acc_add = [&](int col, double a, double b) {
        const unsigned key = ((unsigned)(col - col_lo) << 4 | (unsigned)r) + 1u;
        unsigned h = ent_slot<HS>(key);
        int probe = 0;
        if (PK) {
            unsigned ent;
            while (((ent = s_ekey[h]) >> 11) != key && ++probe < (int)HS) h = ent_next<HS>(h);
            if (probe < (int)HS) {
                double *acc = &s_acc[ent & 2047u];
                *acc = __builtin_fma(a, b, *acc);
            }
        } else {
            while (s_ekey[h] != key && ++probe < (int)HS) h = ent_next<HS>(h);
            if (probe < (int)HS) {
                double *acc = &s_acc[s_epos[h]];
                *acc = __builtin_fma(a, b, *acc);
            }
        }
    };
    if (row < m && nseg_nnz > 0) {
        const int a0 = op.Aptr[I], a1 = op.Aptr[I + 1];
        for (int t0 = a0; t0 < a1; t0 += 16) {
            // 16 A tiles per round, one per lane: their row-r entries are
            // numbered x = 0..total-1 in ascending k (tiles in ascending K,
            // columns ascending inside a tile)
            const int tl = t0 + l;
            const unsigned am_l = tl < a1 ? op.Amask[(long long)tl * 16 + r] : 0u;
            const int cnt = __popc(am_l);
            int incl = cnt;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                const int v = __shfl_up(incl, o, 16);
                if (l >= o) incl += v;
            }
            const int total = __shfl(incl, 15, 16);
            s_gex[r][l] = incl - cnt;
            s_gam[r][l] = (unsigned short)am_l;
            tsg_wave_sync();
            for (int x0 = 0; x0 < total; x0 += 16) {
                // lane l takes entry x0 + l and finds its B range in parallel
                const int x = x0 + l;
                int k = 0, e0 = 0, e1 = 0;
                double a = 0.0;
                bool have = false;
                if (x < total) {
                    int ow = 0;
#pragma unroll
                    for (int st = 8; st > 0; st >>= 1)
                        if (ow + st < 16 && s_gex[r][ow + st] <= x) ow += st;
                    unsigned am = s_gam[r][ow];
                    int j = x - s_gex[r][ow];  // j-th entry of the owner's row
                    for (int q = 0; q < j; q++) am &= ~(1u << (31 - __clz(am)));
                    const int b = 31 - __clz(am);
                    const int t = t0 + ow;
                    k = op.Acol[t] * 16 + 15 - b;
                    a = op.Aval[op.Annz[t] + op.Aptr16[(long long)t * 16 + r] + j];
                    e1 = Browp[k + 1];
                    e0 = lower_bound_i(Bcolx, Browp[k], e1, col_lo);
                    have = e0 < e1 && Bcolx[e0] < col_hi;
                }
                unsigned hv = (unsigned)(__ballot(have) >> gb) & 0xffffu;
                while (hv) {  // entries with B entries in range, ascending k
                    const int src = __ffs(hv) - 1;
                    hv &= hv - 1;
                    const double as = __shfl(a, gb + src, 64);
                    const int es0 = __shfl(e0, gb + src, 64), es1 = __shfl(e1, gb + src, 64);
                    for (int e = es0 + l; e < es1; e += 16) {
                        const int col = Bcolx[e];
                        if (col >= col_hi) break;
                        acc_add(col, as, Bvalx[e]);
                    }
                    tsg_wave_sync();  // the next k of this row reads what lanes wrote
                }
            }
            tsg_wave_sync();  // s_gex / s_gam are rewritten next round
        }
    }
    __syncthreads();
    for (int i = tid; i < nseg_nnz; i += 256) {
        Cval[(long long)nbase + i] = s_acc[i];
        Ccol8[(long long)nbase + i] = s_ecol[i];
    }
}

// ------------------------------------------------------------------ step 3, flat rows
// One product per lane, of sources q0 (lane 0's) to q1 in ascending k along the
// lanes, into sums that products of different sources may share: each lane
// leaves its number at its sum and reads it back, and if some lane finds
// another's the sources are added one by one.
__device__ __forceinline__ void add_in_order(double *sum, unsigned char *tag, bool on, int q, int lane, double a,
                                             double b) {
    const int q0 = __builtin_amdgcn_readlane(q, 0), q1 = __builtin_amdgcn_readlane(q, 63);
    bool clash = false;
    if (q0 != q1) {
        if (on) *tag = (unsigned char)lane;
        tsg_wave_sync();
        clash = __ballot(on && *tag != (unsigned char)lane) != 0;
    }
    if (!clash) {
        if (on) *sum = __builtin_fma(a, b, *sum);
    } else {
        for (int s = q0; s <= q1; s++) {
            if (on && q == s) *sum = __builtin_fma(a, b, *sum);
            tsg_wave_sync();
        }
    }
    tsg_wave_sync();
}
// [b0, b1) cut to list's entries in [lo, hi) (list ascending; an end that is
// not to be cut keeps its place).  Both ends at once and a quarter of the
// range left per step, six loads in flight: a lane's search is a chain of
// round trips, so their number is what it costs.
__device__ __forceinline__ void range_in(const int *__restrict__ list, int &b0, int &b1, bool cut_lo, int lo,
                                         bool cut_hi, int hi) {
    int la = b0, na = cut_lo ? b1 - b0 : 0;  // first entry >= lo is in [la, la + na]
    int lb = b0, nb = cut_hi ? b1 - b0 : 0;  // first entry >= hi is in [lb, lb + nb]
    if (!cut_hi) lb = b1;
    while (na > 0 || nb > 0) {
        int pa[3], pb[3], va[3], vb[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            pa[i] = (int)(((unsigned long long)(unsigned)na * (i + 1)) >> 2);  // < na when na > 0
            pb[i] = (int)(((unsigned long long)(unsigned)nb * (i + 1)) >> 2);
            va[i] = na > 0 ? list[la + pa[i]] : 0;
            vb[i] = nb > 0 ? list[lb + pb[i]] : 0;
        }
        if (na > 0) {
            const int k = (va[0] < lo) + (va[1] < lo) + (va[2] < lo);
            const int from = k == 0 ? 0 : (k == 1 ? pa[0] : k == 2 ? pa[1] : pa[2]) + 1;
            const int to = k == 0 ? pa[0] : k == 1 ? pa[1] : k == 2 ? pa[2] : na;
            la += from;
            na = to - from;
        }
        if (nb > 0) {
            const int k = (vb[0] < hi) + (vb[1] < hi) + (vb[2] < hi);
            const int from = k == 0 ? 0 : (k == 1 ? pb[0] : k == 2 ? pb[1] : pb[2]) + 1;
            const int to = k == 0 ? pb[0] : k == 1 ? pb[1] : k == 2 ? pb[2] : nb;
            lb += from;
            nb = to - from;
        }
    }
    b0 = la;
    b1 = max(lb, la);
}
// Element-wise numeric step with A's and B's row index: one block of eight
// waves per segment of a tile-row (k_seg1_count; at most G3F_NNZ C nonzeros,
// summed in LDS in final order).
//   Hash.  Each row of the segment has its own table of one and a half slots
//   per entry: column offset (20 bits, + 1) and position (12) in one word, in
//   two with WIDE.  Entries are inserted one per lane, their tile from marks,
//   their row from the tile's row offsets, their column from the row mask:
//   a lane per tile walking its masks had 6 of 64 lanes inserting (54k VALU
//   instructions a tile-row of ER 65521, 42k now).
//   Products.  A wave owns two rows, a long one and a short one.  It takes up
//   to 64 of their A entries (sources) at a time, cuts their B rows to the
//   segment's columns, numbers the products through in ascending k and takes
//   64 at a time, one per lane.  Two of them can meet in one C entry only if
//   they come from different sources: each lane leaves its number at its
//   entry and reads it back, and a batch in which some lane finds another's
//   is added source by source.  So every C entry still sums its products in
//   ascending k, without atomics.
// Four blocks (32 waves) fit a CU; it is bound by the latency of each block's
// phases (waves wait 72% of their cycles) and by VALU (busy 59%, ER 65521).  Against 16 lanes per C row taking one
// source at a time (4.5 entries of a source in a segment of ER 65521), a
// search per source and segment of 1536: ER 65521 A^2 0.62 -> 0.545 ms, banded
// 39989 (half-bandwidth 20) 0.29 -> 0.167, R-MAT scale 16 A*A^T 12.9 -> 7.7.
// Segments of 1920 / 2048 / 2496 / 3200 nonzeros: ER 573 / 533 / 545 / 579 us,
// R-MAT 8.4 / 8.2 / 7.7 / 8.8 ms.
#define G3F_NNZ 2496
#define G3F_THREADS 512
#define G3F_WAVES (G3F_THREADS / 64)
#define G3F_SLOTS (G3F_NNZ + G3F_NNZ / 2 + 32)
#define G3F_ROUNDS 4
#define G3F_BATCH (64 * G3F_ROUNDS)
#define G3F_SPAN 65535  // tile columns of a tile-row: offsets + 1 below 2^20
__device__ __forceinline__ unsigned flat_home(unsigned key, unsigned n) {
    return (unsigned)(((unsigned long long)(key * 2654435761u) * n) >> 32);
}
template <bool WIDE>
__global__ void __launch_bounds__(G3F_THREADS)
k_step3_flat(const int *__restrict__ Arowp, const int *__restrict__ Acolx, const double *__restrict__ Avalx,
             const int *__restrict__ Browp, const int *__restrict__ Bcolx, const double *__restrict__ Bvalx, int m,
             const int4 *__restrict__ segs, const int *__restrict__ nseg, const int *__restrict__ Cptr,
             const int *__restrict__ Ccol, const unsigned short *__restrict__ Cmask,
             const unsigned char *__restrict__ Cptr16, const int *__restrict__ Cnnz, unsigned char *__restrict__ Ccol8,
             double *__restrict__ Cval, const unsigned char *__restrict__ heavy) {
    __shared__ double s_acc[G3F_NNZ];
    __shared__ unsigned s_key[G3F_SLOTS];
    __shared__ unsigned short s_pos[WIDE ? G3F_SLOTS : 1];
    __shared__ unsigned char s_tag[G3F_NNZ];
    __shared__ unsigned s_mark[G3F_WAVES][G3F_BATCH / 4];
    __shared__ int s_cnt[G3F_WAVES][16], s_rb[17];
    __shared__ unsigned char s_ord[16];
    static_assert(G3F_NNZ <= 4096, "positions take 12 bits of a slot");
    static_assert(G3F_NNZ >= G3E_NNZ, "the segment array is sized for segments of G3E_NNZ");
    static_assert(G3F_WAVES == 8, "two rows per wave");
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    // the grid is an upper bound: the first *nseg blocks (spread evenly over
    // the XCDs) take the segments, each XCD a contiguous range
    const int ns = *nseg;
    const unsigned blk = tsg_block();
    if (blk >= (unsigned)ns) return;  // block-uniform
    const int4 sg = segs[tsg_xcd_block(blk, (unsigned)ns)];
    const int I = sg.x, cend = Cptr[I + 1];
    const int c0 = Cptr[I] + sg.y, u = sg.z - sg.y;
    const int nbase = Cnnz[c0], n = Cnnz[c0 + u] - nbase;
    if (n == 0) return;  // block-uniform
    const int col_lo = Ccol[c0] * 16, col_hi = Ccol[c0 + u - 1] * 16 + 16;
    const bool first = sg.w == 0, last = c0 + u == cend;
    for (int i = tid; i < n; i += G3F_THREADS) s_acc[i] = 0.0;
    for (int i = tid; i < n + n / 2 + 32; i += G3F_THREADS) s_key[i] = 0u;
    // entries of each row of the segment; rows left to k_step3_heavy take no slots
    unsigned skip = 0;
    if (heavy) {
        const int row = 16 * I + (lane & 15);
        skip = (unsigned)__ballot(row < m && heavy[row]) & 0xffffu;
    }
    {
        unsigned v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = 0u;
        for (int i = tid; i < u; i += G3F_THREADS) {
            const long long t = c0 + i;
            unsigned x[8];
            tile_widen_lens(tile_row_lens(reinterpret_cast<const uint4 *>(Cptr16)[t], Cnnz[t + 1] - Cnnz[t]), x);
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] += x[q];
        }
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = (unsigned)__builtin_amdgcn_readlane(tsg_wave_incl_scan_dpp((int)v[q]), 63);
        if (lane < 16) s_cnt[wave][lane] = tile_row_of(v, lane);
    }
    __syncthreads();
    if (tid < 16) {
        int c = 0;
        for (int w = 0; w < G3F_WAVES; w++) c += s_cnt[w][tid];
        if ((skip >> tid) & 1u) c = 0;
        const int slots = c ? c + c / 2 + 2 : 0;
        const int incl = tsg_row16_incl_scan_dpp(slots);
        s_rb[tid] = incl - slots;
        if (tid == 15) s_rb[16] = incl;
        int rank = 0;  // by entries, longest first
        for (int j = 0; j < 16; j++) {
            const int cj = __builtin_amdgcn_readlane(c, j);
            rank += cj > c || (cj == c && j < tid);
        }
        s_ord[rank] = (unsigned char)tid;
    }
    __syncthreads();
    // the segment's entries into their rows' tables, their columns to memory
    unsigned char *mk = reinterpret_cast<unsigned char *>(s_mark[wave]);
    const int per = min(64, (u + G3F_WAVES - 1) / G3F_WAVES);  // few, fuller tiles: every wave has some
    for (int tg = per * wave; tg < u; tg += per * G3F_WAVES) {
        const int te = min(u, tg + per);
        for (int tb = tg; tb < te;) {
            const long long tl = c0 + min(tb + lane, te - 1);
            const int n0 = Cnnz[tl] - nbase, n1 = Cnnz[tl + 1] - nbase, Jl = Ccol[tl];
            const int start = __builtin_amdgcn_readfirstlane(n0);
            const int nt = __popcll(__ballot(tb + lane < te && n1 - start <= G3F_BATCH));
            const int total = __builtin_amdgcn_readlane(n1, nt - 1) - start;
            if (total > 0) {
                s_mark[wave][lane] = 0u;
                tsg_wave_sync();
                if (lane < nt && n1 > n0) mk[n0 - start] = (unsigned char)(lane + 1);
                tsg_wave_sync();
                int prev = 0;
                for (int x0 = 0; x0 < total; x0 += 64) {
                    const int x = x0 + lane;
                    const int k = max(prev, tsg_wave_incl_max_dpp((int)mk[x])) - 1;
                    prev = __builtin_amdgcn_readlane(k, 63) + 1;
                    const long long t = c0 + tb + k;
                    const int j = x - (__shfl(n0, k, 64) - start), J = __shfl(Jl, k, 64);
                    const uint4 p = reinterpret_cast<const uint4 *>(Cptr16)[t];
                    const int r = __popc(bytes_le(p.x, j & 255)) + __popc(bytes_le(p.y, j & 255)) +
                                  __popc(bytes_le(p.z, j & 255)) + __popc(bytes_le(p.w, j & 255)) - 1;
                    unsigned mr = Cmask[t * 16 + r];
                    const unsigned pw = (r & 8) ? ((r & 4) ? p.w : p.z) : ((r & 4) ? p.y : p.x);
                    int skipn = j - (int)((pw >> (8 * (r & 3))) & 255u);
                    if (x < total && !((skip >> r) & 1u)) {  // (k_step3_heavy writes its rows' columns)
                        // entry j of the tile: the (j - row offset)-th column of row r
                        for (; skipn > 0; skipn--) mr &= ~(0x80000000u >> __clz((int)mr));
                        const int c = __clz((int)mr) - 16, pos = start + x, rb = s_rb[r];
                        Ccol8[(long long)nbase + pos] = (unsigned char)c;
                        const unsigned rs = (unsigned)(s_rb[r + 1] - rb), key = (unsigned)(J * 16 + c - col_lo) + 1u;
                        unsigned h = flat_home(key, rs);
                        const unsigned ent = WIDE ? key : key << 12 | (unsigned)pos;
                        while (atomicCAS(&s_key[rb + h], 0u, ent) != 0u) h = h + 1 == rs ? 0u : h + 1;
                        if (WIDE) s_pos[rb + h] = (unsigned short)pos;
                    }
                }
                tsg_wave_sync();
            }
            tb += nt;
        }
    }
    __syncthreads();
    // two rows per wave, a long one with a short one; their A entries (row ra's
    // first) are taken together, so products of both share a batch.  Rows
    // without entries here, or left to k_step3_heavy, are not walked.
    const int ra = s_ord[wave], rz = s_ord[15 - wave];
    int xa = 0, na = 0, xz = 0, nz = 0;
    if (s_rb[ra + 1] > s_rb[ra]) {
        xa = Arowp[min(16 * I + ra, m)];
        na = Arowp[min(16 * I + ra + 1, m)] - xa;
    }
    if (s_rb[rz + 1] > s_rb[rz]) {
        xz = Arowp[min(16 * I + rz, m)];
        nz = Arowp[min(16 * I + rz + 1, m)] - xz;
    }
    for (int xc = 0; xc < na + nz; xc += 64) {
        int b0 = 0, len = 0, rb = 0, rs = 0;
        double a = 0.0;
        if (xc + lane < na + nz) {
            const bool z = xc + lane >= na;
            const int x = z ? xz + (xc + lane - na) : xa + xc + lane, r = z ? rz : ra;
            const int k = Acolx[x];
            a = Avalx[x];
            b0 = Browp[k];
            int b1 = Browp[k + 1];
            rb = s_rb[r];
            rs = s_rb[r + 1] - rb;
            range_in(Bcolx, b0, b1, !first, col_lo, !last, col_hi);
            len = b1 - b0;
        }
        const int incl = tsg_wave_incl_scan_dpp(len), pre = incl - len, delta = b0 - pre, reg = rb | rs << 16;
        const int total = __builtin_amdgcn_readlane(incl, 63);
        int prev = 0;
        for (int base = 0; base < total; base += G3F_BATCH) {
            s_mark[wave][lane] = 0u;
            tsg_wave_sync();
            if (len > 0 && pre >= base && pre < base + G3F_BATCH) mk[pre - base] = (unsigned char)(lane + 1);
            tsg_wave_sync();
            int q[G3F_ROUNDS], col[G3F_ROUNDS];
            double b[G3F_ROUNDS];
#pragma unroll
            for (int i = 0; i < G3F_ROUNDS; i++) {
                q[i] = max(prev, tsg_wave_incl_max_dpp((int)mk[64 * i + lane]));
                prev = __builtin_amdgcn_readlane(q[i], 63);
            }
#pragma unroll
            for (int i = 0; i < G3F_ROUNDS; i++) {  // every lane loads in bounds
                const int e = __shfl(delta, q[i] - 1, 64) + min(base + 64 * i + lane, total - 1);
                col[i] = Bcolx[e];
                b[i] = Bvalx[e];
            }
#pragma unroll
            for (int i = 0; i < G3F_ROUNDS; i++) {
                if (base + 64 * i >= total) break;  // wave-uniform
                const bool on = base + 64 * i + lane < total;
                const double as = __shfl(a, q[i] - 1, 64);
                const int rg = __shfl(reg, q[i] - 1, 64);
                const unsigned *key0 = s_key + (rg & 0xffff);
                const unsigned n_r = (unsigned)rg >> 16, key = (unsigned)(col[i] - col_lo) + 1u;
                unsigned h = flat_home(key, n_r), ent;
                unsigned probe = 0;
                // (the entry is in C's structure: the probe bound is not reached)
                while ((ent = key0[h], WIDE ? ent : ent >> 12) != key && ++probe < n_r) h = h + 1 == n_r ? 0u : h + 1;
                const int pos = WIDE ? (int)s_pos[(rg & 0xffff) + h] : (int)(ent & 4095u);
                add_in_order(s_acc + pos, s_tag + pos, on, q[i], lane, as, b[i]);
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < n; i += G3F_THREADS) Cval[(long long)nbase + i] = s_acc[i];
}

// ------------------------------------------------------------------ step 3, heavy and long rows
// Rows with many products for the columns of their tile-row (hub rows of
// power-law graphs, and rows that have a few hubs as sources).  In segments
// of a tile-row each would walk all its A entries again in every segment
// and put every entry of C into a hash first (R-MAT scale 16: 68 segments a
// tile-row, 9,800 VALU instructions each).  Here a wave takes one row and a group
// of column parts (HEAVY_PART_COLS columns each; a heavy row one part, so that
// a hub row spreads over many waves, a long row HEAVY_GROUP parts).  It takes
// as many parts at a time as the row's entries in them fit its sums, writes
// for each tile the row's mask and its offset among the sums, walks A row i in
// ascending k, 64 entries (sources) at a time, numbers the products with the B
// entries in these parts through and adds 64 per step (add_in_rounds), then
// copies the sums to C's final positions with their column bytes.
//   Where B row k's entries of a part start and end is read from a table
// made once per product (k_heavy_windows), two groups of sources ahead, so no
// search stands between the loads; blocks go part by part, which keeps the
// parts' columns of B (and of the table) in the L2.  A row's parts are those from
// the first to the last that its tile-row reaches, and it has as many blocks as
// twice the mean asks for, each taking its parts in strides of that: over all parts of
// B a random band (1,000,000 rows, half-width 2000, 24 per row) had 244 million
// blocks for 2.6 million with work, 118.5 ms, now 22.0; 128 diagonal blocks of ER
// 8000 (24 per row) 125 -> 25.6, R-MAT scale 16 10.76 -> 10.78.
//   14 KiB of LDS, eleven waves a CU.  Bound by products behind LDS round
// trips and fragments of B rows (5.1 of 8.4 ms), scattered 8-byte stores (2)
// and the walk over tiles (1.4): L1 taken in 54% of its cycles, VALU busy 36%, LDS
// 31%, 2.6 TB/s of HBM.  R-MAT scale 16 A*A^T, heavy rows with the
// others by k_step3_flat 13.9 ms -> all by this kernel 7.1.  Parts of 1024 in
// groups of 4 / 8 / 16 (whole product) 11.0 / 11.7 / 11.9 ms, of 2048 in groups
// of 2 / 4 / 8 12.1 / 11.8 / 12.0, of 512 in groups of 8 12.1.
#define HEAVY_MIN_PRODUCTS 65536  // reported as heavy (tsg_stats.heavy_rows)
#define HEAVY_PART_LOG 10
#define HEAVY_PART_COLS (1 << HEAVY_PART_LOG)
#define HEAVY_PART_TILES (1 << (HEAVY_PART_LOG - 4))
#define HEAVY_GROUP 4
// A row is split into single parts above C's nonzeros >> 10 products: one
// wave's share of everything, so that no wave ends long after the others.  R-MAT
// A*A^T with 16384 / 65536 / 262144: scale 16 (380 M nonzeros) 12.3 / 11.8 /
// 11.0 ms, scale 14 (30 M) 2.22 / 2.19 / 2.44.
#define HEAVY_SPLIT_LOG 10
#define HEAVY_SPLIT_MAX 262144LL
#define HEAVY_WINDOW_BYTES (512ll << 20)  // largest window table
#define HEAVY_WINDOWS_MAX 65535  // k_heavy_windows has one per grid row (reached with few rows of B and 2^26 columns)
// All rows of a tile-row with more products per row than LONG_MIN_PRODUCTS, and
// than LONG_PER_GROUP for every group of parts that its columns span, go here:
// below, a wave per row and group walks the row's sources and tiles for few
// products and k_step3_flat is better.  What counts is the products a wave gets,
// not the row's against its tiles (more than half as many products as tiles):
// random tiles of 48 entries, 8 a tile-row, 575 products a row, over 12 groups
// 1.16 ms, over 24 groups (96000 rows) 3.76, by k_step3_flat 0.56 and 0.97;
// 24 tiles of 24 entries, 1290 products over 24 groups 5.10 / 2.63 ms; over 8
// groups, 164 a wave, 0.86 / 0.90.  With 100 / 160 / 220 / 320: random tiles (8
// of 64 entries, 116 a wave) 0.81 / 0.58 / 0.58 / 0.58 ms, ER 30000 (40 per row,
// 218 a wave) 1.27 / 1.26 / 1.41 / 1.47, R-MAT scale 16 A*A^T 11.1 / 10.9 / 10.9 / 11.2.
#define LONG_MIN_PRODUCTS 512
#define LONG_PER_GROUP 160
// Only in a large product (or when the caller sets heavy_min_products): in a
// small one the waves of the longest rows end after everything else.  R-MAT
// A^2 with / without long rows: scale 11 (6 edges a vertex) 410 / 353 us, scale 12
// 652 / 563, scale 13 (7 M nonzeros) 1210 / 1192; scale 14 A*A^T (30 M) 2.2 / 2.9 ms.
#define LONG_MIN_NNZ (12LL << 20)
#define CLS_LONG 3  // row class: heavy and long rows only

// Per C row of an element-wise tile-row: 2 heavy (more than min_products
// products, or more than 2048 A entries), 1 long, 0 neither; cnt[0, m) and cnt[m,
// 2m) take the heavy and the long rows as counts for the scan that numbers
// them, info[0] the number of heavy ones, info[2] and [3] the long tile-rows'
// entries of C and their number, info[4..5] the sum of the groups of parts they
// reach, info[6..7] that of the parts which the heavy rows reach.  A tile-row
// with many products for its columns has only heavy and long rows and leaves
// the element-wise class.
// One block per tile-row, 16 lanes per row, so that a long A row's B row
// lengths are not one lane's chain of loads (R-MAT scale 16: 665 -> 92 us).
__global__ void __launch_bounds__(256)
k_heavy_flags(const int *__restrict__ Arowp, const int *__restrict__ Acolx, const int *__restrict__ Browp,
              unsigned char *__restrict__ rowcls, const int *__restrict__ Cptr, const int *__restrict__ Ccol,
              const int *__restrict__ Cnnz, int tilem, int m,
              long long min_products, long long count_products, int take_long, unsigned char *__restrict__ flag, int *__restrict__ cnt,
              int *__restrict__ info) {
    __shared__ long long s_p[16];
    const int I = (int)tsg_block(), r = threadIdx.x >> 4, l = threadIdx.x & 15, i = 16 * I + r;
    if (I >= tilem) return;  // block-uniform
    const bool mine = rowcls[I] == 0;  // block-uniform
    long long p = 0;
    int x0 = 0, x1 = 0;
    if (mine && i < m) {
        x0 = Arowp[i];
        x1 = Arowp[i + 1];
#pragma unroll 4
        for (int x = x0 + l; x < x1; x += 16) {
            const int k = Acolx[x];
            p += Browp[k + 1] - Browp[k];
        }
        p = tsg_group16_sum(p);
    }
    if (l == 0) s_p[r] = p;
    __syncthreads();
    long long all = 0;
    for (int q = 0; q < 16; q++) all += s_p[q];
    bool longer = mine && take_long && all > 16 * LONG_MIN_PRODUCTS;
    if (longer) {
        const int span = Ccol[Cptr[I + 1] - 1] - Ccol[Cptr[I]] + 1;  // tile columns
        longer = all * (HEAVY_GROUP * HEAVY_PART_TILES) > 16LL * LONG_PER_GROUP * span;
    }
    const int h = !mine ? 0 : x1 - x0 > 2048 || p > min_products ? 2 : longer && p > 0 ? 1 : 0;
    if (i < m && l == 0) {
        flag[i] = (unsigned char)h;
        cnt[i] = h == 2;
        cnt[m + i] = h == 1;
    }
    if (!mine) return;  // block-uniform
    // the block's share of info, which every block adds to: one atomic a word
    const int heavy = __syncthreads_count(l == 0 && h == 2);
    const int counted = __syncthreads_count(l == 0 && (x1 - x0 > 2048 || p > count_products));
    if (threadIdx.x == 0 && (heavy || longer)) {
        const int parts = Ccol[Cptr[I + 1] - 1] / HEAVY_PART_TILES - Ccol[Cptr[I]] / HEAVY_PART_TILES + 1;
        unsigned long long *sums = reinterpret_cast<unsigned long long *>(info + 2);
        if (longer) {
            rowcls[I] = CLS_LONG;
            // entries that need no segments
            atomicAdd(sums, 1ULL << 32 | (unsigned)(Cnnz[Cptr[I + 1]] - Cnnz[Cptr[I]]));
            atomicAdd(sums + 1, (unsigned long long)((parts + HEAVY_GROUP - 1) / HEAVY_GROUP));
        }
        if (heavy) {
            atomicAdd(&info[0], heavy);
            atomicAdd(sums + 2, (unsigned long long)heavy * parts);
        }
    }
    if (threadIdx.x == 0 && counted) atomicAdd(&info[1], counted);
}

// rows = the heavy rows, then the long ones, each with the parts [y, z) that its
// tile-row reaches
__global__ void __launch_bounds__(256)
k_heavy_list(const int *__restrict__ off, const unsigned char *__restrict__ flag, int m, const int *__restrict__ Cptr,
             const int *__restrict__ Ccol, int4 *__restrict__ rows) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m || !flag[i]) return;
    rows[off[flag[i] == 2 ? i : m + i]] =
        make_int4(i, Ccol[Cptr[i >> 4]] / HEAVY_PART_TILES, Ccol[Cptr[(i >> 4) + 1] - 1] / HEAVY_PART_TILES + 1, 0);
}

// win[w * m + k] = first entry of B row k at or past column w << shift, w = 0
// .. nw (the last one the row's end).  k along the threads: neighbours search
// neighbouring rows and write one run.
__global__ void __launch_bounds__(256)
k_heavy_windows(const int *__restrict__ Browp, const int *__restrict__ Bcolx, int m, int nw, int shift,
                int *__restrict__ win) {
    const int k = blockIdx.x * 256 + threadIdx.x, w = blockIdx.y;
    if (k >= m) return;
    const int b0 = Browp[k], b1 = Browp[k + 1];
    win[(long long)w * m + k] = w == nw ? b1 : w == 0 ? b0 : lower_bound_i(Bcolx, b0, b1, w << shift);
}

// First of list[lo, hi) (ascending, the same for the whole wave) at or past
// key: 64 probes a step, two steps for 4096 entries.
__device__ __forceinline__ int wave_lower_bound(const int *__restrict__ list, int lo, int hi, int key, int lane) {
    while (lo < hi) {
        const int step = (hi - lo + 63) >> 6, x = lo + lane * step;
        const int below = __popcll(__ballot(x < hi && list[min(x, hi - 1)] < key));
        if (below == 0) return lo;
        hi = min(hi, lo + below * step);
        lo += (below - 1) * step + 1;
    }
    return lo;
}

// One product per lane, in ascending k along the lanes, into sums of which
// several lanes may share one (a lane's bin decides: equal sums, equal bins).
// In each round the lowest pending lane of a bin adds, so a shared sum gets
// its products in lane order.  The winner is the bin's minimum of stamp + lane;
// stamps descend, so bins need no clearing between rounds.  Against
// add_in_order: R-MAT scale 16 A*A^T 7.65 -> 7.07 ms in k_step3_heavy, whose rows
// meet many short sources, but scale 13 A^2 344 -> 400 us in k_step3_flat.
__device__ __forceinline__ void add_in_rounds(double *sum, unsigned *bin, unsigned &stamp, bool on, int lane, double a,
                                             double b) {
    for (;;) {
        stamp -= 64u;
        const unsigned me = stamp + (unsigned)lane;
        if (on) atomicMin(bin, me);
        tsg_wave_sync();
        const unsigned first = *bin;
        const double v = *sum;  // with the bin: one LDS round trip a round
        if (on && first == me) {
            *sum = __builtin_fma(a, b, v);
            on = false;
        }
        tsg_wave_sync();
        if (!__ballot(on)) break;
    }
}
// Blocks of one part: the list in steps of 128 rows (8 XCDs of 16); fewer rows
// than that as they are, with no block but theirs: one that only ends takes its
// XCD some 40 ns (1,000,000 diagonal entries and one row of 3000, whose row alone
// comes here, 977 parts: A^2 8.09 ms in 125,000 blocks, 7.54 in 977).
__host__ __device__ inline int heavy_padded(int nrows) { return nrows < 128 ? nrows : (nrows + 127) & ~127; }
// Long rows taken part by part together: all of them where they reach most of
// B's parts, else this many (then neighbouring rows share B rows, not parts).
// All / 1024: R-MAT scale 16 11.06 / 11.40 ms, block-diagonal ER (24 of 20000, 32 per
// row) 21.1 / 19.2, random band (300,000 rows, half-width 4000, 64 per row) 14.6 / 14.5.
#define LONG_CHUNK 1024
#define HEAVY_ROUNDS 4
#define HEAVY_BINS 256  // of add_in_rounds; products of different sums that share one only take a round more
#define HEAVY_BATCH (64 * HEAVY_ROUNDS)
__global__ void __launch_bounds__(64)
k_step3_heavy(const int *__restrict__ Arowp, const int *__restrict__ Acolx, const double *__restrict__ Avalx,
              const int *__restrict__ win, long long wstride, int nw, int shift, const int *__restrict__ Bcolx,
              const double *__restrict__ Bvalx, const int4 *__restrict__ rows, int nheavy, int nlong,
              int hstep, int lstep, int lchunk, long long first, const int *__restrict__ Cptr, const int *__restrict__ Ccol,
              const unsigned short *__restrict__ Cmask, const unsigned char *__restrict__ Cptr16,
              const int *__restrict__ Cnnz, unsigned char *__restrict__ Ccol8, double *__restrict__ Cval) {
    __shared__ double s_acc[HEAVY_PART_COLS];
    __shared__ unsigned s_word[HEAVY_GROUP * HEAVY_PART_TILES];  // of a tile: the row's mask, and offset in s_acc
    __shared__ unsigned s_bin[HEAVY_BINS];
    __shared__ unsigned s_mark[HEAVY_BATCH / 4];
    const int lane = threadIdx.x;
    unsigned char *mk = reinterpret_cast<unsigned char *>(s_mark);
    // blocks: the heavy rows' items, part by part of each row's own, then the long
    // rows', lchunk rows after the others; 16 rows of the list on one XCD (blocks go
    // to the 8 XCDs in turn), the next 16 on the next
    const long long hb = first + blockIdx.x, heavy_blocks = heavy_padded(nheavy) * (long long)hstep;
    const bool heavy = hb < heavy_blocks;
    const long long h = heavy ? hb : hb - heavy_blocks;
    const int nrows = heavy ? nheavy : nlong, padded = heavy_padded(nrows), group = heavy ? 1 : HEAVY_GROUP;
    const int step = heavy ? hstep : lstep;
    int chunk = 0, in_chunk = padded;
    if (!heavy && lchunk < padded) {
        chunk = (int)(h / ((long long)lchunk * step)) * lchunk;
        in_chunk = min(lchunk, padded - chunk);
    }
    const long long at = h - (long long)chunk * step, g = at / in_chunk;
    const int x = chunk + (int)(at - g * in_chunk);
    int j0 = nrows < 128 ? x : ((x >> 7) * 8 + (x & 7)) * 16 + ((x >> 3) & 15);
    if (j0 >= nrows) return;
    if (!heavy) j0 += nheavy;
    const int4 row = rows[j0];
    const int i = row.x, I = i >> 4, r = i & 15;
    const int c1 = Cptr[I + 1];
    const int xa = Arowp[i], xe = Arowp[i + 1];
    unsigned stamp = 0u;
    auto clear_bins = [&]() {
        for (int j = lane; j < HEAVY_BINS; j += 64) s_bin[j] = 0xffffffffu;
        stamp = 0xffffffc0u;
    };
    for (int p0 = row.y + (int)g * group, tend = Cptr[I]; p0 < row.z; p0 += step * group) {
        int t = wave_lower_bound(Ccol, tend, c1, p0 * HEAVY_PART_TILES, lane);
        tend = wave_lower_bound(Ccol, t, c1, (p0 + group) * HEAVY_PART_TILES, lane);
        while (t < tend) {
            // a run of parts: as many as their entries of the row fit s_acc (one always does)
            const int ps = Ccol[t] / HEAVY_PART_TILES, jb = ps * HEAVY_PART_TILES;
            int pe = p0 + group, te = tend, nn = 0;
            for (int tb = t; tb < te && nn <= HEAVY_PART_COLS; tb += 256) {
                int J[4];
                unsigned cm[4];
    #pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int tt = tb + 64 * v + lane, ti = min(tt, te - 1);
                    J[v] = Ccol[ti];
                    cm[v] = Cmask[(long long)ti * 16 + r];
                    if (tt >= te) cm[v] = 0u;
                }
    #pragma unroll
                for (int v = 0; v < 4; v++) {
                    if (nn > HEAVY_PART_COLS) break;  // wave-uniform
                    const int c = __popc(cm[v]), incl = tsg_wave_incl_scan_dpp(c);
                    if (cm[v]) s_word[J[v] - jb] = cm[v] << 15 | (unsigned)(nn + incl - c);
                    const unsigned long long over = __ballot(nn + incl > HEAVY_PART_COLS);
                    if (over) {  // the run ends before this tile's part
                        pe = __builtin_amdgcn_readlane(J[v], __ffsll((long long)over) - 1) / HEAVY_PART_TILES;
                        nn = HEAVY_PART_COLS + 1;
                    } else {
                        nn += __builtin_amdgcn_readlane(incl, 63);
                    }
                }
            }
            if (nn > HEAVY_PART_COLS) {
                te = wave_lower_bound(Ccol, t, te, pe * HEAVY_PART_TILES, lane);
                nn = HEAVY_PART_COLS;
            }
            if (nn == 0) {  // other rows' tiles
                t = te;
                continue;
            }
            const int lo = ps << HEAVY_PART_LOG, hi = pe << HEAVY_PART_LOG;  // columns (n <= 2^27)
            // sources (A entries) 64 at a time, lane q's B row in the run's windows:
            // the entries two groups ahead, their windows one group ahead
            const long long w0 = (long long)(lo >> shift) * wstride;
            const long long w1 = (long long)min(((hi - 1) >> shift) + 1, nw) * wstride;
            const int inside = (int)((1u << shift) - 1u);
            const bool cut_lo = (lo & inside) != 0, cut_hi = (hi & inside) != 0;
            int k1 = 0, n0 = 0, n1 = 0;
            double a1 = 0.0, a2 = 0.0;
            auto fetch = [&](int xc) {
                k1 = -1;
                a2 = 0.0;
                if (xc + lane < xe) {
                    k1 = Acolx[xc + lane];
                    a2 = Avalx[xc + lane];
                }
            };
            auto window = [&]() {
                n0 = n1 = 0;
                if (k1 >= 0) {
                    n0 = win[w0 + k1];
                    n1 = win[w1 + k1];
                }
                a1 = a2;
            };
            fetch(xa);
            window();
            fetch(xa + 64);
            for (int j = lane; j < nn; j += 64) s_acc[j] = 0.0;
            for (int xc = xa; xc < xe; xc += 64) {
                int b0 = n0, b1 = n1;
                const double a = a1;
                window();
                fetch(xc + 128);
                if (cut_lo || cut_hi) range_in(Bcolx, b0, b1, cut_lo, lo, cut_hi, hi);  // windows wider than parts
                const int len = b1 - b0;
                const int incl = tsg_wave_incl_scan_dpp(len), pre = incl - len, delta = b0 - pre;
                const int total = __builtin_amdgcn_readlane(incl, 63);
                int prev = 0;
                for (int base = 0; base < total; base += HEAVY_BATCH) {
    #pragma unroll
                    for (int v = 0; v < HEAVY_BATCH / 256; v++) s_mark[64 * v + lane] = 0u;
                    if (stamp < 1u << 20) clear_bins();  // a batch has at most 64 * HEAVY_ROUNDS rounds
                    tsg_wave_sync();
                    if (len > 0 && pre >= base && pre < base + HEAVY_BATCH) mk[pre - base] = (unsigned char)(lane + 1);
                    tsg_wave_sync();
                    int q[HEAVY_ROUNDS], col[HEAVY_ROUNDS];
                    double b[HEAVY_ROUNDS];
    #pragma unroll
                    for (int v = 0; v < HEAVY_ROUNDS; v++) {
                        q[v] = max(prev, tsg_wave_incl_max_dpp((int)mk[64 * v + lane]));
                        prev = __builtin_amdgcn_readlane(q[v], 63);
                    }
    #pragma unroll
                    for (int v = 0; v < HEAVY_ROUNDS; v++) {  // every lane loads in bounds
                        const int e = __shfl(delta, q[v] - 1, 64) + min(base + 64 * v + lane, total - 1);
                        col[v] = Bcolx[e];
                        b[v] = Bvalx[e];
                    }
                    // all rounds' places before the first sum changes: their reads are in
                    // flight together
                    double as[HEAVY_ROUNDS];
                    unsigned wd[HEAVY_ROUNDS];
    #pragma unroll
                    for (int v = 0; v < HEAVY_ROUNDS; v++) as[v] = __shfl(a, q[v] - 1, 64);
    #pragma unroll
                    for (int v = 0; v < HEAVY_ROUNDS; v++) wd[v] = s_word[(col[v] >> 4) - jb];
    #pragma unroll
                    for (int v = 0; v < HEAVY_ROUNDS; v++) {
                        if (base + 64 * v >= total) break;  // wave-uniform
                        const bool on = base + 64 * v + lane < total;
                        const int p = (int)(wd[v] & 0x7fffu) + __popc(wd[v] >> (31 - (col[v] & 15)));
                        if (__builtin_amdgcn_readlane(q[v], 0) == __builtin_amdgcn_readlane(q[v], 63)) {  // one source
                            if (on) s_acc[p] = __builtin_fma(as[v], b[v], s_acc[p]);
                            tsg_wave_sync();
                        } else {
                            add_in_rounds(s_acc + p, s_bin + (p & (HEAVY_BINS - 1)), stamp, on, lane, as[v], b[v]);
                        }
                    }
                }
            }
            // the run's entries of row i, into their final positions
            for (int tb = t; tb < te; tb += 256) {
                int J[4], at[4];
                unsigned wd[4];
    #pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int ti = min(tb + 64 * v + lane, te - 1);
                    J[v] = Ccol[ti];
                    wd[v] = Cmask[(long long)ti * 16 + r];
                    at[v] = Cnnz[ti] + Cptr16[(long long)ti * 16 + r];
                    if (tb + 64 * v + lane >= te) wd[v] = 0u;
                }
    #pragma unroll
                for (int v = 0; v < 4; v++) {
                    unsigned cm = wd[v] << 16;
                    if (!cm) continue;
                    const double *d = s_acc + (s_word[J[v] - jb] & 0x7fffu);
                    double *o = Cval + at[v];
                    unsigned char *oc = Ccol8 + at[v];
                    while (cm) {
                        const int c = __clz((int)cm);
                        cm &= ~(0x80000000u >> c);
                        *o++ = *d++;
                        *oc++ = (unsigned char)c;
                    }
                }
            }
            t = te;
            tsg_wave_sync();  // the next run clears the sums
        }
    }
}

// ------------------------------------------------------------------ step 3, row-wise
// One 256-thread block per C tile-row whose C tiles, C nonzeros, A tiles and
// B tile-rows fit in LDS (g3 class, decided by k_row_class).  The
// tile-row's C values accumulate in LDS in their final order (tile by tile,
// row by row, ascending column), so the write-out is one contiguous copy.
// A tiles (I,K) are taken in ascending K; every (B tile q, nonempty A row
// r) task multiplies A row r by the B tile into C tile slot(q), row r.
// C row r belongs to wave g3_owner(r): only that wave ever adds into it,
// and each wave takes its tasks in ascending K, so every C entry receives its
// products in ascending k -- the order of the serial SPA -- with no atomics
// and no barrier between the K-steps for the accumulator's sake.
//
// An A tile with more than one entry has its A tile and its whole B
// tile-row K -- contiguous in row-major tile order -- staged into LDS with
// coalesced loads; an A tile with a single entry (r, k) needs row k of each
// B tile only, which its row's wave loads into registers itself (the
// stencil corner tiles: 18 of the 27 A tiles of a 27-point tile-row).
//
// The staging is software-pipelined: the tile-row's (K, B tile-row) table
// is loaded once, a staged K-step sits in the second LDS buffer while the
// previous one is computed, and the global loads of the step after next
// are in flight meanwhile.  A barrier precedes each staged K-step only.
#define G3_LAMAX 64  // A tiles per tile-row (row table built by wave 0)
// A C tile with at least G3_PADMIN nonzeros is followed by one unused
// accumulator element, so that the starts of equally sized tiles (a
// stencil's repeating 3 / 74 / 3 nonzeros) fall in different LDS banks; the
// lanes of a wave update the same row of many such tiles at once.
#define G3_PADMIN 16

// Dynamic LDS layout of k_step3_rows, from the maxima over its rows.
struct G3Layout {
    int umax, nnzmax, lamax, qb, bnnz, amax;
};
#define G3_NARR 13
__host__ __device__ inline size_t g3_layout(const G3Layout &L, size_t *off) {
    const size_t sz[G3_NARR] = {
        8u * (size_t)L.nnzmax,            // 0 acc
        // 1 B values (2 stages); before the first stage, the C tile columns
        // (int) and their slot ids (u8) of all the row's C tiles
        2u * 8u * (size_t)L.bnnz > 5u * G3_UMAX ? 2u * 8u * (size_t)L.bnnz : 5u * G3_UMAX,
        2u * 8u * (size_t)L.amax,         // 2 A values
        (size_t)L.umax,                   // 3 accumulator pads before each C tile (u8)
        2u * (size_t)L.umax,              // 4 C tile offsets (u16)
        32u * (size_t)L.umax,             // 5 C masks
        16u * (size_t)L.umax,             // 6 C row offsets
        20u * (size_t)L.lamax,            // 7 row table (5 ints per A tile)
        (size_t)L.lamax * (size_t)L.qb,   // 8 pair slots
        2u * 32u * (size_t)L.qb,          // 9 B masks
        2u * 16u * (size_t)L.qb,          // 10 B row offsets
        2u * 2u * ((size_t)L.qb + 1),     // 11 B tile nnz offsets (u16)
        2u * 2u * (size_t)L.qb};          // 12 B nonempty-row bits
    size_t o = 0;
    for (int i = 0; i < G3_NARR; i++) {
        off[i] = o;
        o += (sz[i] + 15) & ~(size_t)15;
    }
    return o;
}

// Pipeline stage registers.  Staging is split by wave so every branch is
// wave-uniform: wave 0 loads the B tile masks (uint4 = 8 rows, 2 per tile),
// row offsets (uint4 per tile) and nnz offsets; wave 1 the A tile (values,
// masks, row offsets); waves 2-3 the B values (4 per lane).  The ring has
// two register slots and runs over the staged (multi-entry) K-steps only: a
// stage is loaded two staged steps before it is computed and stored into
// LDS one staged step before.  The roles share one set of 10 registers per
// slot: wave 0 keeps its two 16-byte words as raw bits in d0:d1 and d2:d3
// (moved, never computed on).
#define G3_SLOT_DECL(S)                                                   \
    double S##d0 = 0.0, S##d1 = 0.0, S##d2 = 0.0, S##d3 = 0.0;            \
    unsigned S##e0 = 0u, S##e1 = 0u

#define G3_LOAD(j, S)                                                                                         \
    do {                                                                                                      \
        const int lb_ = G3_LB(j), q0_ = SROW(3, j);                                                           \
        /* Every lane loads from an in-bounds address (clamped; the lanes past  \
           the stage's data load a valid element and the store skips them), so \
           the loads are straight-line code and the store of this stage, two   \
           K-steps later, waits for these loads only. */                       \
        if (wave == 0) {                                                                                      \
            const long long bq_ = lb_ > 0 ? (long long)q0_ * 16 : 0;                                          \
            const double2 m_ = reinterpret_cast<const double2 *>(op.Bmask + bq_)[min(lane, max(2 * lb_ - 1, 0))]; \
            const double2 o_ = reinterpret_cast<const double2 *>(op.Bptr16 + bq_)[min(lane, max(lb_ - 1, 0))]; \
            S##d0 = m_.x; S##d1 = m_.y; S##d2 = o_.x; S##d3 = o_.y;                                           \
            S##e0 = op.Bnnz[q0_ + min(lane, lb_)]; /* made relative at the store */                           \
        } else if (wave == 1) {                                                                               \
            const int pan_ = G3_PAN(j), pa0_ = SROW(1, j); /* A tiles are never empty */                    \
            S##d0 = op.Aval[pa0_ + min(lane, pan_ - 1)];                                                      \
            S##d1 = op.Aval[pa0_ + min(lane + 64, pan_ - 1)];                                                 \
            S##d2 = op.Aval[pa0_ + min(lane + 128, pan_ - 1)];                                                \
            S##d3 = op.Aval[pa0_ + min(lane + 192, pan_ - 1)];                                                \
            const long long x_ = (long long)(a0 + (j)) * 16 + (lane & 15); /* A tile a0 + j */              \
            S##e0 = op.Amask[x_];                                                                             \
            S##e1 = op.Aptr16[x_];                                                                            \
        } else {                                                                                              \
            const int pbn_ = SROW(5, j), b_ = (wave - 2) * 64 + lane;                                         \
            const int pb0_ = pbn_ > 0 ? SROW(4, j) : 0, pbl_ = max(pbn_ - 1, 0);                              \
            S##d0 = op.Bval[pb0_ + min(b_, pbl_)];                                                            \
            S##d1 = op.Bval[pb0_ + min(b_ + 128, pbl_)];                                                      \
            S##d2 = op.Bval[pb0_ + min(b_ + 256, pbl_)];                                                      \
            S##d3 = op.Bval[pb0_ + min(b_ + 384, pbl_)];                                                      \
        }                                                                                                     \
    } while (0)

#define G3_STORE(j, S, buf)                                                                                   \
    do {                                                                                                      \
        const int lb_ = G3_LB(j);                                                                             \
        if (wave == 0) {                                                                                      \
            if (lane < 2 * lb_) reinterpret_cast<double2 *>(s_bm + (buf) * qb * 16)[lane] = make_double2(S##d0, S##d1); \
            if (lane < lb_) reinterpret_cast<double2 *>(s_bp + (buf) * qb * 16)[lane] = make_double2(S##d2, S##d3); \
            if (lane <= lb_) s_bnnz[(buf) * (qb + 1) + lane] = (unsigned short)((int)S##e0 - SROW(4, j));     \
            /* nonempty-row bits of this half tile, OR-ed with the partner half */                            \
            const unsigned wd_[4] = {(unsigned)__double2loint(S##d0), (unsigned)__double2hiint(S##d0),        \
                                     (unsigned)__double2loint(S##d1), (unsigned)__double2hiint(S##d1)};       \
            unsigned nz_ = 0;                                                                                 \
            _Pragma("unroll") for (int i_ = 0; i_ < 4; i_++) {                                                \
                const int k_ = (lane & 1) * 8 + 2 * i_;                                                       \
                nz_ |= ((wd_[i_] & 0xffffu) ? 1u : 0u) << (15 - k_);                                          \
                nz_ |= ((wd_[i_] >> 16) ? 1u : 0u) << (14 - k_);                                              \
            }                                                                                                 \
            nz_ |= __shfl_xor(nz_, 1, 64);                                                                    \
            if (!(lane & 1) && lane < 2 * lb_) s_bnz[(buf) * qb + (lane >> 1)] = (unsigned short)nz_;         \
        } else if (wave == 1) {                                                                               \
            const int pan_ = G3_PAN(j);                                                                      \
            double *av_ = s_aval + (buf) * amax;                                                              \
            if (lane < pan_) av_[lane] = S##d0;                                                               \
            if (lane + 64 < pan_) av_[lane + 64] = S##d1;                                                     \
            if (lane + 128 < pan_) av_[lane + 128] = S##d2;                                                   \
            if (lane + 192 < pan_) av_[lane + 192] = S##d3;                                                   \
            if (lane < 16) {                                                                                  \
                s_am[buf][lane] = (unsigned short)S##e0;                                                      \
                s_ap[buf][lane] = (unsigned char)S##e1;                                                       \
            }                                                                                                 \
        } else {                                                                                              \
            const int pbn_ = SROW(5, j), b_ = (wave - 2) * 64 + lane;                                         \
            double *bv_ = s_bval + (buf) * bnnzs;                                                             \
            if (b_ < pbn_) bv_[b_] = S##d0;                                                                   \
            if (b_ + 128 < pbn_) bv_[b_ + 128] = S##d1;                                                       \
            if (b_ + 256 < pbn_) bv_[b_ + 256] = S##d2;                                                       \
            if (b_ + 384 < pbn_) bv_[b_ + 384] = S##d3;                                                       \
        }                                                                                                     \
    } while (0)

// Row table entry k of A tile j (k = 1..5): 1 its first value, 2 its entry
// count | the tile count of B tile-row K << 9 | the rank of its first (A
// tile, B tile) pair << 15 (at most 256, 32 and 63 * 32), 3 the first tile
// of B tile-row K, 4 and 5 the first value and value count of that B
// tile-row (for a single-entry tile: 4 = its row | column << 8).
#define SROW(k, j) s_row[((k) - 1) * lamax + (j)]
#define G3_PAN(j) (SROW(2, j) & 511)
#define G3_LB(j) ((SROW(2, j) >> 9) & 63)
#define G3_PB(j) (SROW(2, j) >> 15)

// Wave owning C row r: rows r = 4i + c belong to wave (2, 0, 1, 3)[c], so the
// rows whose single-entry tiles a stencil produces (0 and 15) fall on the
// waves that stage only B values; g3_rbase(w) = the c of wave w.
__device__ __forceinline__ int g3_owner(int r) { return (0xD2 >> (2 * (r & 3))) & 3; }
__device__ __forceinline__ int g3_rbase(int w) { return (0xC9 >> (2 * w)) & 3; }

// Single-entry K-steps of one wave, lane = B tile, in a two-level pipeline
// over the steps the wave owns: the step after next has row k's mask, its
// tile's value offset and row k's offset within the tile in flight (G3_L1:
// sm_*); the next has row k's first two values, the A value, and its C
// row's mask and accumulator offset from the pair's slot (G3_L2: sv_*).
// Every address is in bounds (a lane past the B tile-row or with an empty
// row k loads a valid element and computes nothing).
#define G3_L1(j)                                                                      \
    do {                                                                              \
        const int rk_ = SROW(4, j), nq_ = G3_LB(j);                                  \
        const int q_ = max(SROW(3, j) + min(lane, nq_ - 1), 0);                       \
        const long long x_ = (long long)q_ * 16 + (rk_ >> 8);                         \
        sm_m = op.Bmask[x_];                                                          \
        sm_n = (unsigned)op.Bnnz[q_];                                                 \
        sm_p = op.Bptr16[x_];                                                         \
    } while (0)
#define G3_L2(j)                                                                      \
    do {                                                                              \
        const int nb_ = __popc(sm_m), nq_ = G3_LB(j), rr_ = SROW(4, j) & 15;         \
        const int pos_ = (int)(sm_n + sm_p), bs_ = nb_ > 0 ? pos_ : (int)sm_n;        \
        sv_0 = op.Bval[bs_];                                                          \
        sv_1 = op.Bval[bs_ + min(1, max(nb_ - 1, 0))];                                \
        sv_a = op.Aval[SROW(1, j)];                                                   \
        sv_m = sm_m;                                                                  \
        sv_p = pos_;                                                                  \
        const int sl_ = nq_ > 0 ? s_pslot[G3_PB(j) + min(lane, nq_ - 1)] : 0;         \
        sv_cm = s_cmask[sl_ * 16 + rr_];                                              \
        sv_cb = s_coff[sl_] + s_pad[sl_] + s_cptr[sl_ * 16 + rr_];                    \
    } while (0)
// K-step j = (row rr, column k): row k of the lane's B tile into row rr of
// the pair's C tile, ascending column (values past the second from memory);
// then the pipeline moves one step on
#define G3_SINGLE(j)                                                                  \
    do {                                                                              \
        unsigned bm_ = sv_m;                                                          \
        if (lane < G3_LB(j) && bm_) {                                                 \
            double *ac_ = s_acc + sv_cb;                                              \
            int jb_ = 0;                                                              \
            while (bm_) {                                                             \
                const int bb_ = 31 - __clz(bm_);                                      \
                bm_ &= ~(1u << bb_);                                                  \
                const double b_ = jb_ == 0 ? sv_0 : jb_ == 1 ? sv_1 : op.Bval[sv_p + jb_]; \
                double *acc_ = ac_ + __popc(sv_cm >> (bb_ + 1));                      \
                *acc_ = __builtin_fma(sv_a, b_, *acc_);                               \
                jb_++;                                                                \
            }                                                                         \
        }                                                                             \
        sA = sB;                                                                      \
        if (sA < 64) G3_L2(sA);                                                       \
        sB = g3_pop(own);                                                             \
        if (sB < 64) G3_L1(sB);                                                       \
    } while (0)

// Lowest set bit's index, cleared from m (64 when m is empty).
__device__ __forceinline__ int g3_pop(unsigned long long &m) {
    if (!m) return 64;
    const int b = __ffsll((long long)m) - 1;
    m &= m - 1;
    return b;
}

__global__ void __launch_bounds__(G3_THREADS)
k_step3_rows(TileOperands op, const int *__restrict__ Cptr, const int *__restrict__ Ccol, int tilem,
             const unsigned short *__restrict__ Cmask, const unsigned char *__restrict__ Cptr16,
             const int *__restrict__ Cnnz, const unsigned char *__restrict__ rowcls,
             unsigned char *__restrict__ Ccol8, double *__restrict__ Cval, G3Layout L) {
    extern __shared__ __align__(16) unsigned char g3_smem[];
    size_t off[G3_NARR];
    g3_layout(L, off);
    const int lamax = L.lamax, qb = L.qb, amax = L.amax, bnnzs = L.bnnz;
    double *s_acc = reinterpret_cast<double *>(g3_smem + off[0]);
    double *s_bval = reinterpret_cast<double *>(g3_smem + off[1]);
    double *s_aval = reinterpret_cast<double *>(g3_smem + off[2]);
    int *s_ccol = reinterpret_cast<int *>(g3_smem + off[1]);  // setup only: the B value area
    unsigned char *s_cidx = g3_smem + off[1] + 4 * G3_UMAX;    // setup only
    unsigned short *s_coff = reinterpret_cast<unsigned short *>(g3_smem + off[4]);  // < G3_NNZMAX
    unsigned char *s_pad = g3_smem + off[3];  // accumulator pads before each C tile
    unsigned short *s_cmask = reinterpret_cast<unsigned short *>(g3_smem + off[5]);
    unsigned char *s_cptr = g3_smem + off[6];
    int *s_row = reinterpret_cast<int *>(g3_smem + off[7]);
    unsigned char *s_pslot = g3_smem + off[8];
    unsigned short *s_bm = reinterpret_cast<unsigned short *>(g3_smem + off[9]);
    unsigned char *s_bp = g3_smem + off[10];
    unsigned short *s_bnnz = reinterpret_cast<unsigned short *>(g3_smem + off[11]);
    unsigned short *s_bnz = reinterpret_cast<unsigned short *>(g3_smem + off[12]);
    __shared__ unsigned short s_am[2][16];
    __shared__ unsigned char s_ap[2][16];
    __shared__ int s_wne[G3_THREADS / 64], s_wbig[G3_THREADS / 64];
    __shared__ unsigned long long s_stg, s_own[G3_THREADS / 64];  // staged steps; singles per wave
    static_assert(G3_UMAX <= G3_THREADS, "one C tile per thread in the setup");
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const unsigned blk = tsg_block();
    if (blk >= (unsigned)tilem) return;
    const int I = (int)tsg_xcd_block(blk, (unsigned)tilem);
    if (rowcls[I] != 1) return;  // block-uniform
    const int c0 = Cptr[I], u = Cptr[I + 1] - c0;
    const int nbase = Cnnz[c0], nrow = Cnnz[c0 + u] - nbase;
    const int a0 = op.Aptr[I], la = op.Aptr[I + 1] - a0;
    // C tiles of the tile-row (u <= G3_UMAX), one per thread.  Only the
    // nonempty ones get accumulator metadata (offset, masks, row offsets),
    // at their rank among the nonempty tiles: a task is active only when
    // one of its products exists, so no task lands in an empty C tile.
    // (their masks and row offsets are loaded here, stored after the barrier)
    int ccol = 0, cnz0 = 0, cnz1 = 0;
    bool ne = false;
    uint4 cmk0 = make_uint4(0u, 0u, 0u, 0u), cmk1 = cmk0, cpt = cmk0;
    if (tid < u) {
        ccol = Ccol[c0 + tid];
        cnz0 = Cnnz[c0 + tid];
        cnz1 = Cnnz[c0 + tid + 1];
        ne = cnz1 > cnz0;
        const uint4 *cm = reinterpret_cast<const uint4 *>(Cmask + (long long)(c0 + tid) * 16);
        cmk0 = cm[0];
        cmk1 = cm[1];
        cpt = reinterpret_cast<const uint4 *>(Cptr16 + (long long)(c0 + tid) * 16)[0];
    }
    const unsigned long long neb = __ballot(ne), bgb = __ballot(cnz1 - cnz0 >= G3_PADMIN);
    if (lane == 0) {
        s_wne[wave] = __popcll(neb);
        s_wbig[wave] = __popcll(bgb);
    }
    // row table: one entry per A tile of the tile-row (wave 0, la <= 64)
    if (wave == 0) {
        int lb = 0, pan = 0, rk = 0;
        if (lane < la) {
            const int p = a0 + lane, K = op.Acol[p];
            const int pa0 = op.Annz[p], q0 = op.Bptr[K], q1 = op.Bptr[K + 1];
            pan = op.Annz[p + 1] - pa0;
            const int pb0 = op.Bnnz[q0], pb1 = op.Bnnz[q1];
            // the row masks: a single entry's row and column
            const uint4 *amk = reinterpret_cast<const uint4 *>(op.Amask + (long long)p * 16);
            const uint4 m0 = amk[0], m1 = amk[1];
            const unsigned w[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
#pragma unroll
            for (int r = 15; r >= 0; r--) {
                const unsigned m = (w[r >> 1] >> (16 * (r & 1))) & 0xffffu;
                if (m) rk = r | ((__clz((int)m) - 16) << 8);
            }
            lb = q1 - q0;
            SROW(1, lane) = pa0;
            SROW(3, lane) = q0;
            SROW(4, lane) = pan == 1 ? rk : pb0;
            SROW(5, lane) = pb1 - pb0;
        }
        const int incl = tsg_wave_incl_scan(lb);
        if (lane < la) SROW(2, lane) = pan | (lb << 9) | ((incl - lb) << 15);
        const unsigned long long stg = __ballot(pan > 1);
        unsigned long long ow[G3_THREADS / 64];
#pragma unroll
        for (int w = 0; w < G3_THREADS / 64; w++) ow[w] = __ballot(pan == 1 && g3_owner(rk & 15) == w);
        if (lane == 0) {
            s_stg = stg;
#pragma unroll
            for (int w = 0; w < G3_THREADS / 64; w++) s_own[w] = ow[w];
        }
    }
    __syncthreads();
    // the ring's first three stages need only the row table: their loads
    // are in flight while the C tile slots and pair slots are set up
    unsigned long long rest = s_stg, own = s_own[wave];
    int fa = g3_pop(rest), fb = g3_pop(rest);  // staged steps 0 and 1 (64: none)
    G3_SLOT_DECL(R0_);
    G3_SLOT_DECL(R1_);
    if (fa < 64) G3_LOAD(fa, R0_);
    if (fb < 64) G3_LOAD(fb, R1_);
    unsigned sm_m = 0u, sm_n = 0u, sm_p = 0u, sv_m = 0u, sv_cm = 0u;
    int sv_p = 0, sv_cb = 0;
    double sv_0 = 0.0, sv_1 = 0.0, sv_a = 0.0;
    int sA = g3_pop(own), sB = g3_pop(own);  // this wave's next two single-entry steps
    if (sA < 64) G3_L1(sA);
    int ci = __popcll(neb & ((1ull << lane) - 1ull)), pad = __popcll(bgb & ((1ull << lane) - 1ull));
    for (int w = 0; w < wave; w++) {
        ci += s_wne[w];
        pad += s_wbig[w];
    }
    int un = 0, npad = 0;
#pragma unroll
    for (int w = 0; w < G3_THREADS / 64; w++) {
        un += s_wne[w];
        npad += s_wbig[w];
    }
    // C tile slot of every (A tile, B tile) pair of the tile-row.  When the
    // row's C tile columns span at most the accumulator's bytes, the
    // accumulator area first holds a direct map column -> slot (every pair's
    // column is in the row's C tile list, so unmapped bytes are never read);
    // otherwise a binary search over the sorted C tile columns.  An empty
    // tile maps to the next nonempty tile's slot (< 256); no task uses it.
    const int jlo = Ccol[c0], jspan = Ccol[c0 + u - 1] - jlo + 1;
    const bool direct = jspan <= 8 * L.nnzmax;
    unsigned char *s_map = reinterpret_cast<unsigned char *>(s_acc);
    if (tid < u) {
        s_ccol[tid] = ccol;
        s_cidx[tid] = (unsigned char)ci;
        if (direct) s_map[ccol - jlo] = (unsigned char)ci;
        if (ne) {
            s_coff[ci] = (unsigned short)(cnz0 - nbase);
            s_pad[ci] = (unsigned char)pad;
            reinterpret_cast<uint4 *>(s_cmask)[2 * ci] = cmk0;
            reinterpret_cast<uint4 *>(s_cmask)[2 * ci + 1] = cmk1;
            reinterpret_cast<uint4 *>(s_cptr)[ci] = cpt;
        }
    }
    // B tile columns of the row's (A tile j, B tile qi) pairs, xx = j * G3_QB
    // + qi: those of the first 32 A tiles are loaded here, so that their
    // latency overlaps the barrier (the rest after it)
    static_assert(G3_QB == 32, "pair index split by shifts");
    static_assert(G3_LAMAX * G3_QB <= 8 * G3_THREADS, "eight pairs per thread");
    int pj[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int xx = tid + G3_THREADS * t, j = xx >> 5, qi = xx & 31;
        pj[t] = xx < la * G3_QB && qi < G3_LB(j) ? op.Bcol[SROW(3, j) + qi] : -1;
    }
    __syncthreads();
    // the pair's slot index is its rank G3_PB(j) + qi
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int xx = tid + G3_THREADS * t, j = xx >> 5, qi = xx & 31;
        const int J = t < 4 ? pj[t & 3] : xx < la * G3_QB && qi < G3_LB(j) ? op.Bcol[SROW(3, j) + qi] : -1;
        if (J < 0) continue;
        const int x = G3_PB(j) + qi;
        if (direct) {
            s_pslot[x] = s_map[J - jlo];
        } else {
            int lo = 0, hi = u - 1;  // J is in the step-1 list
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (s_ccol[mid] < J) lo = mid + 1; else hi = mid;
            }
            s_pslot[x] = s_cidx[lo];
        }
    }
    __syncthreads();  // the map area becomes the accumulator
    for (int i = tid; i < nrow + npad; i += G3_THREADS) s_acc[i] = 0.0;
    if (sA < 64) G3_L2(sA);
    if (sB < 64) G3_L1(sB);
    if (fa < 64) G3_STORE(fa, R0_, 0);
    __syncthreads();

    // compute staged K-step j from buffer buf: the tasks of this wave's rows
    auto compute = [&](int j, int buf) {
        const int nq = G3_LB(j), pbase = G3_PB(j);
        const int ncand = nq * 4;
        const unsigned short *sbz = s_bnz + buf * qb;
        // candidate tasks (B tile qi, A row rb + 4i) meeting at least one
        // nonempty B row, compacted into a register queue: position Q of the
        // queue is lane Q & 63 of qlo (Q < 64) or qhi (Q >= 64).  There are
        // at most two chunks of 64 candidates (ncand <= G3_QB * 4 = 128), so
        // qn <= 64 before each chunk.  Each chunk is moved by one forward
        // permute over all 64 lanes: active lanes to the queue positions
        // qn.., inactive ones after them, so every lane receives exactly one
        // value and the permute needs no LDS memory.
        int qn = 0, qlo = 0, qhi = 0;
        const int rb = g3_rbase(wave);
        for (int c = 0; c < ncand; c += 64) {
            const int x = c + lane;
            int code = 0;
            bool act = false;
            if (x < ncand) {
                const int qi = x >> 2, rr = rb + 4 * (x & 3);
                act = (s_am[buf][rr] & sbz[qi]) != 0;
                code = (qi << 4) | rr;
            }
            const unsigned long long bal = __ballot(act);
            const int na = __popcll(bal), below = __popcll(bal & ((1ull << lane) - 1ull));
            const int rank = act ? below : na + (lane - below);
            const int got = __builtin_amdgcn_ds_permute(((qn + rank) & 63) << 2, code);
            if (lane >= qn && lane < qn + na) qlo = got;
            if (lane + 64 < qn + na) qhi = got;
            qn += na;
        }
        const unsigned short *sbm = s_bm + buf * qb * 16;
        const unsigned char *sbp = s_bp + buf * qb * 16;
        const unsigned short *sbnnz = s_bnnz + buf * (qb + 1);
        const double *sbv = s_bval + buf * bnnzs;
        const double *sav = s_aval + buf * amax;
        for (int t0 = 0; t0 < qn; t0 += 64) {
            if (t0 + lane >= qn) break;
            const int code = t0 ? qhi : qlo;
            const int qi = code >> 4, rr = code & 15;
            const int slot = s_pslot[pbase + qi];
            const unsigned cm = s_cmask[slot * 16 + rr];
            const int cbase = s_coff[slot] + s_pad[slot] + s_cptr[slot * 16 + rr];
            const unsigned short *bm16 = sbm + qi * 16;
            const unsigned char *bp16 = sbp + qi * 16;
            const double *bvt = sbv + sbnnz[qi];
            unsigned am = s_am[buf][rr];
            const double *av = sav + s_ap[buf][rr];
            int ia = 0;
            while (am) {  // A row entries, ascending k
                const int b = 31 - __clz(am);
                am &= ~(1u << b);
                const int k = 15 - b;
                const double a = av[ia++];
                unsigned bm = bm16[k];
                const double *brow = bvt + bp16[k];
                int jb = 0;
                while (bm) {  // B row k entries, ascending column
                    const int bb = 31 - __clz(bm);
                    bm &= ~(1u << bb);
                    double *acc = &s_acc[cbase + __popc(cm >> (bb + 1))];
                    *acc = __builtin_fma(a, brow[jb++], *acc);
                }
            }
        }
    };
    // single-entry steps before the first staged step
    while (sA < fa) G3_SINGLE(sA);
    // staged step fa (number f) from buffer f & 1 and ring slot SR; then the
    // next staged step fb is stored from slot SN, the singles between them
    // are taken, and staged step fc is loaded into slot SR.  A barrier
    // precedes every staged step: its stores are visible, and the buffer it
    // overwrote was last read two staged steps before.
    int f = 0;
#define G3_ITER(SN, SR)                                 \
    if (fa < 64) {                                      \
        compute(fa, f & 1);                             \
        if (fb < 64) G3_STORE(fb, SN, (f + 1) & 1);     \
        const int fc = g3_pop(rest);                    \
        while (sA < fb) G3_SINGLE(sA);                  \
        if (fc < 64) G3_LOAD(fc, SR);                   \
        if (fb < 64) __syncthreads();                   \
        fa = fb;                                        \
        fb = fc;                                        \
        f++;                                            \
    }
    while (fa < 64) {
        G3_ITER(R1_, R0_)
        G3_ITER(R0_, R1_)
    }
#undef G3_ITER
    __syncthreads();  // every wave's rows are complete
    // write out, one C tile row at a time: values from the padded
    // accumulator, columns from the masks
    for (int x = tid; x < un * 16; x += G3_THREADS) {
        const int slot = x >> 4;
        unsigned cm = s_cmask[x];
        const int fo = s_coff[slot] + s_cptr[x];
        const double *av = s_acc + fo + s_pad[slot];
        unsigned char *oc = Ccol8 + nbase + fo;
        double *ov = Cval + (long long)nbase + fo;
        int jj = 0;
        while (cm) {
            const int bb = 31 - __clz(cm);
            cm &= ~(1u << bb);
            oc[jj] = (unsigned char)(15 - bb);
            ov[jj] = av[jj];
            jj++;
        }
    }
}
#undef SROW

// ------------------------------------------------------------------ step 3, row lines
// One block per C tile-row with at most LN_UMAX C tiles and LN_NNZ C
// nonzeros, from A's and B's row index.  A group of G lanes (16, 32 or 64:
// the first that holds the longest B row the tile-row meets, above 64 in two
// pieces) owns a C row: it takes the row's A entries k in ascending order, one
// per step, its lanes the entries of B row k, and adds the products to the
// row's entries in LDS.  One B row never meets an entry of C twice and groups
// never share one, so there are no atomics and no checks, and every C entry
// sums its products in ascending k.
//   Sources (A entries) are held 16 at a time, one per lane and the same in
// every 16 lanes of the group, so that a source reaches its group by a DPP row
// broadcast folded into its use, and the LDS takes only the five accesses
// below.  B rows are loaded four steps ahead.
//   Position of a product: the slot of its tile column from a byte map of
// the columns modulo a power of two (binary search in a tile-row wider than
// the map whose columns collide there), then one word with the C row's mask
// and offset in that tile: offset + bits of the mask before the column.
// Values are summed in final order with a gap after every 16, which moves
// the equal tiles of a stencil to different LDS banks; the column byte is
// left beside the sum.  Both are written out as one run, past the L2 (it
// holds the B rows that the next tile-rows read again: 2.26 -> 2.06 ms).
//   Four blocks (32 waves) a CU; the L1 is taken in four of five of its cycles,
// VALU and LDS are busy in two of three (half of the LDS's are bank conflicts),
// HBM carries 2.6 TB/s.  27-point 128^3 periodic 4.00 ms by
// k_step3_rows -> 2.06 (1.5 G products, 729 a C row), 61x47x53 385 -> 133 us,
// banded 39989 (half-bandwidth 20) 165 us by k_step3_flat -> 97.  With the
// sources broadcast by ds_bpermute (four more LDS accesses) 2.65 ms, with 80
// registers and six waves a SIMD 2.19.
#define LN_THREADS 512
#define LN_UMAX 256      // u8 slots
#define LN_NNZ 4096      // 34 KiB of sums; offsets of a tile row fit 15 bits
#define LN_MAP 8192      // bytes of the largest column map
#define LN_MAP_MIN 1024  // any slot byte stays inside LDS behind the mask words
#define LN_ANNZ 2048     // A entries of the tile-row (one row's are a serial chain)
#define LN_BROW 128      // entries of a B row: two pieces of 64
// Lanes idle where the longest B row is far from the mean: k_step3_flat is
// the better one there.  R-MAT scale 11 A*A^T whole product 388 us with 2 *
// mean + 16, 401 with 4 *, and 388 without row lines; ER (Poisson rows, means 4
// to 14) 102..150 us against 137..197 by k_step3_flat.
#define LN_SKEW 2
#define LN_SKEW0 16
#define LN_CLASS 4       // row class LN_CLASS + g: groups of 16 << g lanes
struct LinesLayout {
    int nnz, umax, map;
};
// LDS (all of it dynamic, so from address 0): the byte of entry p is at base +
// p, its sum at 8 * ln_pos(base + p): with base a multiple of 16 the sums start
// at 8.5 * base, behind the bytes, and one register addresses both.  Word 0
// is the collision flag.
__host__ __device__ inline int ln_pos(int p) { return p + (p >> 4); }
__host__ __device__ inline size_t lines_layout(const LinesLayout &L, int *base, size_t off[4]) {
    *base = ((L.nnz + 8) * 2 / 15 + 16) & ~15;
    off[0] = 8 * (size_t)ln_pos(*base);                                   // sums
    off[1] = 8 * (size_t)(ln_pos(*base + L.nnz) + 1);                     // mask and offset words, [row][tile]
    off[2] = off[1] + 64 * (size_t)L.umax;                                // tile columns
    off[3] = off[2] + 4 * (size_t)L.umax;                                 // column map
    return off[3] + (size_t)L.map;
}
__global__ void __launch_bounds__(LN_THREADS, 8)
k_step3_lines(const int *__restrict__ Arowp, const int *__restrict__ Acolx, const double *__restrict__ Avalx,
              const int *__restrict__ Browp, const int *__restrict__ Bcolx, const double *__restrict__ Bvalx, int m,
              int tilem, const int *__restrict__ Cptr, const int *__restrict__ Ccol,
              const unsigned short *__restrict__ Cmask, const unsigned char *__restrict__ Cptr16,
              const int *__restrict__ Cnnz, const unsigned char *__restrict__ rowcls,
              unsigned char *__restrict__ Ccol8, double *__restrict__ Cval, LinesLayout L) {
    extern __shared__ __align__(16) unsigned char s_lds[];
    typedef __attribute__((address_space(3))) double *lds_f64;
    typedef __attribute__((address_space(3))) unsigned char *lds_u8;
    int base;
    size_t off[4];
    lines_layout(L, &base, off);
    int *s_flag = reinterpret_cast<int *>(s_lds);
    unsigned char *s_byte = s_lds + base;
    double *s_acc = reinterpret_cast<double *>(s_lds + off[0]);
    unsigned *s_meta = reinterpret_cast<unsigned *>(s_lds + off[1]);
    int *s_col = reinterpret_cast<int *>(s_lds + off[2]);
    unsigned char *s_map = s_lds + off[3];
    const unsigned blk = tsg_block();
    if (blk >= (unsigned)tilem) return;
    const int I = (int)tsg_xcd_block(blk, (unsigned)tilem);
    const int cls = rowcls[I];
    if (cls < LN_CLASS) return;  // block-uniform
    const int tid = threadIdx.x, lane = tid & 63, nt = blockDim.x;
    const int gl = 4 + cls - LN_CLASS, G = 1 << gl;
    const int t = tid & (G - 1), ngrp = nt >> gl;
    const int c0 = Cptr[I], u = Cptr[I + 1] - c0;
    const int nbase = Cnnz[c0], nrow = Cnnz[c0 + u] - nbase;
    const int span = Ccol[c0 + u - 1] - Ccol[c0] + 1;
    const unsigned mapbits = 31 - __clz(L.map);
    // sources of the group's row, 16 lanes deep: [b0, last] its B row (a lane
    // without one: a far b0 and entry 0), k and av those of the next 16
    int x1 = 0, xk = 0, kk = -1, b0 = 0, last = 0;
    double a = 0.0, av = 0.0;
    auto fetch = [&]() {  // A entries xk + lane
        kk = -1;
        av = 0.0;
        if (xk + (lane & 15) < x1) {
            kk = Acolx[xk + (lane & 15)];
            av = Avalx[xk + (lane & 15)];
        }
        xk += 16;
    };
    int p0 = 0, p1 = 0;
    double an = 0.0;
    auto bounds = [&]() {  // their B rows
        p0 = p1 = 0;
        if (kk >= 0) {
            p0 = Browp[kk];
            p1 = Browp[kk + 1];
        }
        an = av;
    };
    auto take = [&]() {
        a = an;
        b0 = p1 > p0 ? p0 : 0x40000000;
        last = p1 > p0 ? p1 - 1 : 0;
    };
    auto start = [&](int r) {
        const int row = 16 * I + r;
        xk = x1 = 0;
        if (r < 16 && row < m) {
            xk = Arowp[row];
            x1 = Arowp[row + 1];
        }
        fetch();
    };
    int r = tid >> gl;
    start(r);
    bounds();
    fetch();
    if (tid == 0) *s_flag = 0;
    for (int i = tid; i < ln_pos(nrow) + 1; i += nt) s_acc[i] = 0.0;
    for (int i = tid; i < u; i += nt) {
        const long long c = c0 + i;
        const int J = Ccol[c], at = base + Cnnz[c] - nbase;
        const uint4 m0 = reinterpret_cast<const uint4 *>(Cmask)[2 * c], m1 = reinterpret_cast<const uint4 *>(Cmask)[2 * c + 1];
        const uint4 p = reinterpret_cast<const uint4 *>(Cptr16)[c];
        const unsigned mw[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
        const unsigned pw[4] = {p.x, p.y, p.z, p.w};
        s_col[i] = J;
        s_map[(unsigned)J & (L.map - 1)] = (unsigned char)i;
#pragma unroll
        for (int q = 0; q < 16; q++) {
            // bits 30..15: columns 0..15; bits 14..0: base + offset
            const unsigned mk = q & 1 ? (mw[q >> 1] >> 1) & 0x7fff8000u : (mw[q >> 1] & 0xffffu) << 15;
            s_meta[q * L.umax + i] = mk | (unsigned)(at + (int)((pw[q >> 2] >> (8 * (q & 3))) & 255u));
        }
    }
    __syncthreads();
    // consecutive columns never collide in the map; others are looked at
    bool direct = span <= L.map;
    if (!direct) {
        for (int i = tid; i < u; i += nt)
            if (s_map[(unsigned)s_col[i] & (L.map - 1)] != i) *s_flag = 1;
        __syncthreads();
        direct = *s_flag == 0;
    }
    for (; r < 16; r += ngrp) {
        const unsigned *meta = s_meta + r * L.umax;
        auto slot_search = [&](int J) -> int {
            int lo = 0, hi = u - 1;  // J is in the list
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (s_col[mid] < J) lo = mid + 1; else hi = mid;
            }
            return lo;
        };
        // a lane past its B row may look up any column: every read stays in LDS
        auto slot_map = [&](int col) -> int { return s_map[__builtin_amdgcn_ubfe((unsigned)col, 4, mapbits)]; };
        auto place = [&](unsigned w, int col) -> int {
            return (int)(w & 0x7fffu) + __popc(w >> ((~col & 15) | 16));
        };
        auto add = [&](int pos, int col, double as, double b) {
            lds_f64 p = (lds_f64)(unsigned)(ln_pos(pos) << 3);
            *p = __builtin_fma(as, b, *p);
            *(lds_u8)(unsigned)pos = (unsigned char)col;  // low four bits: the column in its tile
        };
        for (;;) {
            take();
            const unsigned long long has = __ballot(b0 < 0x40000000), cnt = __ballot(x1 > xk - 32 + (lane & 15));
            if (!__any(x1 > xk - 32)) break;
            // steps: the longest row of the wave decides
            unsigned long long fold = cnt | cnt >> 32;
            fold |= fold >> 16;
            const int ns = 32 - __clz((int)(fold & 0xffffu));
            bounds();
            fetch();
            // batches of four loads, one batch in flight ahead of the one that is
            // added: four sources, or two with two pieces each
            auto batches = [&](auto two) {
                constexpr int P = decltype(two)::value ? 2 : 1;
                int col[2][4];
                bool on[2][4];  // an entry of the B row
                double b[2][4];
                auto load = [&](int s, int w) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int e = tsg_row16_bcast(b0, s + i / P) + t + (i % P) * G;
                        const int ec = min(e, tsg_row16_bcast(last, s + i / P));
                        on[w][i] = e == ec;
                        col[w][i] = Bcolx[(unsigned)ec];
                        b[w][i] = Bvalx[(unsigned)ec];
                    }
                };
                load(0, 0);
#pragma unroll
                for (int s = 0; s < 16; s += 4 / P) {
                    if (s >= ns) break;
                    const int w = (s * P >> 2) & 1;
                    if (s + 4 / P < 16 && s + 4 / P < ns) load(s + 4 / P, w ^ 1);
                    int pos[4];
                    unsigned mw[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) mw[i] = meta[slot_map(col[w][i])];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        pos[i] = place(mw[i], col[w][i]);
                        asm("" : "+v"(pos[i]));  // of every lane: not sunk into a branch each
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const double as = tsg_row16_bcast(a, s + i / P);
                        if (on[w][i]) add(pos[i], col[w][i], as, b[w][i]);
                        tsg_wave_sync();
                    }
                }
            };
            if (direct && __any(last - b0 >= G)) {
                batches(std::true_type{});
            } else if (direct && has) {
                batches(std::false_type{});
            } else {  // columns that collide in the map
                for (int s = 0; s < ns; s++) {
                    const int at = (lane & 48) + s;
                    const int bs = __shfl(b0, at, 64), be = __shfl(last, at, 64);
                    const double as = __shfl(a, at, 64);
                    for (int e = bs + t; e <= be; e += G) {
                        const int c = Bcolx[e];
                        add(place(meta[slot_search(c >> 4)], c), c, as, Bvalx[e]);
                    }
                    tsg_wave_sync();
                }
            }
        }
        if (r + ngrp < 16) {
            start(r + ngrp);
            bounds();
            fetch();
        }
    }
    __syncthreads();
    for (int i = tid; i < nrow; i += nt) __builtin_nontemporal_store(s_acc[ln_pos(i)], Cval + (long long)nbase + i);
    // column bytes, by the words of the run
    const int head = (4 - (nbase & 3)) & 3;  // bytes before the first whole word
    unsigned char *out = Ccol8 + nbase;
    const int words = max(0, nrow - head) >> 2;
    for (int i = tid; i < words; i += nt) {
        const unsigned *w = reinterpret_cast<const unsigned *>(s_byte) + i;
        const unsigned v = head ? __builtin_amdgcn_alignbyte(w[1], w[0], head) : w[0];
        __builtin_nontemporal_store(v & 0x0f0f0f0fu, reinterpret_cast<unsigned *>(out + head) + i);
    }
    if (tid < 8) {  // the ragged ends
        const int i = tid < 4 ? tid : head + 4 * words + tid - 4;
        if (i < nrow && (tid < 4 ? i < head : true)) out[i] = s_byte[i] & 15;
    }
}

// Step-3 class of every C tile-row: 1 = row-wise kernel (its C tiles, C
// nonzeros, A tiles and B tile-rows are within the G3 caps), 0 = tile-parallel
// kernel, 2 = nothing to compute, LN_CLASS + g = row lines with groups of 16 <<
// g lanes (lines set: both operands carry their row index).  Per block,
// part[CLS_WORDS * block + i]: i = 0 the class-0 rows, i = 1..6 the maxima
// over class-1 rows of (nonempty C tiles, C nonzeros plus accumulator pads,
// A tiles, B tiles per B tile-row, B nonzeros per B tile-row, A tile
// nonzeros) for the LDS layout, i = 7..10 those over the row-lines rows of (C
// nonzeros, C tiles, tile-column span, g + 1), i = 11 the rows of classes 0 and
// 1, i = 12 the element segments of the class-0 rows, at most.
// 16 lanes per tile-row (16 tile-rows per block): the lanes walk the row's A
// tiles and C tiles in strides of 16, so the dependent loads of different A
// tiles are in flight together.  k_row_class_reduce folds the blocks' partials
// into out (sums and maxima): no atomics, which on one cache
// line would serialise across the thousands of blocks.
#define CLS_WORDS 13
// By DPP: the classes' folds are a dozen reductions each (27d 61x47x53: k_row_class
// 7.3 -> 5.9 us, k_row_class_reduce 4.9 -> 4.0).  Every lane active; values not negative.
__device__ __forceinline__ int cls_sum(int v) { return __builtin_amdgcn_readlane(tsg_wave_incl_scan_dpp(v), 63); }
__device__ __forceinline__ int cls_max(int v) { return __builtin_amdgcn_readlane(tsg_wave_incl_max_dpp(v), 63); }
__device__ __forceinline__ bool cls_sums(int i) { return i == 0 || i >= 11; }
__device__ __forceinline__ int g16_max(int v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 16));
    return v;
}
__global__ void __launch_bounds__(256)
k_row_class(TileOperands op, const int *__restrict__ Cptr, const int *__restrict__ Ccol, const int *__restrict__ Cnnz, int tilem,
            unsigned char *__restrict__ cls, int *part, int none_fit, const int *__restrict__ longest,
            int *__restrict__ ticket, int *__restrict__ out, int *__restrict__ host) {
    __shared__ int s_red[4][CLS_WORDS];
    const int r = threadIdx.x & 15, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int I = blockIdx.x * 16 + (threadIdx.x >> 4);
    int unfit = 0, mu = 0, mn = 0, ml = 0, mq = 0, mb = 0, ma = 0;
    int ln = 0, lu = 0, ls = 0, lg = 0, other = 0, segs = 0;
    if (I < tilem) {  // uniform in the 16-lane group
        const int c0 = Cptr[I], c1 = Cptr[I + 1];
        const int nrow = Cnnz[c1] - Cnnz[c0];
        unsigned char k;
        if (nrow == 0) {
            k = 2;
        } else {
            const int a0 = op.Aptr[I], a1 = op.Aptr[I + 1];
            bool ok = !none_fit && c1 - c0 <= G3_UMAX && nrow <= G3_NNZMAX && a1 - a0 <= G3_LAMAX;
            if (longest && c1 - c0 <= LN_UMAX && nrow <= LN_NNZ && op.Annz[a1] - op.Annz[a0] <= LN_ANNZ) {  // group-uniform
                int mx = 0, sum = 0;
                for (int p = a0 + r; p < a1; p += 16) {
                    const int K = op.Acol[p];
                    mx = max(mx, longest[K]);
                    sum += op.Bnnz[op.Bptr[K + 1]] - op.Bnnz[op.Bptr[K]];
                }
                mx = g16_max(mx);
                const int mean = tsg_group16_sum(sum) / (16 * max(a1 - a0, 1)), g = mx <= 16 ? 0 : mx <= 32 ? 1 : 2;
                if (mx <= LN_BROW && mx <= LN_SKEW * mean + LN_SKEW0) {
                    lg = g + 1;
                    ln = nrow;
                    lu = c1 - c0;
                    ls = Ccol[c1 - 1] - Ccol[c0] + 1;
                    ok = false;
                }
            }
            if (ok) {  // group-uniform
                int bad = 0, lq = 0, lbn = 0, lan = 0, ne = 0;
                for (int p = a0 + r; p < a1; p += 16) {
                    const int K = op.Acol[p];
                    const int q0 = op.Bptr[K], q1 = op.Bptr[K + 1];
                    const int bn = op.Bnnz[q1] - op.Bnnz[q0];
                    bad |= q1 - q0 > G3_QB || bn > G3_BNNZ;
                    lq = max(lq, q1 - q0);
                    lbn = max(lbn, bn);
                    lan = max(lan, op.Annz[p + 1] - op.Annz[p]);
                }
                // nonempty C tiles (the row-wise kernel's slots) and those
                // followed by an accumulator pad
                int nbig = 0;
                for (int t = c0 + r; t < c1; t += 16) {
                    const int tn = Cnnz[t + 1] - Cnnz[t];
                    ne += tn > 0;
                    nbig += tn >= G3_PADMIN;
                }
                ok = g16_max(bad) == 0;
                ne = tsg_group16_sum(ne);
                nbig = tsg_group16_sum(nbig);
                lq = g16_max(lq); lbn = g16_max(lbn); lan = g16_max(lan);
                if (ok) {
                    mu = ne; mn = nrow + nbig; ml = a1 - a0; mq = lq; mb = lbn; ma = lan;
                }
            }
            k = lg ? LN_CLASS + lg - 1 : ok ? 1 : 0;
        }
        if (r == 0) cls[I] = k;
        unfit = r == 0 && k == 0;
        other = r == 0 && k <= 1;
        segs = unfit ? nrow / (G3F_NNZ - 255) + 1 : 0;
    }
    // the sums of a wave's four rows in one word (segments beyond counting: 2047 a row)
    const int sums = cls_sum(unfit | other << 8 | min(segs, 2047) << 16);
    unfit = sums & 255;
    other = (sums >> 8) & 255;
    segs = sums >> 16;
    mu = cls_max(mu); mn = cls_max(mn); ml = cls_max(ml);
    mq = cls_max(mq); mb = cls_max(mb); ma = cls_max(ma);
    ln = cls_max(ln); lu = cls_max(lu); ls = cls_max(ls); lg = cls_max(lg);
    if (lane == 0) {
        s_red[wave][0] = unfit; s_red[wave][1] = mu; s_red[wave][2] = mn; s_red[wave][3] = ml;
        s_red[wave][4] = mq; s_red[wave][5] = mb; s_red[wave][6] = ma;
        s_red[wave][7] = ln; s_red[wave][8] = lu; s_red[wave][9] = ls; s_red[wave][10] = lg;
        s_red[wave][11] = other; s_red[wave][12] = segs;
    }
    __syncthreads();
    if (threadIdx.x < CLS_WORDS) {
        const int i = threadIdx.x;
        int v = s_red[0][i];
#pragma unroll
        for (int w = 1; w < 4; w++) v = cls_sums(i) ? v + s_red[w][i] : max(v, s_red[w][i]);
        part[CLS_WORDS * (long long)blockIdx.x + i] = v;
        if (ticket) __threadfence();
    }
    if (!ticket) return;
    // few blocks: the last one to get here folds the partials
    __shared__ int s_last;
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(ticket, 1) == (int)gridDim.x - 1;
    __syncthreads();
    if (!s_last) return;
    __threadfence();
    for (int i = wave; i < CLS_WORDS; i += 4) {  // at most CLS_ONE blocks: a lane each, the words over the waves
        const int v = lane < (int)gridDim.x ? part[CLS_WORDS * lane + i] : 0;
        const int x = cls_sums(i) ? cls_sum(v) : cls_max(v);
        if (lane == 0) {
            out[i] = x;
            if (host) host[i] = x;
        }
    }
}

// out = sums (words 0, 11, 12) and maxima of the nb blocks' k_row_class partials
// (one block of 1024 threads).  host (may be NULL): pinned memory that gets
// the CLS_WORDS words too.
__global__ void __launch_bounds__(1024)
k_row_class_reduce(const int *__restrict__ part, int nb, int *__restrict__ out, int *__restrict__ host) {
    __shared__ int s_r[16][CLS_WORDS];
    int v[CLS_WORDS];
#pragma unroll
    for (int i = 0; i < CLS_WORDS; i++) v[i] = 0;
    for (int b = threadIdx.x; b < nb; b += 1024) {
        const int *p = part + CLS_WORDS * (long long)b;
#pragma unroll
        for (int i = 0; i < CLS_WORDS; i++) v[i] = cls_sums(i) ? v[i] + p[i] : max(v[i], p[i]);
    }
#pragma unroll
    for (int i = 0; i < CLS_WORDS; i++) v[i] = cls_sums(i) ? cls_sum(v[i]) : cls_max(v[i]);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int i = 0; i < CLS_WORDS; i++) s_r[wave][i] = v[i];
    __syncthreads();
    if (threadIdx.x < CLS_WORDS) {
        const int i = threadIdx.x;
        int r = s_r[0][i];
        for (int w = 1; w < 16; w++) r = cls_sums(i) ? r + s_r[w][i] : max(r, s_r[w][i]);
        out[i] = r;
        if (host) host[i] = r;
    }
}

// ------------------------------------------------------------------ host
// Step-1 count only: number of C tiles of A*B (structurally empty ones
// included), from the row-major tile indices.
extern "C" int tsg_spgemm_count_tiles(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, long long *out) {
    if (A->n != B->m) { tsg_set_error("count_tiles: inner dimensions differ"); return TSG_ERR_ARG; }
    int *cnt;
    TSG_TRY(tsg_alloc_t(ctx, &cnt, (size_t)A->tilem + 1));
    if (A->tilem > 0) {
        hipLaunchKernelGGL((k_step1<false, 256>), dim3(tsg_div_up(A->tilem, S1_WAVES)), dim3(64 * S1_WAVES), 0,
                           ctx->stream, A->tile_ptr, A->tile_colidx, A->tilem, B->tile_ptr, B->tile_colidx,
                           (const int4 *)nullptr, (const unsigned *)nullptr, (const int *)nullptr, cnt,
                           (int *)nullptr, (int *)nullptr, (unsigned *)nullptr, (int *)nullptr);
        TSG_LAUNCH_CHECK();
    }
    long long tot = 0;
    int st = tsg_scan_i32(ctx, cnt, cnt, A->tilem, &tot);
    tsg_free(ctx, cnt);
    *out = tot;
    return st;
}

// ------------------------------------------------------------------ no-allocation tile count
// tsg_spgemm_count_tiles_noalloc keeps its scratch in one fixed device
// array per GPU (loaded with the code object, held until the process
// ends): the per-tile-row C tile counts, then the per-block partial sums.
// Host code never passes the array's name to a kernel (there it is only a
// host-side stand-in); the device address comes from hipGetSymbolAddress,
// taken once per device with that device current, and kernels receive it
// as an argument.
#define NOALLOC_PARTS 1024  // partial sums (int64), at the end of the array
static_assert(TSG_NOALLOC_SCRATCH_BYTES % 256 == 0, "scratch is a whole number of 256-byte lines");
static_assert((long long)TSG_NOALLOC_MAX_TILE_ROWS * 4 + NOALLOC_PARTS * 8 <= TSG_NOALLOC_SCRATCH_BYTES,
              "counts and partials fit the scratch array");
static __device__ __align__(256) unsigned char scratch[TSG_NOALLOC_SCRATCH_BYTES];

#define NOALLOC_MAX_DEVICES 64
static std::mutex g_scratch_mu;
static unsigned char *g_scratch_dev[NOALLOC_MAX_DEVICES];  // device address of `scratch`, per device

static int noalloc_scratch(int device, unsigned char **out) {
    *out = nullptr;
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) {
        tsg_set_error("count_tiles_noalloc: device %d outside [0, %d)", device, NOALLOC_MAX_DEVICES);
        return TSG_ERR_ARG;
    }
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_dev[device]) {
        int cur = -1;
        TSG_HIP(hipGetDevice(&cur));
        if (cur != device) TSG_HIP(hipSetDevice(device));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess || !p) {
            tsg_set_error("count_tiles_noalloc: hipGetSymbolAddress(scratch) on device %d -> %s", device,
                          hipGetErrorString(e));
            return TSG_ERR_HIP;
        }
        g_scratch_dev[device] = static_cast<unsigned char *>(p);
    }
    *out = g_scratch_dev[device];
    return TSG_OK;
}

// Sum of n int32 counts: block b adds a grid-stride share into part[b]
// (every slot written, so nothing needs clearing), then one block adds the
// partials into *out.
__global__ void __launch_bounds__(256)
k_noalloc_partial(const int *__restrict__ cnt, int n, long long *__restrict__ part) {
    long long s = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) s += cnt[i];
    s = tsg_wave_sum(s);
    __shared__ long long w[4];
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = w[0] + w[1] + w[2] + w[3];
}
__global__ void __launch_bounds__(256)
k_noalloc_final(const long long *__restrict__ part, int nparts, long long *__restrict__ out) {
    long long s = 0;
    for (int i = threadIdx.x; i < nparts; i += 256) s += part[i];
    s = tsg_wave_sum(s);
    __shared__ long long w[4];
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *out = w[0] + w[1] + w[2] + w[3];
}

extern "C" int tsg_spgemm_count_tiles_noalloc(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B,
                                              long long *d_out) {
    if (!ctx || !A || !B || !d_out) { tsg_set_error("count_tiles_noalloc: null argument"); return TSG_ERR_ARG; }
    if (A->n != B->m) { tsg_set_error("count_tiles_noalloc: inner dimensions differ"); return TSG_ERR_ARG; }
    if (A->tilem < 0 || A->tilem > TSG_NOALLOC_MAX_TILE_ROWS) {
        tsg_set_error("count_tiles_noalloc: A has %d tile-rows; the fixed scratch holds at most %d", A->tilem,
                      TSG_NOALLOC_MAX_TILE_ROWS);
        return TSG_ERR_ARG;
    }
    if (A->tilem > 0 && (!A->tile_ptr || !A->tile_colidx || !B->tile_ptr || !B->tile_colidx)) {
        tsg_set_error("count_tiles_noalloc: missing tile index arrays");
        return TSG_ERR_ARG;
    }
    unsigned char *scr;
    TSG_TRY(noalloc_scratch(ctx->device, &scr));
    int *cnt = reinterpret_cast<int *>(scr);
    long long *part = reinterpret_cast<long long *>(scr + TSG_NOALLOC_SCRATCH_BYTES - NOALLOC_PARTS * 8);
    int nparts = (int)std::min<long long>(NOALLOC_PARTS, std::max(1u, tsg_div_up(A->tilem, 256)));
    if (A->tilem > 0) {
        hipLaunchKernelGGL((k_step1<false, 256>), dim3(tsg_div_up(A->tilem, S1_WAVES)), dim3(64 * S1_WAVES), 0,
                           ctx->stream, A->tile_ptr, A->tile_colidx, A->tilem, B->tile_ptr, B->tile_colidx,
                           (const int4 *)nullptr, (const unsigned *)nullptr, (const int *)nullptr, cnt,
                           (int *)nullptr, (int *)nullptr, (unsigned *)nullptr, (int *)nullptr);
        TSG_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_noalloc_partial, dim3(nparts), dim3(256), 0, ctx->stream, (const int *)cnt, A->tilem, part);
    hipLaunchKernelGGL(k_noalloc_final, dim3(1), dim3(256), 0, ctx->stream, (const long long *)part, nparts, d_out);
    TSG_LAUNCH_CHECK();
    return TSG_OK;
}

static int ev_ms(hipEvent_t a, hipEvent_t b, double *ms) {
    float f = 0.f;
    TSG_HIP(hipEventElapsedTime(&f, a, b));
    *ms = f;
    return TSG_OK;
}

// Launch helpers shared by the synchronous pipeline and the enqueue-only
// (graph-capturable) one.
static TileOperands make_operands(const tsg_dtiles *A, const tsg_dtiles *B) {
    TileOperands op;
    op.Aptr = A->tile_ptr; op.Acol = A->tile_colidx; op.Annz = A->tile_nnz; op.Aptr16 = A->csr_ptr;
    op.Amask = A->mask; op.Aval = A->val;
    op.Bptr = B->tile_ptr; op.Bcol = B->tile_colidx;
    op.Bcscptr = B->csc_ptr; op.Bcscrow = B->csc_rowidx; op.Bcscid = B->csc_tileid; op.Bnnz = B->tile_nnz;
    op.Bptr16 = B->csr_ptr; op.Bmask = B->mask; op.Bval = B->val;
    op.Arowp = A->rowx_ptr; op.Acolx = A->rowx_col; op.Avalx = A->rowx_val;
    return op;
}

// Step-1 bitmap window in 32-bit words per wave: 128 (4096 tile columns, 4 KiB
// of LDS per block with the pair lists), 256 (8192), 1024 (32768, 16 KiB) or
// 2048 (65536, 32 KiB).  By default B gets the narrowest window that holds all
// its tile columns up to 65536, so a row of a product without band structure needs
// one window, with no more LDS (and, for the kept-row bitmap ORs, registers) than
// that takes; wider B (banded operands such as stencils) keeps 256.  The words a
// lane does not hold are rows in flight: with 128 words eight kept B tile-rows
// are loaded together, with 256 two (hub tile-rows are one wave's chain of these
// loads).  Count pass with 256 / 128 words: R-MAT scale 16 A*A^T 965 / 640 us, ER 65521
// 143 / 94, ER 20011 77 / 43; twelve and sixteen rows together 627 / 634, 97 / 93,
// 45 / 43.  The count pass's bitmaps are kept for the fill pass up to 1 GiB.
int tsg_s1_words(const tsg_dtiles *B, const tsg_tune &t) {
    if (t.s1_window_words == 256 || t.s1_window_words == 1024 || t.s1_window_words == 2048) return t.s1_window_words;
    if (B->tilen <= 4096) return 128;
    if (B->tilen > 8192 && B->tilen <= 32768) return 1024;
    return B->tilen > 32768 && B->tilen <= 65536 ? 2048 : 256;
}
static size_t keep_bytes(long long tilem, int words) {
    const size_t b = (size_t)tilem * (size_t)words * 4;
    return b <= ((size_t)1 << 30) ? b : 0;
}

// B's tile-row bitmaps for step 1 (k_brow_desc, k_brow_fill): a descriptor
// per B tile-row, then the words.  0 when B has no tile row index or the
// word offsets would not fit 32 bits (step 1 then enumerates every
// candidate).
static size_t brow_bits_bytes(const tsg_dtiles *B) {
    if (!B || B->tilem <= 0 || !B->tile_rowidx) return 0;
    const long long words = 2ll * B->numtile + 2ll * B->tilem;
    if (words >= 0x7fffffffLL) return 0;
    return (size_t)B->tilem * 16 + (size_t)words * 4;
}
// scr: SCR_WORDS words to be cleared, any among them (both may be NULL)
static int launch_brow_bits(hipStream_t s, const tsg_dtiles *B, void *buf, const int4 **desc,
                            const unsigned **bits, int *scr, int *any, int *longest) {
    *desc = nullptr;
    *bits = nullptr;
    const bool make = buf && brow_bits_bytes(B), one = make && B->tilem <= BROW_ONE_ROWS && B->numtile <= BROW_ONE;
    if (scr && !one) TSG_HIP(hipMemsetAsync(scr, 0, 4 * SCR_WORDS, s));
    if (!make) return TSG_OK;
    int4 *d = (int4 *)buf;
    unsigned *w = (unsigned *)((char *)buf + (size_t)B->tilem * 16);
    const int *browp = B->rowx_ptr;
    if (!browp) longest = nullptr;
    if (one) {
        hipLaunchKernelGGL(k_brow_one, dim3(1), dim3(1024), 0, s, (const int *)B->tile_ptr, (const int *)B->tile_rowidx,
                           (const int *)B->tile_colidx, B->tilem, B->numtile, d, w, scr, any, browp, B->m, longest);
    } else {
        hipLaunchKernelGGL(k_brow_desc, dim3(tsg_div_up(B->tilem, 256)), dim3(256), 0, s, (const int *)B->tile_ptr,
                           (const int *)B->tile_colidx, B->tilem, d, any, browp, B->m, longest);
        if (B->numtile > 0)
            hipLaunchKernelGGL(k_brow_fill, dim3(tsg_div_up(B->numtile, 256)), dim3(256), 0, s,
                               (const int *)B->tile_rowidx, (const int *)B->tile_colidx, (long long)B->numtile,
                               (const int4 *)d, w, (const int *)any);
    }
    TSG_LAUNCH_CHECK();
    *desc = d;
    *bits = w;
    return TSG_OK;
}

template <int BMW>
static void launch_step1_w(hipStream_t s, const tsg_dtiles *A, const tsg_dtiles *B, tsg_dtiles *C, bool fill,
                           unsigned *bmstore, const int4 *bdesc, const unsigned *bbits, const int *bany, int *rowspan) {
    const dim3 g(tsg_div_up(C->tilem, S1_WAVES)), blk(64 * S1_WAVES);
    if (fill)
        hipLaunchKernelGGL((k_step1<true, BMW>), g, blk, 0, s, A->tile_ptr, A->tile_colidx, A->tilem, B->tile_ptr,
                           B->tile_colidx, bdesc, bbits, bany, C->tile_ptr, C->tile_colidx, C->tile_rowidx, bmstore,
                           rowspan);
    else
        hipLaunchKernelGGL((k_step1<false, BMW>), g, blk, 0, s, A->tile_ptr, A->tile_colidx, A->tilem, B->tile_ptr,
                           B->tile_colidx, bdesc, bbits, bany, C->tile_ptr, (int *)nullptr, (int *)nullptr, bmstore,
                           rowspan);
}
static int launch_step1(hipStream_t s, const tsg_dtiles *A, const tsg_dtiles *B, tsg_dtiles *C, bool fill,
                        int words, unsigned *bmstore, const int4 *bdesc, const unsigned *bbits,
                        const int *bany, int *rowspan) {
    if (C->tilem <= 0) return TSG_OK;
    auto launch = words == 128    ? launch_step1_w<128>
                  : words == 1024 ? launch_step1_w<1024>
                  : words == 2048 ? launch_step1_w<2048>
                                  : launch_step1_w<256>;
    launch(s, A, B, C, fill, bmstore, bdesc, bbits, bany, rowspan);
    TSG_LAUNCH_CHECK();
    return TSG_OK;
}

// Device scratch of one SpGEMM beyond C itself.
struct SpgemmWork {
    long long *part1;  // scan partials: C tile pointers
    long long *part2;  // scan partials: C tile nnz
    long long *part3;  // scan partials: segment counts
    int *segcnt;       // tilem+1 step-3 segment counts -> offsets (total at [tilem])
    int *segctr;       // S2_KINDS step-2 segment counters
    unsigned char *rowcls;
    int *cls_out;
    int *cls_part;  // k_row_class partials, CLS_WORDS ints per block
    void *bbits;       // B's tile-row bitmaps for step 1 (may be NULL)
    int *longest;      // longest row of each B tile-row (enqueue-only pipeline)
    int4 *seg2;        // step-2 segments
    unsigned *bmstore; // step-1 bitmaps kept from the count pass (may be NULL)
    int4 *seg3;        // step-3 element segments
    long long seg3_cap;
    // heavy rows (synchronous pipeline only; NULL = none)
    unsigned char *hflag;  // per C row
    int4 *hrows;           // the heavy rows, the long ones
    int nheavy, nlong, ncounted;
    int hstep, lstep;      // blocks of a heavy row, of a long one
    int lchunk;            // long rows taken part by part together
    const int *hwin;       // B rows' window table (k_heavy_windows), its stride and shift
    long long hstride, hwin_bytes;
    int hnw, hshift;
};

static size_t up16(size_t x) { return (x + 15) & ~(size_t)15; }

// Offsets of the work arrays inside one buffer; returns its size.  The
// step-3 segments go last (the synchronous pipeline adds them only once
// C's nonzero count is known).
#define WORK_NARR 12

static size_t work_layout(long long tilem, long long numtile, long long nnz, size_t off[WORK_NARR],
                          int s1w = 256, size_t bbytes = 0, size_t longest_bytes = 0) {
    const size_t sz[WORK_NARR] = {
        8 * (size_t)tsg_scan_partial_count(tilem), 8 * (size_t)tsg_scan_partial_count(numtile),
        8 * (size_t)tsg_scan_partial_count(tilem), 4 * ((size_t)tilem + 1), (size_t)tilem + 1, 4 * CLS_WORDS,
        16 * (size_t)seg2_bound(tilem, numtile),
        keep_bytes(tilem, s1w),  // step-1 bitmaps (enqueue-only pipeline)
        4 * CLS_WORDS * (size_t)((tilem + 15) / 16 + 1),  // row-class partials
        bbytes + longest_bytes,                // B's tile-row bitmaps, longest rows (enqueue-only pipeline)
        4 * S2_KINDS,
        16 * (size_t)(tilem + nnz / (G3E_NNZ - 255) + 2)};
    size_t o = 0;
    for (int i = 0; i < WORK_NARR; i++) {
        off[i] = o;
        o += up16(sz[i]);
    }
    return o;
}

static SpgemmWork work_at(void *base, long long tilem, long long numtile, long long nnz, void *seg3_base,
                          int s1w = 256, size_t bbytes = 0, size_t longest_bytes = 0) {
    size_t off[WORK_NARR];
    work_layout(tilem, numtile, nnz, off, s1w, bbytes, bbytes ? longest_bytes : 0);
    char *b = (char *)base;
    SpgemmWork w;
    w.part1 = (long long *)(b + off[0]);
    w.part2 = (long long *)(b + off[1]);
    w.part3 = (long long *)(b + off[2]);
    w.segcnt = (int *)(b + off[3]);
    w.rowcls = (unsigned char *)(b + off[4]);
    w.cls_out = (int *)(b + off[5]);
    w.seg2 = (int4 *)(b + off[6]);
    w.bmstore = keep_bytes(tilem, s1w) ? (unsigned *)(b + off[7]) : nullptr;
    w.cls_part = (int *)(b + off[8]);
    w.bbits = bbytes ? (void *)(b + off[9]) : nullptr;
    w.longest = bbytes ? (int *)(b + off[9] + bbytes) : nullptr;
    w.segctr = (int *)(b + off[10]);
    w.seg3 = (int4 *)(seg3_base ? (char *)seg3_base : b + off[11]);
    w.seg3_cap = tilem + nnz / (G3E_NNZ - 255) + 2;
    w.hflag = nullptr;
    w.hrows = nullptr;
    w.nheavy = w.nlong = w.ncounted = w.hstep = w.lstep = w.lchunk = w.hnw = w.hshift = 0;
    w.hwin = nullptr;
    w.hstride = w.hwin_bytes = 0;
    return w;
}

// Step-3 element segments of the tile-rows of class `want` into w.seg3 (cap
// = its capacity, at least the count); the count lands in w.segcnt[tilem].
static int launch_segments(hipStream_t s, const tsg_dtiles *C, const SpgemmWork &w, int want, int max_nnz,
                           const unsigned char *cls) {
    hipLaunchKernelGGL(k_seg1_count, dim3(tsg_div_up(C->tilem, 256)), dim3(256), 0, s, C->tile_ptr, C->tile_nnz,
                       C->tilem, cls, want, max_nnz, w.segcnt);
    TSG_LAUNCH_CHECK();
    TSG_TRY(tsg_scan_i32_enqueue(s, w.segcnt, w.segcnt, C->tilem, w.part3));
    if (w.seg3_cap > 0) {
        hipLaunchKernelGGL(k_seg1_fill, dim3((unsigned)tsg_div_up(w.seg3_cap, 256)), dim3(256), 0, s, C->tile_ptr,
                           C->tile_nnz, C->tilem, (const int *)w.segcnt, max_nnz, w.seg3);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

static int launch_step2(hipStream_t s, const TileOperands &op, const tsg_dtiles *B, tsg_dtiles *C,
                        const tsg_spgemm_plan &P, const SpgemmWork &w) {
    if (C->numtile <= 0) return TSG_OK;
    if (P.all) {
        const unsigned nblk = tp_grid(tsg_div_up(C->numtile, S23_WAVES * TILES_PER_WAVE));
        hipLaunchKernelGGL(k_step2_tiles, dim3(nblk), dim3(64 * S23_WAVES), 0, s, op, C->tile_rowidx, C->tile_colidx, C->numtile,
                           C->mask, C->csr_ptr, C->tile_nnz);
        TSG_LAUNCH_CHECK();
        return TSG_OK;
    }
    const int *n2 = P.n2;
    // only tile-row-long tile-pair segments: no list
    const bool list = n2[1] || n2[2] || n2[3] || P.s2u >= G2_UMAX;
    const int4 base = make_int4(0, n2[0], n2[0] + n2[1], n2[0] + n2[1] + n2[2]);
    if (list) {
        hipLaunchKernelGGL(k_seg2_fill, dim3(tsg_div_up(C->tilem, 256)), dim3(256), 0, s, C->tile_ptr, C->tile_colidx,
                           op.Aptr, op.Annz, C->tilem, P.s3_elem, P.elem_all, op.Arowp ? 1 : 0, base, w.segctr, w.seg2);
        TSG_LAUNCH_CHECK();
    }
    if (n2[0] > 0) {
        const int s2u = P.s2u > 0 ? P.s2u : G2_UMAX;
        const size_t lds2 = (4 * G2_MSTRIDE + 4) * (size_t)s2u + (((size_t)P.s2map + 15) & ~(size_t)15);
        const int nseg = list ? n2[0] : C->tilem;
        hipLaunchKernelGGL(k_step2_rows, tsg_grid(nseg, G2_THREADS), dim3(G2_THREADS), lds2, s, op,
                           list ? (const int4 *)w.seg2 : (const int4 *)nullptr, nseg, C->tile_ptr, C->tile_colidx, C->mask,
                           C->csr_ptr, C->tile_nnz, s2u, P.s2map);
        TSG_LAUNCH_CHECK();
    }
    if (n2[1] > 0) {
        hipLaunchKernelGGL(k_step2_elem, tsg_grid(n2[1], G2_THREADS), dim3(G2_THREADS), 0, s, op, (const int *)B->rowx_ptr,
                           (const int *)B->rowx_col, (const int4 *)(w.seg2 + base.y), n2[1], C->tile_ptr, C->tile_colidx,
                           C->mask, C->csr_ptr, C->tile_nnz);
        TSG_LAUNCH_CHECK();
    }
    for (int k = 2; k < 4; k++) {
        if (n2[k] <= 0) continue;
        const int width = k == 2 ? P.s2w : G2D_WIN;
        const int threads = k == 2 ? 256 : 1024;
        const size_t lds = g2d_lds(width, threads);
        // kind 3: a few blocks per CU take the windows in turn (one at a time fits)
        const unsigned grid = (unsigned)std::min(n2[k], k == 2 ? 1 << 23 : 4096);
        hipLaunchKernelGGL(k_step2_dense, dim3(grid), dim3(threads), lds, s, op.Arowp, op.Acolx, C->m,
                           (const int *)B->rowx_ptr, (const int *)B->rowx_col,
                           (const int4 *)(w.seg2 + (k == 2 ? base.z : base.w)), n2[k], C->tile_ptr, C->tile_colidx,
                           C->mask, C->csr_ptr, C->tile_nnz, width);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

// ticket (may be NULL): a cleared word for k_row_class's last block
#define CLS_ONE 64
static_assert(CLS_ONE <= 64, "k_row_class folds a block per lane");
static int launch_row_class(hipStream_t s, const TileOperands &op, tsg_dtiles *C, unsigned char *rowcls,
                            int *cls_part, int *cls_out, int none_fit, const int *longest, int *ticket = nullptr,
                            int *host = nullptr) {
    const int nb = (int)tsg_div_up(C->tilem, 16);
    if (nb > CLS_ONE) ticket = nullptr;
    hipLaunchKernelGGL(k_row_class, dim3(nb), dim3(256), 0, s, op, C->tile_ptr, C->tile_colidx, C->tile_nnz, C->tilem,
                       rowcls, cls_part, none_fit, longest, ticket, cls_out, host);
    TSG_LAUNCH_CHECK();
    if (!ticket) {
        hipLaunchKernelGGL(k_row_class_reduce, dim3(1), dim3(1024), 0, s, (const int *)cls_part, nb, cls_out, host);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

static int launch_step3(hipStream_t s, const TileOperands &op, const tsg_dtiles *B, tsg_dtiles *C,
                        const tsg_spgemm_plan &P, const SpgemmWork &w, hipEvent_t *ev = nullptr) {
    if (C->nnz <= 0) return TSG_OK;
    const bool rows = !P.all && (P.s3_lines || P.s3_rows);
    if (ev && rows) TSG_HIP(hipEventRecord(ev[0], s));
    if (!P.all && P.s3_lines) {
        LinesLayout L;
        L.nnz = P.ln[0]; L.umax = P.ln[1]; L.map = P.ln[2];
        int base;
        size_t off[4];
        hipLaunchKernelGGL(k_step3_lines, tsg_grid(C->tilem, P.ln[3]), dim3(P.ln[3]), lines_layout(L, &base, off), s, op.Arowp, op.Acolx,
                           op.Avalx, (const int *)B->rowx_ptr, (const int *)B->rowx_col, (const double *)B->rowx_val,
                           C->m, C->tilem, C->tile_ptr, C->tile_colidx, C->mask, C->csr_ptr, C->tile_nnz,
                           (const unsigned char *)w.rowcls, C->csr_col, C->val, L);
        TSG_LAUNCH_CHECK();
    }
    if (!P.all && P.s3_rows) {
        G3Layout L;
        L.umax = P.g3[0]; L.nnzmax = P.g3[1]; L.lamax = P.g3[2];
        L.qb = P.g3[3]; L.bnnz = P.g3[4]; L.amax = P.g3[5];
        size_t off[G3_NARR];
        const size_t lds = g3_layout(L, off);
        hipLaunchKernelGGL(k_step3_rows, tsg_grid(C->tilem, G3_THREADS), dim3(G3_THREADS), lds, s, op, C->tile_ptr, C->tile_colidx,
                           C->tilem, C->mask, C->csr_ptr, C->tile_nnz, (const unsigned char *)w.rowcls, C->csr_col,
                           C->val, L);
        TSG_LAUNCH_CHECK();
    }
    if (ev && rows) TSG_HIP(hipEventRecord(ev[1], s));
    if (!P.all && P.s3_unfit && P.s3_elem) {
        const bool rx = op.Arowp != nullptr;
        TSG_TRY(launch_segments(s, C, w, 0, rx ? G3F_NNZ : G3E_NNZ, w.rowcls));
        if (rx)
            hipLaunchKernelGGL(P.s3span < G3F_SPAN ? k_step3_flat<false> : k_step3_flat<true>, tsg_grid(w.seg3_cap, G3F_THREADS), dim3(G3F_THREADS), 0, s, op.Arowp, op.Acolx,
                               op.Avalx, (const int *)B->rowx_ptr, (const int *)B->rowx_col,
                               (const double *)B->rowx_val, C->m, (const int4 *)w.seg3,
                               (const int *)(w.segcnt + C->tilem), C->tile_ptr, C->tile_colidx, C->mask, C->csr_ptr,
                               C->tile_nnz, C->csr_col, C->val, (const unsigned char *)w.hflag);
        else
            hipLaunchKernelGGL(P.s3span < G3E_PK_SPAN ? k_step3_elem<true> : k_step3_elem<false>,
                               tsg_grid(w.seg3_cap, 256), dim3(256), 0, s, op, (const int *)B->rowx_ptr,
                               (const int *)B->rowx_col, (const double *)B->rowx_val, C->m, (const int4 *)w.seg3,
                               (const int *)(w.segcnt + C->tilem), C->tile_ptr, C->tile_colidx, C->mask, C->csr_ptr,
                               C->tile_nnz, C->csr_col, C->val);
        TSG_LAUNCH_CHECK();
        if (w.hflag) {
            const long long total = heavy_padded(w.nheavy) * (long long)w.hstep + heavy_padded(w.nlong) * (long long)w.lstep;
            for (long long at = 0; at < total; at += 1 << 25) {  // a launch takes fewer than 2^32 threads
                hipLaunchKernelGGL(k_step3_heavy, dim3((unsigned)std::min(total - at, 1LL << 25)), dim3(64), 0, s,
                                   op.Arowp, op.Acolx, op.Avalx, w.hwin, w.hstride, w.hnw, w.hshift,
                                   (const int *)B->rowx_col, (const double *)B->rowx_val, (const int4 *)w.hrows,
                                   w.nheavy, w.nlong, w.hstep, w.lstep, w.lchunk, at, C->tile_ptr, C->tile_colidx, C->mask, C->csr_ptr,
                                   C->tile_nnz, C->csr_col, C->val);
                TSG_LAUNCH_CHECK();
            }
        }
    } else if (P.all || P.s3_unfit) {
        const unsigned nblk = tp_grid(tsg_div_up(C->numtile, S23_WAVES * TILES_PER_WAVE));
        hipLaunchKernelGGL(k_step3, dim3(nblk), dim3(64 * S23_WAVES), 0, s, op, C->tile_ptr, C->tile_rowidx,
                           C->tile_colidx, C->numtile, C->mask, C->csr_ptr, C->tile_nnz, C->csr_col, C->val,
                           P.dense_min, P.all, (const unsigned char *)w.rowcls);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}

static int alloc_c_tiles(tsg_ctx *ctx, tsg_dtiles *C, long long numtileC) {
    TSG_TRY(tsg_alloc_t(ctx, &C->tile_colidx, (size_t)numtileC + 1));
    TSG_TRY(tsg_alloc_t(ctx, &C->tile_rowidx, (size_t)numtileC + 1));
    TSG_TRY(tsg_alloc_t(ctx, &C->mask, (size_t)numtileC * 16 + 16));
    TSG_TRY(tsg_alloc_t(ctx, &C->csr_ptr, (size_t)numtileC * 16 + 16));
    TSG_TRY(tsg_alloc_t(ctx, &C->tile_nnz, (size_t)numtileC + 1));
    return TSG_OK;
}

// Temporaries of one pipeline run, freed on every exit (stream-ordered: the
// caching allocator hands a block out again only behind the work queued on
// the context stream).
struct SpgemmTemps {
    unsigned *keep = nullptr;
    void *scr = nullptr, *wbuf = nullptr, *w3buf = nullptr, *bb = nullptr;
    unsigned char *hflag = nullptr;
    int *hcnt = nullptr, *hinfo = nullptr, *hwin = nullptr, *span = nullptr, *longest = nullptr;
    int4 *hrows = nullptr;
    tsg_dcsr rowx[2] = {};
    hipEvent_t ev[6] = {};
    int nev = 0;
};

static void free_temps(tsg_ctx *ctx, SpgemmTemps &t) {
    void *ps[] = {t.keep, t.scr, t.wbuf, t.w3buf, t.hflag, t.hcnt, t.hinfo, t.hwin, t.hrows, t.span, t.bb, t.longest};
    for (void *p : ps) tsg_free(ctx, p);
    for (tsg_dcsr &r : t.rowx) tsg_dcsr_free(ctx, &r);
    for (int i = 0; i < t.nev; i++) (void)hipEventDestroy(t.ev[i]);
    t = SpgemmTemps();
}

// Row indices made for one product whose operands have none: worth it when
// most tile-rows will go by row lines.  The index costs one pass over an operand.
// A^2 without / with it: 27-point 128^3 5.54 / 3.91 ms, 61x47x53 605 / 396 us,
// 36x33x37 (1.1 M entries) 252 / 188, 5-point 700x310 326 / 251, banded 90000
// (half-bandwidth 6) 283 / 182.  Below a million entries its launches and
// read-back weigh as much; hypersparse tiles mostly have more C tiles than row
// lines take; and rows of more than LN_BROW entries would leave dense tiles to
// k_step3_flat (banded 20000, half-bandwidth 64, 626 / 939 us).
#define AUTO_INDEX_NNZ (1 << 20)
#define AUTO_INDEX_TILE 4  // entries per tile
#define AUTO_INDEX_ROW 96  // entries per row
// The index is read off the tiles' entries, in-tile columns among them, which
// steps 1 to 3 do without: an operand may come without csr_col (the drop-in
// entry point's, and tsg_tiles_from_csc_order's of one that has none) and then
// stays on the tile kernels.
#define ELEM_MAX_N ((1 << 27) - 32)  // columns of a B that the element kernels take
static bool auto_index(const tsg_dtiles *t) {
    return t->csr_col && t->nnz >= AUTO_INDEX_NNZ && t->nnz >= AUTO_INDEX_TILE * (long long)t->numtile &&
           t->nnz <= AUTO_INDEX_ROW * (long long)t->m;
}
// Tiles dense enough (28 entries and more, which meet in some 50 products), and
// few enough to a tile-row of A and a tile column of B, that k_step3 is the
// better one for many tile-rows that row lines do not take.  Then the index is
// made after step 2, when the classes of the tile-rows are known: where at
// least half go by lines and the rest is few enough to run at once as segments of
// k_step3_flat (if C's tiles have several pairs: one of k_step3 is a chain of
// them), or where seven in eight go by lines (and the rest by k_step3); else not at all.  A^2, index before
// step 1 with the rest in segments / index after step 2 with the rest by k_step3 /
// no index: bands of half-width 10 and 64, 20% of the rows wide (375 tile-rows,
// 750 segments) 0.50 / 0.67 / 0.74 ms, 50% (1870 segments) 0.86 / 0.80 / 0.79; 12 and 70,
// 60000 rows, 10% wide 0.61 / 0.91 / 1.06; 20 and 100, 30% wide (1690) 1.10 / 1.25 /
// 1.11; random tiles, 8 of 48 entries a tile-row, none by lines, 0.63 / - / 0.35, within
// 8 of the diagonal (1.9 pairs), most by lines, 0.37 / 0.29 / 0.38; 5 of 200 there (1.3
// pairs) 0.40 / 0.39 / 0.33.
#define AUTO_DENSE_TILE 28  // entries per tile, geometric mean of A and B
#define AUTO_DENSE_LIST 16  // tiles per tile-row of A and per tile column of B
#define AUTO_SEGMENTS 1536  // four blocks of k_step3_flat fit a CU
#define AUTO_PAIRS 1.6      // per tile of C
static bool auto_dense(const tsg_dtiles *A, const tsg_dtiles *B) {
    return (double)A->nnz * B->nnz >= (double)(AUTO_DENSE_TILE * AUTO_DENSE_TILE) * A->numtile * B->numtile &&
           A->numtile <= AUTO_DENSE_LIST * (long long)A->tilem && B->numtile <= AUTO_DENSE_LIST * (long long)B->tilen;
}
// longest[K] = entries of the longest row of B's tile-row K, from its masks: 16 lanes a tile-row, a row each.
__global__ void __launch_bounds__(256)
k_longest_rows(const int *__restrict__ Bptr, const unsigned short *__restrict__ Bmask, int tilem, int *__restrict__ longest) {
    const int K = blockIdx.x * 16 + (threadIdx.x >> 4), r = threadIdx.x & 15;
    if (K >= tilem) return;
    int c = 0;
    for (int t = Bptr[K]; t < Bptr[K + 1]; t++) c += __popc((unsigned)Bmask[(long long)t * 16 + r]);
    c = g16_max(c);
    if (r == 0) longest[K] = c;
}
static int make_index(tsg_ctx *ctx, const tsg_dtiles *t, tsg_dcsr *r, tsg_dtiles *with) {
    *with = *t;
    const int st = tsg_tile2csr(ctx, t, r);
    if (st == TSG_OK) {
        with->rowx_ptr = r->rowptr;
        with->rowx_col = r->colidx;
        with->rowx_val = r->val;
    }
    return st == TSG_ERR_NOMEM ? TSG_OK : st;  // no room: the tile kernels need none
}

// symbolic: steps 1 and 2 and the step-3 plan (row classes, element
// segments, heavy-row work list) only; C's values and in-tile columns are
// neither allocated nor computed.  stats then carries C's exact tile and
// nonzero counts and the heavy-row scratch the numeric step would add.
static int spgemm_run(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, const tsg_tune *tune_in,
                      tsg_dtiles *C, tsg_stats *stats, tsg_spgemm_plan *plan_out, bool symbolic, bool may_index,
                      SpgemmTemps &T) {
    if (!A || !B || A->n != B->m) {
        tsg_set_error("tsg_spgemm: inner dimensions differ (%d vs %d)", A ? A->n : -1, B ? B->m : -1);
        return TSG_ERR_ARG;
    }
    if (!B->csc_ptr) { tsg_set_error("tsg_spgemm: B needs its CSC tile index (tsg_tiles_build_csc)"); return TSG_ERR_STATE; }
    tsg_tune tune;
    if (tune_in) tune = *tune_in; else tsg_tune_default(&tune);
    if (tune.dense_acc_min_nnz < 1) tune.dense_acc_min_nnz = 1;
    tsg_spgemm_plan P;
    memset(&P, 0, sizeof(P));
    P.all = tune.force_tile_parallel ? 1 : 0;
    P.dense_min = tune.dense_acc_min_nnz;
    hipStream_t s = ctx->stream;

    hipEvent_t *ev = T.ev;
    const bool timed = stats != nullptr;
    if (timed) {
        memset(stats, 0, sizeof(*stats));
        for (; T.nev < 6; T.nev++) TSG_HIP(hipEventCreate(&ev[T.nev]));
        TSG_HIP(hipEventRecord(ev[0], s));
        TSG_HIP(hipEventRecord(ev[4], s));
        TSG_HIP(hipEventRecord(ev[5], s));
    }
    tsg_dtiles ax, bx;
    may_index = may_index && tune.element_mode == 0 && !P.all && B->n <= ELEM_MAX_N && !(A->rowx_ptr && B->rowx_ptr) &&
                auto_index(A) && auto_index(B);
    auto index_operands = [&]() -> int {
        auto borrow = [](const tsg_dtiles *t, const tsg_dtiles *from, tsg_dtiles *with) {
            *with = *t;
            with->rowx_ptr = from->rowx_ptr;
            with->rowx_col = from->rowx_col;
            with->rowx_val = from->rowx_val;
        };
        // one matrix: either's index is the other's.  Every array it is read from
        // and every size counts: A may be B's leading tile-rows (the same arrays,
        // fewer rows), or share all but one of them
        const bool same = A->m == B->m && A->n == B->n && A->numtile == B->numtile && A->nnz == B->nnz &&
                          A->tile_ptr == B->tile_ptr && A->tile_colidx == B->tile_colidx && A->tile_nnz == B->tile_nnz &&
                          A->csr_ptr == B->csr_ptr && A->csr_col == B->csr_col && A->val == B->val;
        if (!A->rowx_ptr) {
            if (same && B->rowx_ptr) borrow(A, B, &ax);
            else TSG_TRY(make_index(ctx, A, &T.rowx[0], &ax));
            A = &ax;
        }
        if (!B->rowx_ptr) {
            if (same) borrow(B, A, &bx);
            else TSG_TRY(make_index(ctx, B, &T.rowx[1], &bx));
            B = &bx;
        }
        return TSG_OK;
    };
    const bool index_later = may_index && !B->rowx_ptr && auto_dense(A, B);
    if (may_index && !index_later) TSG_TRY(index_operands());
    // element path: B carries its row index, and C's columns fit the
    // 28-bit entry keys of the element kernel's LDS hash
    // element-wise keys: (column offset) << 4 in 32 bits, and tile columns
    // below 2^23 - 1 for the step-2 hash slots
    P.s3_elem = B->rowx_ptr != nullptr && tune.element_mode != 1 && B->n <= ELEM_MAX_N;
    P.elem_all = B->rowx_ptr != nullptr && tune.element_mode == 2;
    P.lines = A->rowx_ptr && P.s3_elem && !P.elem_all && brow_bits_bytes(B) > 0;
    C->m = A->m;
    C->n = B->n;
    C->tilem = A->tilem;
    C->tilen = B->tilen;
    // ---- step 1
    TSG_TRY(tsg_alloc_t(ctx, &C->tile_ptr, (size_t)C->tilem + 1));
    if (tune.s1_window_words != 0 && tune.s1_window_words != 256 && tune.s1_window_words != 1024 &&
        tune.s1_window_words != 2048) {
        tsg_set_error("spgemm: s1_window_words %d is not 0, 256, 1024 or 2048", tune.s1_window_words);
        return TSG_ERR_ARG;
    }
    P.s1w = tsg_s1_words(B, tune);
    const size_t kb = keep_bytes(C->tilem, P.s1w);
    if (kb) TSG_TRY(tsg_alloc(ctx, (void **)&T.keep, kb));
    static_assert(4 * SCR_WORDS == 128, "bins, flags, row statistics");
    TSG_TRY(tsg_alloc(ctx, &T.scr, 128));
    void *scr = T.scr;
    unsigned long long *bins = (unsigned long long *)scr;
    int *bany = reinterpret_cast<int *>(static_cast<char *>(scr) + 32);  // some B tile-row bitmap kept
    int *st2 = reinterpret_cast<int *>(static_cast<char *>(scr) + 64);   // k_row_stats
    int *ticket = reinterpret_cast<int *>(static_cast<char *>(scr) + 36);  // k_row_class
    TSG_TRY(tsg_alloc_t(ctx, &T.span, (size_t)C->tilem + 1));
    const int4 *bdesc = nullptr;
    const unsigned *bbits = nullptr;
    if (const size_t bbb = C->tilem > 0 ? brow_bits_bytes(B) : 0) {
        TSG_TRY(tsg_alloc(ctx, &T.bb, bbb));
        if (P.lines) TSG_TRY(tsg_alloc_t(ctx, &T.longest, (size_t)B->tilem));
    }
    TSG_TRY(launch_brow_bits(s, B, T.bb, &bdesc, &bbits, (int *)scr, bany, T.longest));
    TSG_TRY(launch_step1(s, A, B, C, false, P.s1w, T.keep, bdesc, bbits, bany, T.span));
    // C's tile-row offsets; their total and the step-2 sizing maxima come
    // back in one read-back
    long long numtileC = 0;
    int smax[ROW_STATS] = {};
    const int rx = A->rowx_ptr ? 1 : 0;
    if (C->tilem > 0 && C->tilem <= ROW_STATS_ONE) {
        hipLaunchKernelGGL(k_row_stats_one, dim3(1), dim3(1024), 0, s, C->tile_ptr, (const int *)T.span, A->tile_ptr,
                           A->tile_nnz, C->tilem, P.s3_elem, P.elem_all, rx, ctx->pinned);
        TSG_LAUNCH_CHECK();
        TSG_HIP(hipStreamSynchronize(s));
        numtileC = *(volatile long long *)ctx->pinned;
        if (numtileC > 0x7fffffffLL) {
            tsg_set_error("prefix sum total %lld exceeds int32", numtileC);
            return TSG_ERR_OVERFLOW;
        }
    } else {
        if (C->tilem > 0) {
            hipLaunchKernelGGL(k_row_stats, dim3(std::min<unsigned>(ROW_STATS_BLOCKS, tsg_div_up(C->tilem, 1024))),
                               dim3(1024), 0, s, (const int *)C->tile_ptr, (const int *)T.span, A->tile_ptr,
                               A->tile_nnz, C->tilem, P.s3_elem, P.elem_all, rx, st2);
            TSG_LAUNCH_CHECK();
        }
        TSG_TRY(tsg_scan_i32(ctx, C->tile_ptr, C->tile_ptr, C->tilem, &numtileC, st2, ROW_STATS));
    }
    memcpy(smax, ctx->pinned + 1, sizeof(smax));
    tsg_free(ctx, T.span);
    T.span = nullptr;
    P.numtileC = numtileC;
    C->numtile = (int)numtileC;
    TSG_TRY(alloc_c_tiles(ctx, C, numtileC));
    size_t woff[WORK_NARR];
    const size_t wbytes = work_layout(C->tilem, numtileC, 0, woff);
    TSG_TRY(tsg_alloc(ctx, &T.wbuf, woff[WORK_NARR - 1]));  // everything but the step-3 segments
    (void)wbytes;
    void *wbuf = T.wbuf;
    SpgemmWork w = work_at(wbuf, C->tilem, numtileC, 0, nullptr);
    TSG_TRY(launch_step1(s, A, B, C, true, P.s1w, T.keep, bdesc, bbits, bany, w.segctr));
    tsg_free(ctx, T.keep);
    T.keep = nullptr;
    tsg_free(ctx, T.bb);
    T.bb = nullptr;
    if (timed) TSG_HIP(hipEventRecord(ev[1], s));
    // step-2 LDS sizing: the largest segment and the widest tile-row span
    P.s2u = G2_UMAX;
    P.s2map = 0;
    if (numtileC > 0) {
        const int umax = smax[0], span = smax[1], mspan = smax[2];
        P.s2u = std::max(1, umax);
        P.s2map = umax <= 256 ? mspan : 0;
        P.s3span = span;
        for (int k = 0; k < S2_KINDS; k++) P.n2[k] = smax[3 + k];
        P.s2w = smax[7];
    }
    // ---- step 2
    TileOperands op = make_operands(A, B);
    TSG_TRY(launch_step2(s, op, B, C, P, w));
    if (timed && numtileC > 0) {
        hipLaunchKernelGGL(k_bins, dim3(std::min<unsigned>(2048, tsg_div_up(numtileC, 256))), dim3(256), 0, s,
                           C->tile_nnz, numtileC, tune.dense_acc_min_nnz, bins);
        TSG_LAUNCH_CHECK();
    }
    // C's tile offsets, then the step-3 row classes (which need only the
    // device offsets); C's nonzero count and the class maxima come back in
    // one read-back
    long long nnzC = 0;
    void *part2v;
    TSG_TRY(tsg_scratch(ctx, (size_t)tsg_scan_partial_count(numtileC) * sizeof(long long), &part2v));
    long long *part2 = (long long *)part2v;
    const bool classes = !P.all && numtileC > 0;
    {
        long long *pin = ctx->pinned;  // [0] the total, then the class words
        tsg_scan_publish pub;
        pub.host = pin;
        TSG_TRY(tsg_scan_i32_enqueue(s, C->tile_nnz, C->tile_nnz, numtileC, part2, pub));
        if (timed) TSG_HIP(hipEventRecord(ev[2], s));
        if (classes && index_later) {
            TSG_TRY(tsg_alloc_t(ctx, &T.longest, (size_t)B->tilem));
            hipLaunchKernelGGL(k_longest_rows, dim3(tsg_div_up(B->tilem, 16)), dim3(256), 0, s, (const int *)B->tile_ptr,
                               (const unsigned short *)B->mask, B->tilem, T.longest);
            TSG_LAUNCH_CHECK();
        }
        const volatile int *h = reinterpret_cast<const int *>(pin + 1);
        auto classify = [&](const int *longest, int *cls_ticket) -> int {
            TSG_TRY(launch_row_class(s, op, C, w.rowcls, w.cls_part, w.cls_out, P.elem_all, longest, cls_ticket, (int *)(pin + 1)));
            TSG_HIP(hipStreamSynchronize(s));
            return TSG_OK;
        };
        if (classes) TSG_TRY(classify(T.longest, ticket));
        else TSG_HIP(hipStreamSynchronize(s));
        nnzC = *(volatile long long *)pin;
        if (nnzC > 0x7fffffffLL) {
            tsg_set_error("prefix sum total %lld exceeds int32", nnzC);
            return TSG_ERR_OVERFLOW;
        }
        if (classes && index_later && h[10] > 0) {  // some tile-rows would go by row lines
            int cls[CLS_WORDS];
            for (int i = 0; i < CLS_WORDS; i++) cls[i] = h[i];
            const double pairs = (double)A->numtile * B->numtile / std::max(1, B->tilen);
            const bool few = 2LL * cls[11] <= C->tilem && cls[12] <= AUTO_SEGMENTS && pairs >= AUTO_PAIRS * numtileC;
            if (few || 8LL * cls[11] <= C->tilem) TSG_TRY(index_operands());
            if (A->rowx_ptr && B->rowx_ptr) {
                op = make_operands(A, B);
                P.s3_elem = few;
                for (int i = 0; i < CLS_WORDS; i++) ((int *)(pin + 1))[i] = cls[i];  // (making the index read back there)
            } else {
                TSG_TRY(classify(nullptr, nullptr));
            }
        }
        if (classes) {
            P.s3_unfit = h[0] > 0;
            P.s3_rows = h[1] > 0;
            for (int i = 0; i < 6; i++) P.g3[i] = std::max(1, (int)h[1 + i]);
            P.s3_lines = h[10] > 0;
            P.ln[0] = h[7];
            P.ln[1] = h[8];
            for (P.ln[2] = LN_MAP_MIN; P.ln[2] < std::min((int)h[9], LN_MAP);) P.ln[2] *= 2;
            P.ln[3] = std::min(LN_THREADS, 16 * (8 << h[10]));
        }
    }
    P.nnzC = nnzC;
    C->nnz = (int)nnzC;
    // ---- step 3
    if (!symbolic) {
        TSG_TRY(tsg_alloc_t(ctx, &C->csr_col, (size_t)nnzC + 1));
        TSG_TRY(tsg_alloc_t(ctx, &C->val, (size_t)nnzC + 1));
    }
    if (nnzC > 0) {
        if (!P.all && P.s3_unfit && P.s3_elem) {
            const SpgemmWork w3 = work_at(wbuf, C->tilem, numtileC, nnzC, nullptr);
            TSG_TRY(tsg_alloc(ctx, &T.w3buf, 16 * (size_t)w3.seg3_cap));
            w.seg3 = (int4 *)T.w3buf;
            w.seg3_cap = w3.seg3_cap;
            if (op.Arowp && !tune.no_heavy_rows) {
                // rows with very many products: one wave each (k_step3_heavy)
                const int m = C->m;
                TSG_TRY(tsg_alloc_t(ctx, &T.hflag, (size_t)m + 16));
                TSG_TRY(tsg_alloc_t(ctx, &T.hcnt, 2 * (size_t)m + 1));
                TSG_TRY(tsg_alloc_t(ctx, &T.hinfo, 8));
                TSG_HIP(hipMemsetAsync(T.hinfo, 0, 32, s));
                const long long counted = tune.heavy_min_products > 0 ? tune.heavy_min_products : HEAVY_MIN_PRODUCTS;
                const bool large = nnzC >= LONG_MIN_NNZ;
                const long long split = tune.heavy_min_products > 0 || !large
                                            ? counted
                                            : std::min(nnzC >> HEAVY_SPLIT_LOG, HEAVY_SPLIT_MAX);
                hipLaunchKernelGGL(k_heavy_flags, tsg_grid(C->tilem, 256), dim3(256), 0, s, op.Arowp, op.Acolx,
                                   (const int *)B->rowx_ptr, w.rowcls, C->tile_ptr, C->tile_colidx, C->tile_nnz, C->tilem, m, split,
                                   counted,
                                   large || tune.heavy_min_products > 0 ? 1 : 0, T.hflag, T.hcnt, T.hinfo);
                TSG_LAUNCH_CHECK();
                long long nh = 0;
                TSG_TRY(tsg_scan_i32(ctx, T.hcnt, T.hcnt, 2LL * m, &nh, T.hinfo, 8));
                const volatile int *info = (const volatile int *)(ctx->pinned + 1);
                const int nheavy = info[0];
                w.ncounted = info[1];
                const long long done = (unsigned)info[2], ntl = info[3];
                const long long groups = (unsigned)info[4] | (long long)info[5] << 32;
                const long long parts = (unsigned)info[6] | (long long)info[7] << 32;
                w.seg3_cap = C->tilem + (nnzC - done) / (G3E_NNZ - 255) + 2;  // blocks: those past the segments only end
                if (nh > 0) {
                    TSG_TRY(tsg_alloc_t(ctx, &T.hrows, (size_t)nh));
                    hipLaunchKernelGGL(k_heavy_list, dim3(tsg_div_up(m, 256)), dim3(256), 0, s, (const int *)T.hcnt,
                                       (const unsigned char *)T.hflag, m, C->tile_ptr, C->tile_colidx, T.hrows);
                    TSG_LAUNCH_CHECK();
                    // the narrowest windows whose table is small enough; one window is B's row pointers
                    int shift = HEAVY_PART_LOG;
                    long long nw = ((long long)B->n + (1 << shift) - 1) >> shift;
                    while (nw > 1 && (nw + 1 > HEAVY_WINDOWS_MAX || 4 * (nw + 1) * B->m > HEAVY_WINDOW_BYTES)) {
                        shift++;
                        nw = (nw + 1) >> 1;
                    }
                    while (nw > 1 && !symbolic) {  // wider ones where that much is not to be had
                        const int st = tsg_alloc(ctx, (void **)&T.hwin, (size_t)(4 * (nw + 1) * B->m));
                        if (st == TSG_OK) break;
                        if (st != TSG_ERR_NOMEM) return st;
                        shift++;
                        nw = (nw + 1) >> 1;
                    }
                    w.hflag = T.hflag;
                    w.hrows = T.hrows;
                    w.nheavy = nheavy;
                    w.nlong = (int)nh - nheavy;
                    // twice the mean; a row with more takes several a block
                    const long long most = ((long long)B->n + HEAVY_PART_COLS - 1) / HEAVY_PART_COLS;
                    w.hstep = (int)std::min(most, 2 * (parts / std::max(nheavy, 1) + 1));
                    w.lstep = (int)std::min((most + HEAVY_GROUP - 1) / HEAVY_GROUP, 2 * (groups / std::max(ntl, 1LL) + 1));
                    w.lchunk = w.lstep * HEAVY_GROUP >= most ? heavy_padded(w.nlong) : LONG_CHUNK;
                    w.hnw = (int)nw;
                    w.hshift = nw > 1 ? shift : 31;
                    w.hstride = nw > 1 ? B->m : 1;
                    w.hwin_bytes = nw > 1 ? 4 * (nw + 1) * B->m : 0;
                    w.hwin = B->rowx_ptr;
                    if (nw > 1 && !symbolic) {
                        hipLaunchKernelGGL(k_heavy_windows, dim3(tsg_div_up(B->m, 256), (unsigned)nw + 1), dim3(256), 0, s,
                                           (const int *)B->rowx_ptr, (const int *)B->rowx_col, B->m, (int)nw, shift,
                                           T.hwin);
                        TSG_LAUNCH_CHECK();
                        w.hwin = T.hwin;
                    }
                }
            }
        }
        if (!symbolic) TSG_TRY(launch_step3(s, op, B, C, P, w, timed ? ev + 4 : nullptr));
    }
    if (timed) {
        TSG_HIP(hipEventRecord(ev[3], s));
        TSG_HIP(hipEventSynchronize(ev[3]));
        TSG_TRY(ev_ms(ev[0], ev[1], &stats->t_step1_ms));
        TSG_TRY(ev_ms(ev[1], ev[2], &stats->t_step2_ms));
        TSG_TRY(ev_ms(ev[2], ev[3], &stats->t_step3_ms));
        TSG_TRY(ev_ms(ev[0], ev[3], &stats->t_total_ms));
        TSG_TRY(ev_ms(ev[4], ev[5], &stats->t_step3_rows_ms));
        unsigned long long hb[4];
        TSG_HIP(hipMemcpyAsync(hb, bins, sizeof(hb), hipMemcpyDeviceToHost, s));
        TSG_HIP(hipStreamSynchronize(s));
        stats->tiles_empty = (long long)hb[0];
        stats->tiles_sparse_acc = (long long)hb[1];
        stats->tiles_dense_acc = (long long)hb[2];
        stats->numtileC = numtileC;
        stats->nnzC = nnzC;
        stats->heavy_rows = w.ncounted;
        stats->heavy_bytes = w.hwin_bytes + (w.hflag ? 9LL * C->m + 16LL * ((long long)w.nheavy + w.nlong) : 0);
    }
    if (plan_out) *plan_out = P;
    return TSG_OK;
}

int tsg_spgemm_planned(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, const tsg_tune *tune_in,
                       tsg_dtiles *C, tsg_stats *stats, tsg_spgemm_plan *plan_out, bool symbolic, bool may_index) {
    memset(C, 0, sizeof(*C));
    SpgemmTemps T;
    int st = spgemm_run(ctx, A, B, tune_in, C, stats, plan_out, symbolic, may_index, T);
    const bool indexed = T.rowx[0].rowptr || T.rowx[1].rowptr;
    free_temps(ctx, T);
    if (st != TSG_OK) tsg_tiles_free(ctx, C);  // a partly built C goes back too
    if (st == TSG_ERR_NOMEM && indexed) {  // the indices made for this product may be what it lacked
        st = spgemm_run(ctx, A, B, tune_in, C, stats, plan_out, symbolic, false, T);
        free_temps(ctx, T);
        if (st != TSG_OK) tsg_tiles_free(ctx, C);
    }
    return st;
}


extern "C" int tsg_spgemm(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, const tsg_tune *tune_in,
                          tsg_dtiles *C, tsg_stats *stats) {
    return tsg_spgemm_planned(ctx, A, B, tune_in, C, stats, nullptr, false, true);
}

size_t tsg_spgemm_work_bytes(const tsg_dtiles *C, const tsg_dtiles *B, int s1w) {
    size_t off[WORK_NARR];
    const size_t bb = brow_bits_bytes(B);
    return work_layout(C->tilem, C->numtile, C->nnz, off, s1w, bb, bb ? 4 * (size_t)B->tilem : 0);
}

int tsg_spgemm_enqueue(hipStream_t s, const tsg_dtiles *A, const tsg_dtiles *B, tsg_dtiles *C,
                       const tsg_spgemm_plan &P, void *work) {
    const SpgemmWork w = work_at(work, C->tilem, C->numtile, C->nnz, nullptr, P.s1w, brow_bits_bytes(B),
                                 4 * (size_t)B->tilem);
    const int4 *bdesc = nullptr;
    const unsigned *bbits = nullptr;
    if (C->tilem > 0) TSG_TRY(launch_brow_bits(s, B, w.bbits, &bdesc, &bbits, nullptr, nullptr, w.longest));
    TSG_TRY(launch_step1(s, A, B, C, false, P.s1w, w.bmstore, bdesc, bbits, nullptr, nullptr));
    TSG_TRY(tsg_scan_i32_enqueue(s, C->tile_ptr, C->tile_ptr, C->tilem, w.part1));
    TSG_TRY(launch_step1(s, A, B, C, true, P.s1w, w.bmstore, bdesc, bbits, nullptr, w.segctr));
    const TileOperands op = make_operands(A, B);
    TSG_TRY(launch_step2(s, op, B, C, P, w));
    TSG_TRY(tsg_scan_i32_enqueue(s, C->tile_nnz, C->tile_nnz, C->numtile, w.part2));
    if (C->nnz > 0) {
        if (!P.all) TSG_TRY(launch_row_class(s, op, C, w.rowcls, w.cls_part, w.cls_out, P.elem_all, P.lines ? w.longest : nullptr));
        TSG_TRY(launch_step3(s, op, B, C, P, w));
    }
    return TSG_OK;
}

// ------------------------------------------------------------------ chunks
// Row lengths of B from its tile masks: row 16K+r is the popcount of row r
// over the tiles of tile-row K.
__global__ void __launch_bounds__(256)
k_tile_row_lengths(const int *__restrict__ Bptr, const unsigned short *__restrict__ Bmask, int m,
                   int *__restrict__ len) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    const int K = i >> 4, r = i & 15;
    int c = 0;
    for (int t = Bptr[K]; t < Bptr[K + 1]; t++) c += __popc((unsigned)Bmask[(long long)t * 16 + r]);
    len[i] = c;
}

// Intermediate products of every A tile-row: sum over A's nonzeros (i, k)
// of B's row length k.  One wave per tile-row, lanes over its tiles.
__global__ void __launch_bounds__(256)
k_tile_row_products(const int *__restrict__ Aptr, const int *__restrict__ Acol, const unsigned short *__restrict__ Amask,
                    int tilem, const int *__restrict__ blen, int bm, unsigned long long *__restrict__ out) {
    const int I = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (I >= tilem) return;
    unsigned long long s = 0;
    for (int t = Aptr[I] + lane; t < Aptr[I + 1]; t += 64) {
        const int k0 = Acol[t] * 16;
        const uint4 *m4 = reinterpret_cast<const uint4 *>(Amask + (long long)t * 16);
        const uint4 a = m4[0], b = m4[1];
        const unsigned w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        int cc[16];
#pragma unroll
        for (int c = 0; c < 16; c++) cc[c] = 0;
#pragma unroll
        for (int q = 0; q < 8; q++)
#pragma unroll
            for (int c = 0; c < 16; c++) cc[c] += ((w[q] >> (15 - c)) & 1u) + ((w[q] >> (31 - c)) & 1u);
#pragma unroll
        for (int c = 0; c < 16; c++)
            if (cc[c] && k0 + c < bm) s += (unsigned long long)cc[c] * (unsigned long long)blen[k0 + c];
    }
    s = tsg_wave_sum(s);
    if (lane == 0) out[I] = s;
}

int tsg_tile_row_products(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, unsigned long long *d_out) {
    if (A->n != B->m) { tsg_set_error("tile_row_products: inner dimensions differ"); return TSG_ERR_ARG; }
    int *blen;
    TSG_TRY(tsg_alloc_t(ctx, &blen, (size_t)B->m + 1));
    if (B->m > 0) {
        hipLaunchKernelGGL(k_tile_row_lengths, dim3(tsg_div_up(B->m, 256)), dim3(256), 0, ctx->stream, B->tile_ptr,
                           B->mask, B->m, blen);
        TSG_LAUNCH_CHECK();
    }
    if (A->tilem > 0) {
        hipLaunchKernelGGL(k_tile_row_products, dim3(tsg_div_up(A->tilem, 4)), dim3(256), 0, ctx->stream, A->tile_ptr,
                           A->tile_colidx, A->mask, A->tilem, blen, B->m, d_out);
        TSG_LAUNCH_CHECK();
    }
    tsg_free(ctx, blen);
    return TSG_OK;
}

// Tile-row ranges of A whose intermediate products stay within
// max_products each (a single tile-row above it forms its own chunk).
// Every chunk's C then has at most max_products nonzeros.
extern "C" int tsg_spgemm_chunk_plan(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, long long max_products,
                                     int max_chunks, int *bounds, int *nchunks, unsigned long long *products_total) {
    if (!A || !B || !bounds || !nchunks || max_chunks < 1 || max_products < 1) {
        tsg_set_error("tsg_spgemm_chunk_plan: bad arguments");
        return TSG_ERR_ARG;
    }
    unsigned long long *d;
    TSG_TRY(tsg_alloc_t(ctx, &d, (size_t)A->tilem + 1));
    TSG_TRY(tsg_tile_row_products(ctx, A, B, d));
    std::vector<unsigned long long> h((size_t)A->tilem + 1);
    if (A->tilem > 0)
        TSG_HIP(hipMemcpyAsync(h.data(), d, 8 * (size_t)A->tilem, hipMemcpyDeviceToHost, ctx->stream));
    TSG_HIP(hipStreamSynchronize(ctx->stream));
    tsg_free(ctx, d);
    int n = 0;
    bounds[0] = 0;
    unsigned long long acc = 0, tot = 0;
    for (int I = 0; I < A->tilem; I++) {
        tot += h[I];
        if (acc > 0 && acc + h[I] > (unsigned long long)max_products) {
            if (n + 1 >= max_chunks) {
                tsg_set_error("tsg_spgemm_chunk_plan: more than %d chunks needed", max_chunks);
                return TSG_ERR_ARG;
            }
            bounds[++n] = I;
            acc = 0;
        }
        acc += h[I];
    }
    bounds[++n] = A->tilem;
    *nchunks = n;
    if (products_total) *products_total = tot;
    return TSG_OK;
}

// C rows [16*r0, min(16*r1, m)) of A*B: A restricted to tile-rows [r0, r1)
// as a view (tile_ptr offset into A's, every other array shared).
extern "C" int tsg_spgemm_tile_rows(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, int r0, int r1,
                                    const tsg_tune *tune, tsg_dtiles *C, tsg_stats *stats) {
    return tsg_spgemm_tile_rows_ex(ctx, A, B, r0, r1, tune, C, stats, false);
}

int tsg_spgemm_tile_rows_ex(tsg_ctx *ctx, const tsg_dtiles *A, const tsg_dtiles *B, int r0, int r1,
                            const tsg_tune *tune, tsg_dtiles *C, tsg_stats *stats, bool symbolic) {
    if (!A || r0 < 0 || r1 < r0 || r1 > A->tilem) {
        memset(C, 0, sizeof(*C));
        tsg_set_error("tsg_spgemm_tile_rows: bad tile-row range [%d, %d)", r0, r1);
        return TSG_ERR_ARG;
    }
    tsg_dtiles v = *A;
    v.tile_ptr = A->tile_ptr + r0;
    if (A->rowx_ptr) v.rowx_ptr = A->rowx_ptr + 16 * (long long)r0;  // indices stay absolute
    v.tilem = r1 - r0;
    v.m = std::min(16 * r1, A->m) - 16 * r0;
    if (v.m < 0) v.m = 0;
    return tsg_spgemm_planned(ctx, &v, B, tune, C, stats, nullptr, symbolic);
}
