// scan.hip -- device exclusive prefix sums (replaces the thrust scan the
// reference calls in src/utils_cuda_scan.h:268-332).
//
// Reduce-then-scan, no inter-block waiting.  The pipeline scans arrays from
// a few hundred counts (where a launch is the cost) to tens of millions:
//   up to 16384 counts       one launch, one block of 1024 threads
//   up to 4096 blocks of     two: each 256-thread block sums a tile of 4096
//     4096 counts            counts (int64 partial), then rescans it from
//                            the sum of the partials before it
//   more                     three: one block scans the partials in between
// The last block leaves the total and, when asked, publishes it (and a few
// words of an earlier kernel's) in pinned host memory, so a read-back is a
// stream wait with no copy behind the scan.  Against four launches (reduce,
// partials, down, total) plus copies, whole products: 5-point 64^2 A^2 169
// -> 108 us, 27d 61x47x53 651 -> 621 us, ER 65521 1.96 -> 1.92 ms.  The
// two-launch form re-reads at most 32 KB of partials per block from L2.
#include "tsg_internal.h"

#define SCAN_THREADS 256
#define SCAN_ITEMS 16
#define SCAN_TILE (SCAN_THREADS * SCAN_ITEMS)

__global__ void __launch_bounds__(SCAN_THREADS)
k_scan_reduce(const int *__restrict__ in, long long n, long long *__restrict__ partial) {
    const long long base = (long long)blockIdx.x * SCAN_TILE;
    long long s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        long long i = base + (long long)j * SCAN_THREADS + threadIdx.x;
        if (i < n) s += in[i];
    }
    s = tsg_wave_sum(s);
    __shared__ long long ws[SCAN_THREADS / 64];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        for (int w = 0; w < SCAN_THREADS / 64; w++) t += ws[w];
        partial[blockIdx.x] = t;
    }
}

// Single block: exclusive scan of nb int64 partials in place; total -> partial[nb].
__global__ void __launch_bounds__(1024)
k_scan_partials(long long *partial, long long nb) {
    __shared__ long long ws[16];
    __shared__ long long carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (long long b0 = 0; b0 < nb; b0 += 1024) {
        long long i = b0 + threadIdx.x;
        long long v = i < nb ? partial[i] : 0;
        long long inc = tsg_wave_incl_scan(v);
        const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
        if (lane == 63) ws[w] = inc;
        __syncthreads();
        long long woff = 0;
        for (int k = 0; k < w; k++) woff += ws[k];
        long long excl = carry + woff + inc - v;
        __syncthreads();
        if (i < nb) partial[i] = excl;
        if (threadIdx.x == 1023) carry = excl + v;
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[nb] = carry;
}

// 16 consecutive counts of a thread from base; a whole, 16-byte aligned run
// moves as four int4 loads and stores (the scalar form strides the lanes 64
// bytes apart and splits every cache line over 16 instructions).
__device__ __forceinline__ bool scan_load16(const int *in, const int *out, long long base, long long n, int v[SCAN_ITEMS]) {
    static_assert(SCAN_ITEMS == 16, "four int4 per thread");
    const bool vec = base + SCAN_ITEMS <= n && !(((uintptr_t)in | (uintptr_t)out) & 15);
    if (vec) {
        const int4 *in4 = reinterpret_cast<const int4 *>(in + base);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int4 t = in4[q];
            v[4 * q] = t.x;
            v[4 * q + 1] = t.y;
            v[4 * q + 2] = t.z;
            v[4 * q + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < SCAN_ITEMS; j++) v[j] = base + j < n ? in[base + j] : 0;
    }
    return vec;
}
__device__ __forceinline__ void scan_store16(bool vec, int *out, long long base, long long n, long long off,
                                             const int v[SCAN_ITEMS]) {
    int o[SCAN_ITEMS];
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        o[j] = (int)off;
        off += v[j];
    }
    if (vec) {
        int4 *out4 = reinterpret_cast<int4 *>(out + base);
#pragma unroll
        for (int q = 0; q < 4; q++) out4[q] = make_int4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
    } else {
#pragma unroll
        for (int j = 0; j < SCAN_ITEMS; j++)
            if (base + j < n) out[base + j] = o[j];
    }
}
// One thread: the total behind the scan, and in the host's memory.
__device__ __forceinline__ void scan_finish(long long total, long long nb, long long *partial, int *out, long long n,
                                            tsg_scan_publish pub) {
    partial[nb] = total;
    out[n] = total > 0x7fffffffLL ? 0x7fffffff : (int)total;
    if (pub.host) {
        pub.host[0] = total;
        for (int i = 0; i < pub.nwords; i++) reinterpret_cast<int *>(pub.host + 1)[i] = pub.words[i];
    }
}

// partial: one per block, scanned (SCANNED) or as k_scan_reduce left them.
template <bool SCANNED>
__global__ void __launch_bounds__(SCAN_THREADS)
k_scan_down(const int *in, long long n, long long *partial, int *out, tsg_scan_publish pub) {
    const long long base = (long long)blockIdx.x * SCAN_TILE + (long long)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    const bool vec = scan_load16(in, out, base, n, v);
    __shared__ long long ws[SCAN_THREADS / 64], wb[SCAN_THREADS / 64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    long long s = 0, before = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) s += v[j];
    if (!SCANNED) {
        for (int b = threadIdx.x; b < (int)blockIdx.x; b += SCAN_THREADS) before += partial[b];
        before = tsg_wave_sum(before);
    }
    const long long inc = tsg_wave_incl_scan(s);
    if (lane == 63) ws[w] = inc;
    if (lane == 0) wb[w] = before;
    __syncthreads();
    if (SCANNED) before = partial[blockIdx.x];
    else {
        before = 0;
        for (int k = 0; k < SCAN_THREADS / 64; k++) before += wb[k];
    }
    long long off = before + inc - s;
    for (int k = 0; k < w; k++) off += ws[k];
    scan_store16(vec, out, base, n, off, v);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_THREADS - 1)
        scan_finish(off + s, gridDim.x, partial, out, n, pub);
}

#define SCAN_ONE_THREADS 1024
#define SCAN_ONE (SCAN_ONE_THREADS * SCAN_ITEMS)
__global__ void __launch_bounds__(SCAN_ONE_THREADS)
k_scan_one(const int *in, long long n, long long nb, long long *partial, int *out, tsg_scan_publish pub) {
    const long long base = (long long)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    const bool vec = scan_load16(in, out, base, n, v);
    __shared__ long long ws[SCAN_ONE_THREADS / 64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    long long s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) s += v[j];
    const long long inc = tsg_wave_incl_scan(s);
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    long long off = inc - s;
    for (int k = 0; k < w; k++) off += ws[k];
    scan_store16(vec, out, base, n, off, v);
    if (threadIdx.x == SCAN_ONE_THREADS - 1) scan_finish(off + s, nb, partial, out, n, pub);
}

long long tsg_scan_partial_count(long long n) {
    return (n <= 0 ? 1 : (n + SCAN_TILE - 1) / SCAN_TILE) + 1;
}

#define SCAN_TWO_BLOCKS 4096
int tsg_scan_i32_enqueue(hipStream_t stream, const int *in, int *out, long long n, long long *partial,
                         tsg_scan_publish pub) {
    if (n < 0) { tsg_set_error("tsg_scan_i32: n < 0"); return TSG_ERR_ARG; }
    const long long nb = tsg_scan_partial_count(n) - 1;
    if (n <= SCAN_ONE) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(SCAN_ONE_THREADS), 0, stream, in, n, nb, partial, out, pub);
        TSG_LAUNCH_CHECK();
        return TSG_OK;
    }
    hipLaunchKernelGGL(k_scan_reduce, dim3((unsigned)nb), dim3(SCAN_THREADS), 0, stream, in, n, partial);
    TSG_LAUNCH_CHECK();
    if (nb <= SCAN_TWO_BLOCKS) {
        hipLaunchKernelGGL(k_scan_down<false>, dim3((unsigned)nb), dim3(SCAN_THREADS), 0, stream, in, n, partial, out,
                           pub);
    } else {
        hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(1024), 0, stream, partial, nb);
        TSG_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_scan_down<true>, dim3((unsigned)nb), dim3(SCAN_THREADS), 0, stream, in, n, partial, out,
                           pub);
    }
    TSG_LAUNCH_CHECK();
    return TSG_OK;
}

int tsg_scan_i32(tsg_ctx *ctx, const int *in, int *out, long long n, long long *total, const int *words, int nwords) {
    if (n < 0) { tsg_set_error("tsg_scan_i32: n < 0"); return TSG_ERR_ARG; }
    void *scr;
    TSG_TRY(tsg_scratch(ctx, (size_t)tsg_scan_partial_count(n) * sizeof(long long), &scr));
    tsg_scan_publish pub;
    if (total) pub = {ctx->pinned, words, nwords};
    TSG_TRY(tsg_scan_i32_enqueue(ctx->stream, in, out, n, (long long *)scr, pub));
    if (total) {
        TSG_HIP(hipStreamSynchronize(ctx->stream));
        *total = *(volatile long long *)ctx->pinned;
        if (*total > 0x7fffffffLL) {
            tsg_set_error("prefix sum total %lld exceeds int32", *total);
            return TSG_ERR_OVERFLOW;
        }
    }
    return TSG_OK;
}

// Plain streaming copy (16 B per lane per iteration): the reference point
// for reading hardware byte counters against a known byte count.
__global__ void __launch_bounds__(256)
k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, long long n16) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n16; i += (long long)gridDim.x * 256)
        dst[i] = src[i];
}

extern "C" int tsg_copy_kernel(tsg_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if ((bytes & 15) || ((uintptr_t)dst & 15) || ((uintptr_t)src & 15)) {
        tsg_set_error("tsg_copy_kernel: 16-byte aligned sizes and pointers only");
        return TSG_ERR_ARG;
    }
    const long long n16 = (long long)(bytes / 16);
    if (n16 > 0) {
        hipLaunchKernelGGL(k_copy16, dim3((unsigned)std::min<long long>((n16 + 255) / 256, 8192)), dim3(256), 0,
                           ctx->stream, (const uint4 *)src, (uint4 *)dst, n16);
        TSG_LAUNCH_CHECK();
    }
    return TSG_OK;
}
