// sort.hip -- stable descending order of bins by an FP64 key.
//
// <- `indices = np.argsort(-h2fdf[..., 0].flatten())` (single_sources.py:89).
// numpy's default argsort is not stable; this order is: key descending, ties by
// ascending bin index (which is also what a stable sort of -key gives).
//
// LSD radix sort over the 64-bit order-preserving image of the key, 8 bits per
// pass.  Up to one tile of keys: one workgroup, every pass in LDS (k_sort_one).  More: each pass takes a
// per-tile digit histogram, an exclusive scan of the counts of each digit over the tiles, and a
// stable scatter in which each of a tile's wavefronts ranks a contiguous part of it in chunks of 64,
// equal digits by ballots.  Passes whose digit is the same for every key are skipped on the
// device (the scatter kernel copies).
//
// What bounds it is the chain of one tile, not its traffic (24 bytes per key and pass): sixteen waves per
// tile rank 256 keys each, loaded together (four waves of 1024, a load at a time: 18-20 us per
// pass at any size), and a wave scans a digit's tile counts from the digit totals that the
// histograms add up (one workgroup for all counts: 18 us at 176 tiles).  720,000 keys 0.36 -> 0.20 ms,
// 120,000 0.22 -> 0.16 ms; 2,688 keys 0.30 (24 launches and their gaps) -> 0.04 ms.
#include "common.hpp"
#include "../../include/holohip.h"

namespace hd {

constexpr int SORT_TILE = 4096;     // keys per tile
constexpr int SORT_WAVES = 16;      // waves per tile: each ranks a contiguous part
constexpr int SORT_PART = SORT_TILE / SORT_WAVES;
constexpr int SORT_CHUNKS = SORT_PART / 64;
constexpr int SORT_RADIX = 256;
constexpr int SORT_PASSES = 8;

__device__ __forceinline__ uint64_t desc_key(double v) {
    if (v == 0.0) v = 0.0;   // -0 -> +0
    uint64_t u = (uint64_t)__double_as_longlong(v);
    u = (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);   // ascending image
    return ~u;   // descending
}

// keys and their indices; the digit totals start from zero (as each pass's scatter leaves them)
__global__ void __launch_bounds__(256) k_sort_init(const double* __restrict__ key, int64_t B, int64_t stride, int64_t col,
                                                   uint64_t* __restrict__ k_out, int64_t* __restrict__ v_out,
                                                   uint32_t* __restrict__ total) {
    if (blockIdx.x == 0) total[threadIdx.x] = 0;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    k_out[i] = desc_key(key[i * stride + col]);
    v_out[i] = i;
}

// digit histogram of one tile (256 threads, LDS atomics), stored digit-major, and its share of the totals
__global__ void __launch_bounds__(256) k_sort_hist(const uint64_t* __restrict__ keys, int64_t B, int shift,
                                                   uint32_t* __restrict__ hist, int ntiles, uint32_t* __restrict__ total) {
    __shared__ uint32_t h[SORT_RADIX];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * SORT_TILE;
    uint64_t k[SORT_TILE / 256];
#pragma unroll
    for (int u = 0; u < SORT_TILE / 256; u++) k[u] = keys[min(base + u * 256 + threadIdx.x, B - 1)];
#pragma unroll
    for (int u = 0; u < SORT_TILE / 256; u++)
        if (base + u * 256 + threadIdx.x < B) atomicAdd(&h[(uint32_t)(k[u] >> shift) & 0xff], 1u);
    __syncthreads();
    const uint32_t c = h[threadIdx.x];
    hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = c;
    if (c) atomicAdd(total + threadIdx.x, c);
}

__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v, int lane) {   // inclusive
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(v, off, 64);
        if (lane >= off) v += o;
    }
    return v;
}

// Exclusive scan of the 256 digit totals held one per thread of the first four waves (the others pass
// 0 and take nothing); s_w: four words of LDS.
__device__ __forceinline__ uint32_t digit_scan(uint32_t t, int tid, uint32_t* s_w) {
    const int lane = tid & 63, w = tid >> 6;
    const uint32_t inc = wave_scan_u32(t, lane);
    if (w < 4 && lane == 63) s_w[w] = inc;
    __syncthreads();
    uint32_t base = inc - t;
    for (int q = 0; q < w && q < 4; q++) base += s_w[q];
    return base;
}

// one wave per digit: its tile counts become offsets, from the totals of the digits before it; a block
// of four waves makes the scan of the totals itself.  Flags whether a single digit holds every key
__global__ void __launch_bounds__(256) k_sort_scan(uint32_t* __restrict__ data, int ntiles, int64_t B,
                                                   const uint32_t* __restrict__ total, int* __restrict__ trivial) {
    __shared__ uint32_t s_base[SORT_RADIX], s_w[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t t = total[tid];
    s_base[tid] = digit_scan(t, tid, s_w);
    const int triv = __syncthreads_or(t == (uint32_t)B);
    if (blockIdx.x == 0 && tid == 0) *trivial = triv;
    const int d = blockIdx.x * 4 + w;
    uint32_t run = s_base[d];
    uint32_t* row = data + (int64_t)d * ntiles;
    for (int i = 0; i < ntiles; i += 64) {
        const uint32_t c = (i + lane < ntiles) ? row[i + lane] : 0u;
        const uint32_t inc = wave_scan_u32(c, lane);
        if (i + lane < ntiles) row[i + lane] = run + inc - c;
        run += __shfl(inc, 63, 64);
    }
}

// Positions of a chunk of 64 keys under the running offsets run[] of one wave, which they advance: ranked
// among equal digits by ballots.  The offsets are read and then advanced in program order (LDS
// operations of a wave complete in order), so no workgroup barrier is taken.
__device__ __forceinline__ uint32_t sort_place(uint32_t d, bool valid, uint32_t* run, uint64_t lt_mask) {
    uint64_t eq = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < 8; bit++) {
        const uint64_t b = __ballot(valid && ((d >> bit) & 1));
        eq &= ((d >> bit) & 1) ? b : ~b;
    }
    const uint32_t rank = (uint32_t)__popcll(eq & lt_mask);
    const uint32_t cnt = (uint32_t)__popcll(eq);
    uint32_t pos = 0;
    if (valid) pos = run[d] + rank;
    asm volatile("" ::: "memory");   // every lane's read of run[] before any advance
    if (valid && rank == cnt - 1) run[d] = pos + 1;
    asm volatile("" ::: "memory");
    return pos;
}

// Stable scatter of one tile by sixteen waves; a wave's digit offsets are the tile's plus the counts of
// the parts before it.
__global__ void __launch_bounds__(64 * SORT_WAVES) k_sort_scatter(const uint64_t* __restrict__ kin,
                                                                  const int64_t* __restrict__ vin,
                                                                  uint64_t* __restrict__ kout,
                                                                  int64_t* __restrict__ vout, int64_t B, int shift,
                                                                  const uint32_t* __restrict__ offs, int ntiles,
                                                                  const int* __restrict__ trivial,
                                                                  uint32_t* __restrict__ total) {
    __shared__ uint32_t s_h[SORT_WAVES][SORT_RADIX];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * SORT_TILE;
    const int64_t end = min(base + SORT_TILE, B);
    if (blockIdx.x == 0 && tid < SORT_RADIX) total[tid] = 0;   // for the next pass's histograms
    if (*trivial) {
        for (int64_t i = base + tid; i < end; i += 64 * SORT_WAVES) {
            kout[i] = kin[i];
            vout[i] = vin[i];
        }
        return;
    }
    const int64_t wb = base + (int64_t)w * SORT_PART + lane;
    uint64_t k[SORT_CHUNKS];
    int64_t v[SORT_CHUNKS];
#pragma unroll
    for (int c = 0; c < SORT_CHUNKS; c++) {   // in flight together (indices clamped)
        const int64_t i = min(wb + c * 64, B - 1);
        k[c] = kin[i];
        v[c] = vin[i];
    }
#pragma unroll
    for (int d = lane; d < SORT_RADIX; d += 64) s_h[w][d] = 0;
    // (a wave's own row: its LDS operations complete in order)
#pragma unroll
    for (int c = 0; c < SORT_CHUNKS; c++)
        if (wb + c * 64 < end) atomicAdd(&s_h[w][(uint32_t)(k[c] >> shift) & 0xff], 1u);
    __syncthreads();
    if (tid < SORT_RADIX) {   // thread d: the offsets of digit d for the parts
        uint32_t run = offs[(int64_t)tid * ntiles + blockIdx.x];
#pragma unroll
        for (int q = 0; q < SORT_WAVES; q++) {
            const uint32_t c = s_h[q][tid];
            s_h[q][tid] = run;
            run += c;
        }
    }
    __syncthreads();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int c = 0; c < SORT_CHUNKS; c++) {
        const bool valid = wb + c * 64 < end;
        const uint32_t pos = sort_place((uint32_t)(k[c] >> shift) & 0xff, valid, s_h[w], lt_mask);
        if (valid) {
            kout[pos] = k[c];
            vout[pos] = v[c];
        }
    }
}

// At most one tile of keys: every pass by one workgroup, keys and indices through LDS.
__global__ void __launch_bounds__(64 * SORT_WAVES) k_sort_one(const double* __restrict__ key, int B, int64_t stride,
                                                              int64_t col, int64_t* __restrict__ order) {
    __shared__ uint64_t s_k[SORT_TILE];
    __shared__ uint16_t s_v[SORT_TILE];
    __shared__ uint32_t s_h[SORT_WAVES][SORT_RADIX], s_w[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wb = w * SORT_PART + lane;
    uint64_t k[SORT_CHUNKS];
    uint32_t v[SORT_CHUNKS];
#pragma unroll
    for (int c = 0; c < SORT_CHUNKS; c++) {
        const int i = wb + c * 64;
        k[c] = desc_key(key[(int64_t)min(i, B - 1) * stride + col]);
        v[c] = (uint32_t)i;
    }
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int shift = 0; shift < 64; shift += 8) {
#pragma unroll
        for (int d = lane; d < SORT_RADIX; d += 64) s_h[w][d] = 0;
#pragma unroll
        for (int c = 0; c < SORT_CHUNKS; c++)
            if (wb + c * 64 < B) atomicAdd(&s_h[w][(uint32_t)(k[c] >> shift) & 0xff], 1u);
        __syncthreads();
        uint32_t t = 0;
        if (tid < SORT_RADIX)
#pragma unroll
            for (int q = 0; q < SORT_WAVES; q++) t += s_h[q][tid];
        if (__syncthreads_or(t == (uint32_t)B)) continue;   // one digit holds every key
        uint32_t run = digit_scan(t, tid, s_w);
        if (tid < SORT_RADIX)
#pragma unroll
            for (int q = 0; q < SORT_WAVES; q++) {
                const uint32_t c = s_h[q][tid];
                s_h[q][tid] = run;
                run += c;
            }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < SORT_CHUNKS; c++) {
            const bool valid = wb + c * 64 < B;
            const uint32_t pos = sort_place((uint32_t)(k[c] >> shift) & 0xff, valid, s_h[w], lt_mask);
            if (valid) {
                s_k[pos] = k[c];
                s_v[pos] = (uint16_t)v[c];
            }
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < SORT_CHUNKS; c++) {
            const int i = wb + c * 64;   // (slots past B are never used)
            k[c] = s_k[i];
            v[c] = s_v[i];
        }
    }
#pragma unroll
    for (int c = 0; c < SORT_CHUNKS; c++)
        if (wb + c * 64 < B) order[wb + c * 64] = (int64_t)v[c];
}

}  // namespace hd

using namespace hd;

extern "C" size_t hd_order_workspace_size(int64_t B) {
    int64_t ntiles = cdiv(B, SORT_TILE);
    size_t s = 0;
    s += 2 * (size_t)B * sizeof(uint64_t);   // keys ping-pong (2nd buffer)
    s += (size_t)B * sizeof(int64_t);        // values ping buffer
    s += (size_t)SORT_RADIX * ntiles * sizeof(uint32_t) + 256;   // counts and alignment
    s += 256;                                // trivial flag + alignment
    return s + SORT_RADIX * sizeof(uint32_t);   // a pass's digit totals
}

extern "C" int hd_order_desc(const double* key, int64_t B, int64_t stride, int64_t col, int64_t* order, void* workspace,
                             size_t ws_bytes, void* stream) {
    if (B < 1 || stride < 1 || col < 0 || col >= stride || !key || !order)
        return set_error(HD_ERR_ARG, "hd_order_desc: bad arguments");
    if (B > 0x7fffffffll) return set_error(HD_ERR_SIZE, "hd_order_desc: B too large");
    if (!workspace || ws_bytes < hd_order_workspace_size(B))
        return set_error(HD_ERR_SIZE, "hd_order_desc: workspace too small (%zu < %zu)", ws_bytes,
                         hd_order_workspace_size(B));
    hipStream_t st = (hipStream_t)stream;
    if (B <= SORT_TILE) {
        hipLaunchKernelGGL(k_sort_one, dim3(1), dim3(64 * SORT_WAVES), 0, st, key, (int)B, stride, col, order);
        return check_launch("k_sort_one");
    }
    int ntiles = (int)cdiv(B, SORT_TILE);
    char* p = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
    uint64_t* k0 = (uint64_t*)p;            p += (size_t)B * 8;
    uint64_t* k1 = (uint64_t*)p;            p += (size_t)B * 8;
    int64_t* v1 = (int64_t*)p;              p += (size_t)B * 8;
    p = (char*)(((uintptr_t)p + 15) & ~(uintptr_t)15);
    uint32_t* hist = (uint32_t*)p;          p += (size_t)SORT_RADIX * ntiles * 4;
    uint32_t* total = (uint32_t*)p;         p += (size_t)SORT_RADIX * 4;
    int* triv = (int*)(((uintptr_t)p + 15) & ~(uintptr_t)15);
    int64_t* v0 = order;   // values ping-pong through the output buffer; 8 passes end in v0

    hipLaunchKernelGGL(k_sort_init, dim3((unsigned)cdiv(B, 256)), dim3(256), 0, st, key, B, stride, col, k0, v0,
                       total);
    int rc = check_launch("k_sort_init");
    if (rc) return rc;
    uint64_t* kin = k0; uint64_t* kout = k1;
    int64_t* vin = v0; int64_t* vout = v1;
    for (int pass = 0; pass < SORT_PASSES; pass++) {
        int shift = pass * 8;
        hipLaunchKernelGGL(k_sort_hist, dim3(ntiles), dim3(256), 0, st, kin, B, shift, hist, ntiles, total);
        hipLaunchKernelGGL(k_sort_scan, dim3(SORT_RADIX / 4), dim3(256), 0, st, hist, ntiles, B, total, triv);
        hipLaunchKernelGGL(k_sort_scatter, dim3(ntiles), dim3(64 * SORT_WAVES), 0, st, kin, vin, kout, vout, B, shift,
                           hist, ntiles, triv, total);
        rc = check_launch("k_sort pass");
        if (rc) return rc;
        uint64_t* tk = kin; kin = kout; kout = tk;
        int64_t* tv = vin; vin = vout; vout = tv;
    }
    // after an even number of passes the result is back in k0 / v0 (= order)
    return HD_OK;
}
