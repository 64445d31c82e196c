// realize.hip -- discrete realizations of the binary population and the
// single-source / background split of h_c^2.
//
// <- holodeck/cyutils.pyx: _loudest_hc_from_sorted (1266-1344),
//    _loudest_hc_and_par_from_sorted_redz (1615-1767), _ss_bg_hc (935-1014),
//    _ss_bg_hc_and_par (1068-1178), _sam_poisson_gwb (862-897).
//
// Per (frequency f, realization r) the reference draws a count n_b for every
// bin b, fills L loud slots from bins in a fixed priority order (with
// multiplicity) and sums n_b*h_b over the rest.  This file takes the counts as
// given -- an injected (B,F,R) array, the exact parity path -- and holds the
// merge shared with the drawn-count kernels of realize_gap.hip:
//   * a thread handles one (frequency, realization) column and one chunk of bins;
//   * it keeps the L best instances of its chunk in registers
//     (priority = order rank for the sorted walk, (h desc, bin asc) for argmax)
//     and the FP64 totals sum(n h), sum(n h p_k);
//   * a merge kernel combines the chunk lists per (f, r); the background is
//     total - sum(selected h), which is exactly the reference's accounting
//     (sum(n h) - max for ss_bg_hc; sum((n - taken) h) for the sorted walk,
//     including its treatment of non-integer Normal draws).
#include <algorithm>
#include <type_traits>
#include "common.hpp"
#include "rng.hpp"
#include "../../include/holohip.h"

namespace hd {

constexpr int LMAX = 16;
constexpr int NPAR_MAX = 8;
constexpr int RZ_THREADS = 256;   // columns (f, r) per workgroup, one per thread
constexpr int RZ_MIN_CHUNK = 64;  // bins per chunk, at least
constexpr int RZ_WAVES = 8192;    // waves the chunk count aims at
constexpr int RZ_MAX_CHUNKS = 512;
constexpr uint64_t KEY_NONE = ~0ull;

struct RealizeArgs {
    const double* counts;    // (B,F,R) injected counts
    const double* h2fdf;     // (B,F)
    const int32_t* rank;     // (B) position in order (SORTED) or null
    const double* par;       // (npar,B,F) or null
    int64_t B;
    int F, R, L, mode, flags, npar, nchunks;
    const int64_t* order;    // (B) bin at each position of the sorted walk (final merge, SORTED)
    // partials.  The sorted walk keeps only 32-bit keys (its order ranks: unique, so no bin
    // tie-break, and the bin is order[rank]) in p_key viewed as uint32_t; argmax keeps 64-bit
    // keys and the bins.
    double* p_total;      // (F, nchunks, R)
    double* p_ptot;       // (npar, F, nchunks, R)
    uint64_t* p_key;      // (F, nchunks, L, R): realization fastest
    int32_t* p_bin;       // (F, nchunks, L, R), argmax only
};

constexpr uint32_t KEY32_NONE = 0xffffffffu;

// ascending image of a double, so that larger h -> smaller key when inverted
__device__ __forceinline__ uint64_t h_priority(double h) {
    uint64_t u = (uint64_t)__double_as_longlong(h);
    u = (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
    return ~u;
}

// Running list of the merges: LM slots (LM = L for the common L = 1, 5, 10; 16 slots holding
// any L <= 16 otherwise).  S32: the sorted walk's 32-bit ranks (unique, no bins); else 64-bit
// keys with the bin as tie-break (argmax).
template <int LM, bool S32>
struct MergeList {
    using Key = typename std::conditional<S32, uint32_t, uint64_t>::type;
    static constexpr Key NONE = S32 ? (Key)KEY32_NONE : (Key)KEY_NONE;
    Key k[LM];
    int32_t b[LM];
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int i = 0; i < LM; i++) {
            k[i] = NONE;
            b[i] = 0x7fffffff;
        }
    }
    __device__ __forceinline__ static bool better(Key ka, int32_t ba, Key kb, int32_t bb) {
        return S32 ? (ka < kb) : ((ka < kb) || (ka == kb && ba < bb));
    }
    // (key, bin) of slot L - 1, the worst one kept
    __device__ __forceinline__ void worst(int L, Key& wk, int32_t& wb) const {
        if (LM != 16) {
            wk = k[LM - 1];
            wb = b[LM - 1];
            return;
        }
        wk = NONE;
        wb = 0x7fffffff;
#pragma unroll
        for (int q = 0; q < LM; q++)
            if (q == L - 1) {
                wk = k[q];
                wb = b[q];
            }
    }
    __device__ __forceinline__ void insert(Key key, int32_t bin) {
#pragma unroll
        for (int i = 0; i < LM; i++) {
            const bool sw = better(key, bin, k[i], b[i]);
            const Key tk = k[i];
            const int32_t tb = b[i];
            k[i] = sw ? key : tk;
            b[i] = sw ? bin : tb;
            key = sw ? tk : key;
            bin = sw ? tb : bin;
        }
    }
};

// Chunk partials of given counts.  A thread owns one column (f, r) of the (B, F R) counts and
// walks its chunk's bins: a wave then reads 512 contiguous bytes per bin, across frequency
// boundaries too, so ragged R wastes no lanes.  RZ_U bins are loaded ahead of their use.  Bound by
// the counts' bytes: the chunks are cut so that the launch has about RZ_WAVES waves whatever R is
// (one frequency per workgroup and chunks of 16384 bins left 160 waves at 120,000 x 20 x 50, every
// load's latency exposed: 9.94 ms there, 98 GB/s; 0.30 ms and 3.3 TB/s now).
// LM, S32: the list as in the merges.  NP = 0: no parameters.
constexpr int RZ_U = 8;
template <int LM, bool S32, int NP>
__global__ void __launch_bounds__(RZ_THREADS) k_realize_chunk(RealizeArgs A, int chunk_bins) {
    using List = MergeList<LM, S32>;
    using Key = typename List::Key;
    const int64_t FR = (int64_t)A.F * A.R;
    const int64_t col = (int64_t)blockIdx.x * RZ_THREADS + threadIdx.x;
    if (col >= FR) return;
    const int chunk = blockIdx.y;
    const int f = (int)(col / A.R), r = (int)(col - (int64_t)f * A.R);
    const int F = A.F, R = A.R;
    const int L = (LM == 16) ? A.L : LM;
    const int64_t b0 = (int64_t)chunk * chunk_bins, b1 = min(b0 + (int64_t)chunk_bins, A.B);
    const bool use_list = (A.mode != HD_SEL_NONE);
    const bool skip_zero_h = S32 && (A.flags & HD_FLAG_SKIP_ZERO_H) != 0;
    List list;
    list.init();
    double total = 0.0;
    double ptot[NP > 0 ? NP : 1];
#pragma unroll
    for (int k = 0; k < (NP > 0 ? NP : 1); k++) ptot[k] = 0.0;
    for (int64_t s = b0; s < b1; s += RZ_U) {
        double nn[RZ_U], hh[RZ_U];
        int32_t rk[RZ_U];
#pragma unroll
        for (int u = 0; u < RZ_U; u++) {   // every load issued first (the last bin again past the end)
            const int64_t b = min(s + u, b1 - 1);
            nn[u] = A.counts[b * FR + col];
            hh[u] = A.h2fdf[b * F + f];
            rk[u] = S32 ? A.rank[b] : 0;
        }
#pragma unroll
        for (int u = 0; u < RZ_U; u++) {
            const int64_t b = s + u;
            const double n = nn[u], h = hh[u];
            // the sorted walk skips counts below one (and, on request, bins without strain)
            bool on = b < b1;
            if (S32) on = on && !(n < 1) && !(skip_zero_h && h == 0);
            else on = on && (n != 0);
            if (!on) continue;
            const double nh = n * h;
            total += nh;
            if (NP > 0) {
#pragma unroll
                for (int k = 0; k < (NP > 0 ? NP : 1); k++)
                    if (k < A.npar) ptot[k] += nh * A.par[((int64_t)k * A.B + b) * F + f];
            }
            if (use_list && n > 0 && (S32 || h > 0)) {   // argmax: strict cur > max >= 0
                const Key key = S32 ? (Key)(uint32_t)rk[u] : (Key)h_priority(h);
                const int32_t bb = (int32_t)b;
                const int ninst = (int)min(ceil(n), (double)L);   // the same (key, bin) for every instance
                for (int i = 0; i < ninst; i++) {
                    Key wk;
                    int32_t wb;
                    list.worst(L, wk, wb);
                    if (!List::better(key, bb, wk, wb)) break;
                    list.insert(key, bb);
                }
            }
        }
    }
    const int64_t pr = ((int64_t)f * A.nchunks + chunk) * R + r;
    A.p_total[pr] = total;
    if (NP > 0) {
#pragma unroll
        for (int k = 0; k < (NP > 0 ? NP : 1); k++)
            if (k < A.npar) A.p_ptot[(int64_t)k * F * A.nchunks * R + pr] = ptot[k];
    }
    if (use_list) {
#pragma unroll
        for (int j = 0; j < LM; j++)
            if (j < L) {
                const int64_t o = (((int64_t)f * A.nchunks + chunk) * L + j) * R + r;
                if (S32) {
                    ((uint32_t*)A.p_key)[o] = (uint32_t)list.k[j];
                } else {
                    A.p_key[o] = (uint64_t)list.k[j];
                    A.p_bin[o] = list.b[j];
                }
            }
    }
}

// Merge of chunk partials [c0, c1) of (f, r) into a running list, total and parameter totals.
template <int LM, bool S32>
__device__ __forceinline__ void merge_chunks(const RealizeArgs& A, int f, int r, int c0, int c1,
                                             MergeList<LM, S32>& list, double& total, double (&ptot)[NPAR_MAX]) {
    using Key = typename MergeList<LM, S32>::Key;
    const int F = A.F, R = A.R, NC = A.nchunks;
    const int L = (LM == 16) ? A.L : LM;
    const bool use_list = (A.mode != HD_SEL_NONE);
    for (int c = c0; c < c1; c++) {
        int64_t pr = ((int64_t)f * NC + c) * R + r;
        total += A.p_total[pr];
        for (int k = 0; k < A.npar; k++) ptot[k] += A.p_ptot[(int64_t)k * F * NC * R + pr];
        if (use_list) {
            // the chunk's whole list first: every load issued before any is used (indices clamped
            // to slot L-1, no branch), so a chunk costs one load latency instead of one per slot
            const int64_t o0 = ((int64_t)f * NC + c) * L * (int64_t)R + r;
            Key ck[LM];
            int32_t cb[LM];
#pragma unroll
            for (int j = 0; j < LM; j++) {
                const int64_t o = o0 + (int64_t)min(j, L - 1) * R;
                if (S32) {
                    ck[j] = (Key)((const uint32_t*)A.p_key)[o];
                    cb[j] = 0;   // ranks are unique: no tie-break
                } else {
                    ck[j] = (Key)A.p_key[o];
                    cb[j] = A.p_bin[o];
                }
            }
#pragma unroll
            for (int j = 0; j < LM; j++) {
                if (j >= L || ck[j] == MergeList<LM, S32>::NONE) break;
                Key wk;
                int32_t wb;
                list.worst(L, wk, wb);
                if (!MergeList<LM, S32>::better(ck[j], cb[j], wk, wb)) break;
                list.insert(ck[j], cb[j]);
            }
        }
    }
}

// Groups of the first merge stage, of NC chunks: none for few chunks, 8 where (f, group, r) already
// fills the GPU, else about sqrt(NC), the fewest serial steps over both stages.
int realize_merge_groups(int F, int R, int NC) {
    if (NC <= 16) return 0;
    if ((int64_t)F * R * 8 >= 65536) return 8;
    int g = 8;
    while (g < 32 && g * g < NC) g++;
    return g;
}

// First merge stage: thread per (f, group, r) merges the group's chunks and writes a partial of
// the same layout with G "chunks", so that the final merge reads G partials instead of NC (the
// final merge alone has one thread per (f, r): too few waves to hide its load latency).
template <int LM, bool S32>
__global__ void __launch_bounds__(256) k_realize_group(RealizeArgs A, int G, double* __restrict__ q_total,
                                                       double* __restrict__ q_ptot, uint64_t* __restrict__ q_key,
                                                       int32_t* __restrict__ q_bin) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int F = A.F, R = A.R, NC = A.nchunks;
    const int L = (LM == 16) ? A.L : LM;
    if (t >= (int64_t)F * G * R) return;
    const int r = (int)(t % R), g = (int)((t / R) % G), f = (int)(t / ((int64_t)G * R));
    const int CG = (NC + G - 1) / G;
    const int c0 = min(g * CG, NC), c1 = min(c0 + CG, NC);
    MergeList<LM, S32> list;
    list.init();
    double total = 0.0;
    double ptot[NPAR_MAX];
#pragma unroll
    for (int k = 0; k < NPAR_MAX; k++) ptot[k] = 0.0;
    merge_chunks<LM, S32>(A, f, r, c0, c1, list, total, ptot);
    const int64_t pr = ((int64_t)f * G + g) * R + r;
    q_total[pr] = total;
    for (int k = 0; k < A.npar; k++) q_ptot[(int64_t)k * F * G * R + pr] = ptot[k];
    if (A.mode != HD_SEL_NONE) {
#pragma unroll
        for (int j = 0; j < LM; j++)
            if (j < L) {
                const int64_t o = (((int64_t)f * G + g) * L + j) * R + r;
                if (S32) {
                    ((uint32_t*)q_key)[o] = (uint32_t)list.k[j];
                } else {
                    q_key[o] = (uint64_t)list.k[j];
                    q_bin[o] = list.b[j];
                }
            }
    }
}

template <int LM, bool S32>
__global__ void __launch_bounds__(256) k_realize_merge(RealizeArgs A, double* __restrict__ hc2ss,
                                                       int64_t* __restrict__ ssidx, double* __restrict__ hc2bg,
                                                       double* __restrict__ bgpar) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int F = A.F, R = A.R, NC = A.nchunks;
    const int L = (LM == 16) ? A.L : LM;
    if (t >= (int64_t)F * R) return;
    const int f = (int)(t / R), r = (int)(t % R);
    const bool use_list = (A.mode != HD_SEL_NONE);
    MergeList<LM, S32> list;
    list.init();
    double total = 0.0;
    double ptot[NPAR_MAX];
#pragma unroll
    for (int k = 0; k < NPAR_MAX; k++) ptot[k] = 0.0;
    merge_chunks<LM, S32>(A, f, r, 0, NC, list, total, ptot);
    double sel = 0.0;
    double psel[NPAR_MAX];
#pragma unroll
    for (int k = 0; k < NPAR_MAX; k++) psel[k] = 0.0;
    if (use_list) {
#pragma unroll
        for (int j = 0; j < LM; j++) {
            if (j >= L) continue;
            int64_t o = ((int64_t)f * R + r) * L + j;
            if (list.k[j] == MergeList<LM, S32>::NONE) {
                hc2ss[o] = 0.0;
                ssidx[o] = -1;
            } else {
                const int64_t b = S32 ? A.order[list.k[j]] : (int64_t)list.b[j];
                double h = A.h2fdf[b * F + f];
                hc2ss[o] = h;
                ssidx[o] = b;
                sel += h;
                for (int k = 0; k < A.npar; k++) psel[k] += h * A.par[((int64_t)k * A.B + b) * F + f];
            }
        }
    }
    double bg = total - sel;
    hc2bg[(int64_t)f * R + r] = bg;
    if (bgpar) {
        bool none = use_list && (list.k[0] == MergeList<LM, S32>::NONE) && (A.mode == HD_SEL_ARGMAX);
        for (int k = 0; k < A.npar; k++) {
            double v = none ? __builtin_nan("") : (ptot[k] - psel[k]) / bg;
            bgpar[((int64_t)k * F + f) * R + r] = v;
        }
    }
}

__global__ void k_rank_from_order(const int64_t* __restrict__ order, int64_t B, int32_t* __restrict__ rank) {
    int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= B) return;
    rank[order[p]] = (int32_t)p;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

int realize_merge_groups(int F, int R, int NC);
size_t realize_group_ws(int F, int R, int L, int npar, int G);
int realize_merge_launch(const double* h2fdf, const double* par, const int64_t* order, int64_t B, int F, int R, int L,
                         int mode, int npar, int nchunks, const double* p_total, const double* p_ptot, const uint64_t* p_key,
                         const int32_t* p_bin, double* hc2ss, int64_t* ssidx, double* hc2bg, double* bgpar,
                         void* group_ws, int G, hipStream_t st);

// Bins per chunk of given counts: about RZ_WAVES waves over the columns, at least RZ_MIN_CHUNK
// bins (a chunk's partial costs as much as a few bins) and at most RZ_MAX_CHUNKS chunks (the merge
// walks them).  The workspace query asks before the sizes are checked: empty ones get the least chunk.
static int counts_chunk_bins(int64_t B, int F, int R) {
    if (B < 1 || F < 1 || R < 1) return RZ_MIN_CHUNK;
    const int64_t waves = cdiv((int64_t)F * R, 64);
    int64_t nch = cdiv(RZ_WAVES, waves);
    nch = std::min(nch, std::min((int64_t)RZ_MAX_CHUNKS, cdiv(B, RZ_MIN_CHUNK)));
    return (int)(cdiv(cdiv(B, nch), RZ_U) * RZ_U);
}

template <int LM, bool S32>
static int chunk_launch(const RealizeArgs& A, int bins, hipStream_t st) {
    const dim3 grid((unsigned)cdiv((int64_t)A.F * A.R, RZ_THREADS), (unsigned)A.nchunks);
    if (A.npar == 0)
        hipLaunchKernelGGL((k_realize_chunk<LM, S32, 0>), grid, dim3(RZ_THREADS), 0, st, A, bins);
    else
        hipLaunchKernelGGL((k_realize_chunk<LM, S32, NPAR_MAX>), grid, dim3(RZ_THREADS), 0, st, A, bins);
    return check_launch("k_realize_chunk");
}

static size_t realize_ws(int64_t B, int F, int R, int L, int npar) {
    int64_t nch = cdiv(B, counts_chunk_bins(B, F, R));
    size_t pr = (size_t)F * nch * R;
    size_t s = 0;
    s += align256((size_t)B * 4);               // rank
    s += align256(pr * 8);                      // totals
    s += align256(pr * 8 * (size_t)npar);       // param totals
    s += align256(pr * 8 * (size_t)L);          // keys
    s += align256(pr * 4 * (size_t)L);          // bins
    s += align256(realize_group_ws(F, R, L, npar, realize_merge_groups(F, R, (int)nch)));   // first merge stage
    return s + 256;
}

static int realize_counts_impl(const double* counts, const double* h2fdf, const int64_t* order, int64_t B, int F,
                               int R, int L, int mode, int flags, const double* par, int npar, double* hc2ss,
                               int64_t* ssidx, double* hc2bg, double* bgpar, void* ws, size_t ws_bytes,
                               hipStream_t st) {
    if (B < 1 || F < 1 || R < 1 || L < 0 || !h2fdf || !hc2bg) return set_error(HD_ERR_ARG, "realize: bad sizes/pointers");
    if (B > 0x7fffffffll) return set_error(HD_ERR_SIZE, "realize: B=%lld exceeds 2^31-1", (long long)B);
    if (F > 65535) return set_error(HD_ERR_SIZE, "realize: F=%d > 65535", F);
    if (mode != HD_SEL_SORTED && mode != HD_SEL_ARGMAX && mode != HD_SEL_NONE)
        return set_error(HD_ERR_ARG, "realize: unknown mode %d", mode);
    if (mode == HD_SEL_NONE) L = 0;
    else if (L < 1) return set_error(HD_ERR_ARG, "realize: L must be >= 1 for loud-source modes");
    if (L > LMAX) return set_error(HD_ERR_SIZE, "realize: L=%d > %d", L, LMAX);
    if (npar < 0 || npar > NPAR_MAX || (npar > 0 && !par)) return set_error(HD_ERR_ARG, "realize: npar=%d invalid", npar);
    if (mode == HD_SEL_SORTED && !order) return set_error(HD_ERR_ARG, "realize: sorted mode needs an order");
    if (mode != HD_SEL_NONE && (!hc2ss || !ssidx)) return set_error(HD_ERR_ARG, "realize: hc2ss/ssidx required");
    if (!counts) return set_error(HD_ERR_ARG, "realize: counts required");
    size_t need = realize_ws(B, F, R, L, npar);
    if (!ws || ws_bytes < need) return set_error(HD_ERR_SIZE, "realize: workspace too small (%zu < %zu)", ws_bytes, need);

    RealizeArgs A;
    A.counts = counts;
    A.h2fdf = h2fdf;
    A.par = par;
    A.B = B;
    A.F = F;
    A.R = R;
    A.L = L;
    A.mode = mode;
    A.flags = flags;
    A.npar = npar;
    const int bins = counts_chunk_bins(B, F, R);
    A.nchunks = (int)cdiv(B, bins);
    size_t pr = (size_t)F * A.nchunks * R;
    char* p = (char*)(((uintptr_t)ws + 255) & ~(uintptr_t)255);
    int32_t* rank = (int32_t*)p;  p += align256((size_t)B * 4);
    A.p_total = (double*)p;       p += align256(pr * 8);
    A.p_ptot = (double*)p;        p += align256(pr * 8 * (size_t)npar);
    A.p_key = (uint64_t*)p;       p += align256(pr * 8 * (size_t)L);
    A.p_bin = (int32_t*)p;        p += align256(pr * 4 * (size_t)L);
    void* group_ws = p;
    A.rank = (mode == HD_SEL_SORTED) ? rank : nullptr;
    A.order = order;

    if (mode == HD_SEL_SORTED) {
        hipLaunchKernelGGL(k_rank_from_order, dim3((unsigned)cdiv(B, 256)), dim3(256), 0, st, order, B, rank);
        int rc = check_launch("k_rank_from_order");
        if (rc) return rc;
    }
    int rc;
    if (mode == HD_SEL_SORTED) {
        if (L == 1) rc = chunk_launch<1, true>(A, bins, st);
        else if (L == 5) rc = chunk_launch<5, true>(A, bins, st);
        else if (L == 10) rc = chunk_launch<10, true>(A, bins, st);
        else rc = chunk_launch<16, true>(A, bins, st);
    } else if (mode == HD_SEL_ARGMAX) {
        if (L == 1) rc = chunk_launch<1, false>(A, bins, st);
        else rc = chunk_launch<16, false>(A, bins, st);
    } else {
        rc = chunk_launch<1, false>(A, bins, st);   // no lists
    }
    if (rc) return rc;
    // the same merge as the drawn-count kernels (groups of chunks first when there are many)
    return realize_merge_launch(h2fdf, par, order, B, F, R, L, mode, npar, A.nchunks, A.p_total, A.p_ptot, A.p_key,
                                A.p_bin, hc2ss, ssidx, hc2bg, (npar > 0) ? bgpar : nullptr, group_ws,
                                realize_merge_groups(F, R, A.nchunks), st);
}

// Merge of per-chunk partials, shared with the drawn-count kernel (realize_gap.hip).
size_t realize_group_ws(int F, int R, int L, int npar, int G) {
    return (size_t)F * G * R * (sizeof(double) * (1 + (size_t)npar) + (sizeof(uint64_t) + sizeof(int32_t)) * (size_t)L) +
           4 * 256;
}

// the two merge stages for list capacity LM and key width (S32: the sorted walk's ranks)
template <int LM, bool S32>
static int merge_launch_k(RealizeArgs A, void* group_ws, int G, double* hc2ss, int64_t* ssidx, double* hc2bg, double* bgpar,
                          hipStream_t st) {
    const int F = A.F, R = A.R, L = A.L, npar = A.npar;
    if (G > 0) {
        const size_t n = (size_t)F * G * R;
        char* w = (char*)(((uintptr_t)group_ws + 255) & ~(uintptr_t)255);
        double* q_total = (double*)w;         w += n * sizeof(double);
        double* q_ptot = (double*)w;          w += n * sizeof(double) * (size_t)npar;
        uint64_t* q_key = (uint64_t*)w;       w += n * sizeof(uint64_t) * (size_t)L;
        int32_t* q_bin = (int32_t*)w;
        hipLaunchKernelGGL((k_realize_group<LM, S32>), dim3((unsigned)cdiv((int64_t)n, 256)), dim3(256), 0, st, A, G,
                           q_total, q_ptot, q_key, q_bin);
        int rc = check_launch("k_realize_group");
        if (rc) return rc;
        A.nchunks = G;
        A.p_total = q_total;
        A.p_ptot = q_ptot;
        A.p_key = q_key;
        A.p_bin = q_bin;
    }
    hipLaunchKernelGGL((k_realize_merge<LM, S32>), dim3((unsigned)cdiv((int64_t)F * R, 256)), dim3(256), 0, st, A, hc2ss,
                       ssidx, hc2bg, bgpar);
    return check_launch("k_realize_merge");
}

int realize_merge_launch(const double* h2fdf, const double* par, const int64_t* order, int64_t B, int F, int R, int L,
                         int mode, int npar, int nchunks, const double* p_total, const double* p_ptot, const uint64_t* p_key,
                         const int32_t* p_bin, double* hc2ss, int64_t* ssidx, double* hc2bg, double* bgpar,
                         void* group_ws, int G, hipStream_t st) {
    RealizeArgs A;
    A.counts = nullptr;
    A.h2fdf = h2fdf;
    A.rank = nullptr;
    A.order = order;
    A.par = par;
    A.B = B;
    A.F = F;
    A.R = R;
    A.L = L;
    A.mode = mode;
    A.flags = 0;
    A.npar = npar;
    A.nchunks = nchunks;
    A.p_total = const_cast<double*>(p_total);
    A.p_ptot = const_cast<double*>(p_ptot);
    A.p_key = const_cast<uint64_t*>(p_key);
    A.p_bin = const_cast<int32_t*>(p_bin);
    if (mode == HD_SEL_SORTED) {
        if (L == 1) return merge_launch_k<1, true>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
        if (L == 5) return merge_launch_k<5, true>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
        if (L == 10) return merge_launch_k<10, true>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
        return merge_launch_k<16, true>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
    }
    if (mode == HD_SEL_ARGMAX) {
        if (L == 1) return merge_launch_k<1, false>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
        if (L == 5) return merge_launch_k<5, false>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
        if (L == 10) return merge_launch_k<10, false>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
        return merge_launch_k<16, false>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);
    }
    return merge_launch_k<1, false>(A, group_ws, G, hc2ss, ssidx, hc2bg, bgpar, st);   // no lists
}

int rank_from_order_launch(const int64_t* order, int64_t B, int32_t* rank, hipStream_t st) {
    hipLaunchKernelGGL(k_rank_from_order, dim3((unsigned)cdiv(B, 256)), dim3(256), 0, st, order, B, rank);
    return check_launch("k_rank_from_order");
}

}  // namespace hd

using namespace hd;

extern "C" size_t hd_realize_counts_workspace_size(int64_t B, int F, int R, int L, int npar) {
    return realize_ws(B, F, R, L, npar);
}

extern "C" int hd_realize_counts(const double* counts, const double* h2fdf, const int64_t* order, int64_t B, int F, int R,
                                 int L, int mode, int flags, const double* par, int npar, double* hc2ss,
                                 int64_t* ssidx, double* hc2bg, double* bgpar, void* workspace, size_t ws_bytes,
                                 void* stream) {
    return realize_counts_impl(counts, h2fdf, order, B, F, R, L, mode, flags, par, npar, hc2ss, ssidx, hc2bg, bgpar,
                               workspace, ws_bytes, (hipStream_t)stream);
}

extern "C" void hd_philox4x32_10(const uint32_t* ctr, const uint32_t* key, uint32_t* out) {
    U4 c = {ctr[0], ctr[1], ctr[2], ctr[3]};
    U4 o = philox4x32_10(c, key[0], key[1]);
    out[0] = o.x;
    out[1] = o.y;
    out[2] = o.z;
    out[3] = o.w;
}
