// mlp_fused.hip -- whole passes of the surrogate's MLP (inference, and a training batch) with the
// activations of a block of rows kept in LDS.
//
// No counterpart in the reference (its emulator is a Gaussian process, holodeck/gps/).  The layers are
// at most 256 wide, so a layer by itself is a launch, a read and a write of its activations around a
// product that takes a few microseconds; per row block the whole chain needs only the weights, which
// every block reads from L2.
//
// A workgroup of 8 waves holds 16 MT rows.  Per layer a wave computes output tiles w and w + 8 (of 16
// outputs) for all the rows, its weight fragments loaded straight from global memory into registers a
// layer ahead (a wave's two tiles are the only readers of those weights in the workgroup, so LDS would
// add a pass); the activations are the other operand, from LDS, where a row's 16-byte chunks are
// permuted by the row (chunk ^ (row & 15)) so that the 16 rows of a fragment fall into different banks.
// The weights are the MFMA's A operand: a lane then holds four neighbouring outputs of one row, one
// 8-byte LDS write.  Sums run over k in steps of 32 from zero, then the bias, as k_mlp_gemm's do.
//
// MFMA 16x16x32 operand layout (lane l of 64): A row l%16, k 8*(l/16)..+7; B column l%16, k
// 8*(l/16)..+7; accumulator column l%16, rows 4*(l/16)..+3.
#include "mlp.hpp"
#include "../../include/holohip.h"
#include <algorithm>

namespace hd {

constexpr int FU_THREADS = 512;
constexpr int FU_WAVES = FU_THREADS / 64;
constexpr int FU_WIDTH = 256;                 // units of a hidden layer, at most
constexpr int FU_NK = FU_WIDTH / 32;          // k steps, at most
constexpr int FU_GROUP = 2 * FU_WAVES;        // output tiles of one round of the waves

// element (row m, unit k) of the activations in LDS
__device__ __forceinline__ bf16* fu_at(bf16* act, int m, int k) {
    return act + m * FU_WIDTH + ((((k >> 3) ^ (m & 15)) << 3) | (k & 7));
}

struct FuFrag {
    bf16x8 w[2][FU_NK];
};

// Weight fragments of this wave's tiles t0 and t0 + 8 (rows of W (rows, cols)); rows past the end are
// the last row (their outputs are dropped), k past the end is zero.
__device__ __forceinline__ void fu_load(FuFrag& f, const bf16* __restrict__ W, int rows, int cols, int t0, int lane) {
    const int nk = (cols + 31) >> 5;
    const bool whole = (cols & 31) == 0;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int row = min(16 * (t0 + FU_WAVES * j) + (lane & 15), rows - 1);
        const bf16* p = W + (int64_t)row * cols + 8 * (lane >> 4);
#pragma unroll
        for (int k = 0; k < FU_NK; k++) {
            if (k >= nk) break;
            if (whole) {
                f.w[j][k] = *(const bf16x8*)(p + 32 * k);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    f.w[j][k][e] = (32 * k + 8 * (lane >> 4) + e < cols) ? p[32 * k + e] : (bf16)0.0f;
            }
        }
    }
}

template <int MT>
__device__ __forceinline__ void fu_product(const FuFrag& f, bf16* act, int nk, int lane, f32x4 (&acc)[2][MT]) {
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < FU_NK; k++) {
        if (k >= nk) break;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const bf16x8 a = *(const bf16x8*)fu_at(act, 16 * i + (lane & 15), 32 * k + 8 * (lane >> 4));
#pragma unroll
            for (int j = 0; j < 2; j++)
                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[j][k], a, acc[j][i], 0, 0, 0);
        }
    }
}

struct FuInput {
    const bf16* x;         // (M, in), or
    const double* raw;     // (M, in) with scale = [low, width]
    const double* scale;
};

// An input scaled to the unit box, rounded to FP32 and from there to bf16 (two roundings, as an FP32
// array converted on its own: the register barrier keeps the compiler from merging them).
__device__ __forceinline__ bf16 fu_scaled(double raw, double low, double width) {
    float x = (float)((raw - low) / width);
    asm volatile("" : "+v"(x));
    return (bf16)x;
}
// A target scaled back: product and sum each rounded, as array arithmetic does.
__device__ __forceinline__ double fu_unscaled(float v, double spread, double centre) {
#pragma clang fp contract(off)
    const double p = (double)v * spread;
    return p + centre;
}

// MT: 16-row tiles of the workgroup.  OUT64: doubles y * spread + centre, else FP32.
template <int MT, bool OUT64>
__global__ void __launch_bounds__(FU_THREADS) k_mlp_forward(hd_mlp_net N, FuInput in, int M, float* __restrict__ y,
                                                            double* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) bf16 act[16 * MT * FU_WIDTH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.x * 16 * MT;
    const int nin = N.sizes[0], kin = ((nin + 31) >> 5) << 5;
    FuFrag f;
    fu_load(f, (const bf16*)N.w[0], N.sizes[1], nin, wave, lane);
    for (int e = tid; e < 16 * MT * kin; e += FU_THREADS) {
        const int m = e / kin, k = e - m * kin;
        bf16 v = (bf16)0.0f;
        if (m0 + m < M && k < nin) {
            const int64_t o = (int64_t)(m0 + m) * nin + k;
            v = in.x ? in.x[o] : fu_scaled(in.raw[o], in.scale[k], in.scale[nin + k]);
        }
        *fu_at(act, m, k) = v;
    }
    __syncthreads();
    const int nl = N.n_layers;
    for (int l = 0; l < nl; l++) {
        const int fin = N.sizes[l], fout = N.sizes[l + 1];
        const int nk = (fin + 31) >> 5, tiles = (fout + 15) >> 4;
        const float* bias = N.b[l];
        for (int t0 = wave; t0 - wave < tiles; t0 += FU_GROUP) {   // one round but for a wide output
            if (t0 != wave) fu_load(f, (const bf16*)N.w[l], fout, fin, t0, lane);
            f32x4 acc[2][MT];
            fu_product<MT>(f, act, nk, lane, acc);
            if (l + 1 < nl) {
                fu_load(f, (const bf16*)N.w[l + 1], N.sizes[l + 2], fout, wave, lane);
                __syncthreads();   // every wave has read the activations it now replaces
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int n = 16 * (t0 + FU_WAVES * j) + 4 * (lane >> 4);
                if (t0 + FU_WAVES * j >= tiles) continue;
                float bn[4];
#pragma unroll
                for (int r = 0; r < 4; r++) bn[r] = bias[min(n + r, fout - 1)];
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const int m = 16 * i + (lane & 15);
                    if (l + 1 < nl) {
                        bf16x4 h;
#pragma unroll
                        for (int r = 0; r < 4; r++) h[r] = (bf16)silu(acc[j][i][r] + bn[r]);
                        *(bf16x4*)fu_at(act, m, n) = h;
                    } else if (m0 + m < M) {
                        const int64_t o = (int64_t)(m0 + m) * fout + n;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            if (n + r >= fout) break;
                            const float v = acc[j][i][r] + bn[r];
                            if (OUT64) {
                                const double* s = in.scale + 2 * nin + n + r;
                                out[o + r] = fu_unscaled(v, s[0], s[fout]);
                            } else {
                                y[o + r] = v;
                            }
                        }
                    }
                }
            }
        }
        if (l + 1 < nl) __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// training
// ---------------------------------------------------------------------------
// Workspace of a batch: the hidden activations h[l] (input of layer l), the output gradients dz[l] of
// every layer, the pre-activations in the order k_mlp_rows' threads hold them, and the transposed
// weights wt[l] (in, out padded to 32) of the layers after the first.
struct FuBatch {
    bf16* h[HD_MLP_MAX_LAYERS];
    bf16* dz[HD_MLP_MAX_LAYERS];
    f32x4* z;
    bf16* wt[HD_MLP_MAX_LAYERS];
};

__host__ __device__ __forceinline__ int fu_pad(int n) { return (n + 31) & ~31; }

__global__ void __launch_bounds__(256) k_mlp_transpose(hd_mlp_net N, FuBatch B) {
    const int l = blockIdx.y + 1;
    const int fin = N.sizes[l], fout = N.sizes[l + 1], kp = fu_pad(fout);
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= fin * kp) return;
    const int i = e / kp, o = e - i * kp;
    B.wt[l][e] = (o < fout) ? ((const bf16*)N.w[l])[(int64_t)o * fin + i] : (bf16)0.0f;
}

// Forward, loss and backward of 16 rows: no row needs another one's, so the chain of dz runs on in the
// same workgroup with dz in place of the activations.  A thread's pre-activations of a layer are those
// its own backward epilogue needs, so they pass through global memory (L2) in thread order.
__global__ void __launch_bounds__(FU_THREADS) k_mlp_rows(hd_mlp_net N, FuBatch B, const float* __restrict__ X,
                                                         const float* __restrict__ T, const int64_t* __restrict__ idx,
                                                         int M, float scale, float* __restrict__ loss,
                                                         float* __restrict__ y) {
    __shared__ __attribute__((aligned(16))) bf16 act[16 * FU_WIDTH];
    __shared__ float s_loss[FU_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.x * 16;
    const int m = lane & 15, gm = m0 + m;           // the row this lane's accumulators belong to
    const bool row_on = gm < M;
    const int nl = N.n_layers, nin = N.sizes[0], kin = fu_pad(nin);
    FuFrag f;
    fu_load(f, (const bf16*)N.w[0], N.sizes[1], nin, wave, lane);
    for (int e = tid; e < 16 * kin; e += FU_THREADS) {
        const int r = e / kin, k = e - r * kin;
        bf16 v = (bf16)0.0f;
        if (m0 + r < M && k < nin) {
            v = (bf16)X[(idx ? idx[m0 + r] : (int64_t)(m0 + r)) * nin + k];
            B.h[0][(int64_t)(m0 + r) * nin + k] = v;
        }
        *fu_at(act, r, k) = v;
    }
    __syncthreads();
    const int64_t trow = row_on ? (idx ? idx[gm] : (int64_t)gm) : 0;
    f32x4 acc[2][1];
    for (int l = 0; l < nl - 1; l++) {
        const int fin = N.sizes[l], fout = N.sizes[l + 1];
        fu_product<1>(f, act, (fin + 31) >> 5, lane, acc);
        fu_load(f, (const bf16*)N.w[l + 1], N.sizes[l + 2], fout, wave, lane);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = 16 * (wave + FU_WAVES * j) + 4 * (lane >> 4);
            if (n >= fout) continue;
            f32x4 z;
            bf16x4 h;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                z[r] = acc[j][0][r] + N.b[l][n + r];
                h[r] = (bf16)silu(z[r]);
            }
            B.z[(((int64_t)l * gridDim.x + blockIdx.x) * 2 + j) * FU_THREADS + tid] = z;
            *(bf16x4*)fu_at(act, m, n) = h;
            if (row_on) *(bf16x4*)(B.h[l + 1] + (int64_t)gm * fout + n) = h;
        }
        __syncthreads();
    }
    // output layer: error, its gradient (rounded to bf16) in place of the activations
    {
        const int l = nl - 1, fin = N.sizes[l], fout = N.sizes[l + 1], kp = fu_pad(fout);
        fu_product<1>(f, act, (fin + 31) >> 5, lane, acc);
        if (l > 0) fu_load(f, B.wt[l], fin, kp, wave, lane);
        __syncthreads();
        float e = 0.0f;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = 16 * (wave + FU_WAVES * j) + 4 * (lane >> 4);
            if (n >= kp) continue;
            bf16x4 d;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                d[r] = (bf16)0.0f;
                if (!row_on || n + r >= fout) continue;
                const float v = acc[j][0][r] + N.b[l][n + r];
                if (y) y[(int64_t)gm * fout + n + r] = v;
                const float diff = v - T[trow * fout + n + r];
                d[r] = (bf16)(2.0f * diff * scale);
                B.dz[l][(int64_t)gm * fout + n + r] = d[r];
                e += diff * diff;
            }
            *(bf16x4*)fu_at(act, m, n) = d;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) e += __shfl_down(e, o, 64);
        if (lane == 0) s_loss[wave] = e;
        __syncthreads();
        if (tid == 0) {
            float s = 0.0f;
            for (int w = 0; w < FU_WAVES; w++) s += s_loss[w];
            atomicAdd(loss, s * scale);
        }
    }
    for (int l = nl - 1; l > 0; l--) {   // dz of layer l -> dz of layer l - 1
        const int fin = N.sizes[l], kp = fu_pad(N.sizes[l + 1]);
        f32x4 z[2];
#pragma unroll
        for (int j = 0; j < 2; j++)
            z[j] = B.z[(((int64_t)(l - 1) * gridDim.x + blockIdx.x) * 2 + j) * FU_THREADS + tid];
        fu_product<1>(f, act, kp >> 5, lane, acc);
        if (l > 1) fu_load(f, B.wt[l - 1], N.sizes[l - 1], fin, wave, lane);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = 16 * (wave + FU_WAVES * j) + 4 * (lane >> 4);
            if (n >= fin) continue;
            bf16x4 d;
#pragma unroll
            for (int r = 0; r < 4; r++) d[r] = row_on ? (bf16)(acc[j][0][r] * silu_grad(z[j][r])) : (bf16)0.0f;
            *(bf16x4*)fu_at(act, m, n) = d;
            if (row_on) *(bf16x4*)(B.dz[l - 1] + (int64_t)gm * fin + n) = d;
        }
        __syncthreads();
    }
}

// Eight neighbours of row m of a (M, ld) matrix from column c on (zero past its edges).
__device__ __forceinline__ bf16x8 fu_row8(const bf16* __restrict__ a, int M, int ld, int m, int c) {
    const bf16* p = a + (int64_t)m * ld + c;
    bf16x8 v;
    if (m < M && (ld & 7) == 0 && c + 8 <= ld) return *(const bf16x8*)p;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (m < M && c + e < ld) ? p[e] : (bf16)0.0f;
    return v;
}

struct FuAdam {
    float lr, b1, b2, eps, c1, c2;
};

// Gradient g of weight or bias e of layer l: stored, and taken as an Adam step (Kingma & Ba 2015).
__device__ __forceinline__ void fu_update(const hd_mlp_net& N, const FuBatch& B, const hd_mlp_params& P,
                                          const FuAdam& a, int l, bool is_b, int e, float g) {
    if (P.dw[0]) (is_b ? P.db[l] : P.dw[l])[e] = g;
    if (!P.w[0]) return;
    float* w = is_b ? P.b[l] : P.w[l];
    float* m = is_b ? P.mb[l] : P.mw[l];
    float* v = is_b ? P.vb[l] : P.vw[l];
    const float mi = a.b1 * m[e] + (1.0f - a.b1) * g;
    const float vi = a.b2 * v[e] + (1.0f - a.b2) * g * g;
    m[e] = mi;
    v[e] = vi;
    const float wi = w[e] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
    w[e] = wi;
    if (is_b) return;
    ((bf16*)P.wb[l])[e] = (bf16)wi;
    if (l > 0) {
        const int fin = N.sizes[l];
        const int o = e / fin, i = e - o * fin;
        B.wt[l][(int64_t)i * fu_pad(N.sizes[l + 1]) + o] = (bf16)wi;
    }
}

// Weight and bias gradients of every layer, and the Adam step, in one launch: dW[o, i] = sum_m dz[m, o]
// h[m, i], the sum in steps of 32 rows from the first (the order of k_mlp_gemm).  A workgroup has one 32 x 32
// tile, a wave 16 x 16 of it: small tiles, because the chain over the batch is serial (32 steps at 1024
// rows) and there are only 222 k weights to spread.  Both operands run along their rows, so a slab of 128 rows
// of each is turned in LDS, the next one's loads in flight meanwhile.  The blocks after the tiles'
// sum biases: 32 columns each, in row order.
constexpr int FU_TILE = 32;
constexpr int FU_SLAB = 128;
__host__ __device__ __forceinline__ int fu_tiles(int n) { return (n + FU_TILE - 1) / FU_TILE; }

__global__ void __launch_bounds__(256) k_mlp_wgrad(hd_mlp_net N, FuBatch B, hd_mlp_params P, FuAdam adam, int M,
                                                   int wtiles) {
    constexpr int KP = FU_SLAB + 8;   // padded LDS row: 16-byte alignment kept
    __shared__ __attribute__((aligned(16))) bf16 As[FU_TILE][KP];
    __shared__ __attribute__((aligned(16))) bf16 Bs[FU_TILE][KP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool bias = (int)blockIdx.x >= wtiles;
    int l = 0, t = bias ? blockIdx.x - wtiles : blockIdx.x;
    for (;; l++) {   // the layer this block belongs to
        const int nt = fu_tiles(N.sizes[l + 1]) * (bias ? 1 : fu_tiles(N.sizes[l]));
        if (t < nt) break;
        t -= nt;
    }
    const int fin = N.sizes[l], fout = N.sizes[l + 1], ti = bias ? 1 : fu_tiles(fin);
    const int o0 = (t / ti) * FU_TILE, i0 = (t % ti) * FU_TILE;
    // a slab: thread tid loads 8 columns of rows tid / 4 and tid / 4 + 64 of each operand
    const int lr = tid >> 2, lc = (tid & 3) * 8;
    bf16x8 va[2], vb[2];
    auto load = [&](int r) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            va[q] = fu_row8(B.dz[l], M, fout, r + 64 * q + lr, o0 + lc);
            if (!bias) vb[q] = fu_row8(B.h[l], M, fin, r + 64 * q + lr, i0 + lc);
        }
    };
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.0f;
    const int wm = (wave >> 1) * 16, wn = (wave & 1) * 16;
    load(0);
    for (int r = 0; r < M; r += FU_SLAB) {
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                As[lc + e][lr + 64 * q] = va[q][e];
                if (!bias) Bs[lc + e][lr + 64 * q] = vb[q][e];
            }
        __syncthreads();
        if (r + FU_SLAB < M) load(r + FU_SLAB);
        if (bias) {
            if (tid < FU_TILE) {
#pragma unroll 16
                for (int c = 0; c < FU_SLAB; c++) bsum += (float)As[tid][c];   // zero past the last row
            }
        } else {
            const int fr = lane & 15, fk = (lane >> 4) * 8;
#pragma unroll
            for (int k = 0; k < FU_SLAB; k += 32)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)&As[wm + fr][k + fk],
                                                              *(const bf16x8*)&Bs[wn + fr][k + fk], acc, 0, 0, 0);
        }
        __syncthreads();
    }
    if (bias) {
        if (tid < FU_TILE && o0 + tid < fout) fu_update(N, B, P, adam, l, true, o0 + tid, bsum);
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int o = o0 + wm + 4 * (lane >> 4) + r, c = i0 + wn + (lane & 15);
        if (o < fout && c < fin) fu_update(N, B, P, adam, l, false, o * fin + c, acc[r]);
    }
}

static bool fu_ok(const hd_mlp_net* n) {
    if (!n || n->n_layers < 1 || n->n_layers > HD_MLP_MAX_LAYERS || n->sizes[0] < 1 || n->sizes[0] > FU_WIDTH) return false;
    for (int l = 0; l < n->n_layers; l++) {
        const int fout = n->sizes[l + 1];
        if (fout < 1 || !n->w[l] || !n->b[l]) return false;
        if (((uintptr_t)n->w[l] & 15) != 0) return false;   // 16-byte loads of whole rows of 32
        if (l + 1 < n->n_layers && (fout > FU_WIDTH || (fout & 31) != 0)) return false;
    }
    return true;
}

// Layout of the training workspace at w (w = null: only its size).
static size_t fu_layout(const hd_mlp_net* n, int M, char* w, FuBatch* B) {
    size_t s = 0;
    auto take = [&](size_t bytes) {
        char* p = w ? w + s : nullptr;
        s += (bytes + 255) & ~(size_t)255;
        return p;
    };
    const int nl = n->n_layers;
    const int64_t blocks = cdiv(M, 16);
    for (int l = 0; l < nl; l++) {
        const int fin = n->sizes[l], fout = n->sizes[l + 1];
        B->h[l] = (bf16*)take((size_t)M * fin * 2);
        B->dz[l] = (bf16*)take((size_t)M * fout * 2);
        B->wt[l] = l ? (bf16*)take((size_t)fin * fu_pad(fout) * 2) : nullptr;
    }
    B->z = (f32x4*)take((size_t)std::max(nl - 1, 1) * blocks * 2 * FU_THREADS * sizeof(f32x4));
    return s + 256;
}

template <int MT>
static void forward_launch(const hd_mlp_net& n, const FuInput& in, int M, float* y, double* out, hipStream_t st) {
    const dim3 grid((unsigned)cdiv(M, 16 * MT));
    if (y) hipLaunchKernelGGL((k_mlp_forward<MT, false>), grid, dim3(FU_THREADS), 0, st, n, in, M, y, out);
    else hipLaunchKernelGGL((k_mlp_forward<MT, true>), grid, dim3(FU_THREADS), 0, st, n, in, M, y, out);
}

}  // namespace hd

using namespace hd;

extern "C" int hd_mlp_fused(const hd_mlp_net* net) { return fu_ok(net) ? 1 : 0; }

// Rows per workgroup up to which 16-row blocks are used: as long as they leave at most two workgroups
// per CU, a batch's latency is what counts; beyond, 64 rows share each read of the weights.
constexpr int FU_SMALL_ROWS = 16 * 512;

extern "C" int hd_mlp_forward(const hd_mlp_net* net, const void* x, const double* raw, const double* scale, int M,
                              float* y, double* out, void* stream) {
    if (!fu_ok(net)) return set_error(HD_ERR_ARG, "hd_mlp_forward: network not supported");
    if (M < 1 || (!x && (!raw || !scale)) || (!y && (!out || !scale)))
        return set_error(HD_ERR_ARG, "hd_mlp_forward: bad arguments");
    hipStream_t st = (hipStream_t)stream;
    const FuInput in = {(const bf16*)x, raw, scale};
    KTimer timer("k_mlp_forward", st);
    if (M <= FU_SMALL_ROWS) forward_launch<1>(*net, in, M, y, out, st);
    else forward_launch<4>(*net, in, M, y, out, st);
    return check_launch("k_mlp_forward");
}

extern "C" size_t hd_mlp_train_workspace_size(const hd_mlp_net* net, int M) {
    if (!fu_ok(net) || M < 1) return 0;
    FuBatch B;
    return fu_layout(net, M, nullptr, &B);
}

extern "C" int hd_mlp_train_step(const hd_mlp_net* net, const hd_mlp_params* par, const float* X, const float* T,
                                 const int64_t* idx, int M, float* loss, float* y, int rebuild, float lr, float b1,
                                 float b2, float eps, int step, void* workspace, size_t ws_bytes, void* stream) {
    if (!fu_ok(net) || net->sizes[net->n_layers] > FU_WIDTH)
        return set_error(HD_ERR_ARG, "hd_mlp_train_step: network not supported");
    if (!par || !X || !T || !loss || M < 1 || (par->w[0] && step < 1))
        return set_error(HD_ERR_ARG, "hd_mlp_train_step: bad arguments");
    FuBatch B;
    const size_t need = fu_layout(net, M, nullptr, &B);
    if (!workspace || ws_bytes < need) return set_error(HD_ERR_SIZE, "hd_mlp_train_step: workspace too small");
    fu_layout(net, M, (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255), &B);
    hipStream_t st = (hipStream_t)stream;
    const int nl = net->n_layers;
    if (rebuild && nl > 1) {
        int most = 0;
        for (int l = 1; l < nl; l++) most = std::max(most, net->sizes[l] * fu_pad(net->sizes[l + 1]));
        hipLaunchKernelGGL(k_mlp_transpose, dim3((unsigned)cdiv(most, 256), (unsigned)(nl - 1)), dim3(256), 0, st, *net, B);
        int rc = check_launch("k_mlp_transpose");
        if (rc) return rc;
    }
    const float scale = 1.0f / (float)((int64_t)M * net->sizes[nl]);
    hipLaunchKernelGGL(k_mlp_rows, dim3((unsigned)cdiv(M, 16)), dim3(FU_THREADS), 0, st, *net, B, X, T, idx, M, scale,
                       loss, y);
    int rc = check_launch("k_mlp_rows");
    if (rc) return rc;
    int wtiles = 0, btiles = 0;
    for (int l = 0; l < nl; l++) {
        wtiles += fu_tiles(net->sizes[l + 1]) * fu_tiles(net->sizes[l]);
        btiles += fu_tiles(net->sizes[l + 1]);
    }
    const FuAdam adam = {lr, b1, b2, eps, 1.0f - powf(b1, (float)step), 1.0f - powf(b2, (float)step)};
    hipLaunchKernelGGL(k_mlp_wgrad, dim3((unsigned)(wtiles + btiles)), dim3(256), 0, st, *net, B, *par, adam, M, wtiles);
    return check_launch("k_mlp_wgrad");
}
