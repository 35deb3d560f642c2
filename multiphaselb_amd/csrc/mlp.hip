// Multilayer perceptron of the learned warm start: tanh hidden layers, linear output,
// mean-squared-error loss, Adam.  Matrix products run on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16): weights and activations enter as BF16, products
// accumulate in FP32; the master parameters, the Adam moments, the biases, the loss
// and the activation derivatives stay FP32.
//
// Every product is C[M][N] = A[M][K] * Bt[N][K]^T with both operands row-major in K,
// so each lane loads its 8 consecutive K values of a row with one 16-byte load.  The
// three products of a layer map onto that form by keeping each operand in the layout
// it needs:
//   forward  Z  = X W        A = X   [B][in]   Bt = W^T [out][in]
//   input    dX = dZ W^T     A = dZ  [B][out]  Bt = W   [in][out]
//   weight   dW = X^T dZ     A = X^T [in][B]   Bt = dZ^T [out][B]
// so the forward epilogue writes each activation as [B][w] and [w][B], the backward
// epilogue writes dZ both ways, and the BF16 weight copies exist in both layouts.
// A training iteration (gather, forward, loss, backward, Adam, BF16 refresh) has no
// host-side state: the minibatch index and the Adam step count come from a device
// counter, so one captured graph is replayed for every iteration.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/mplb.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;         // workgroup tile (4 waves of 32 x 32)
constexpr int kKStep = 32;        // K per MFMA
constexpr int kInPad = 32;        // input width rounded up to the K step

enum Epi : int { E_HIDDEN = 0, E_OUT = 1, E_DX = 2, E_DW = 3 };

struct Gemm {
    const __bf16* A;
    int lda;
    const __bf16* Bt;
    int ldb;
    int M, N, K;
    const float* bias;        // E_HIDDEN, E_OUT
    float* out32;             // a (E_HIDDEN), y (E_OUT), dz (E_DX), dW (E_DW)
    int ld32;
    __bf16* outb;             // [M][N] BF16 copy (E_HIDDEN, E_DX)
    int ldob;
    __bf16* outbt;            // [N][M] BF16 copy (E_HIDDEN, E_DX)
    int ldobt;
    const float* act;         // E_DX: activation of the layer's input level, [M][N]
    int ldact;
    int mvalid;               // E_DW: rows m >= mvalid are input padding (not written)
};

__device__ inline __bf16 bf(float x) { return (__bf16)x; }

// The two-launch path keeps every matrix operand in the order its lanes load it: 16 rows x
// 32 K values are 1 KB in one piece, 16 bytes per lane.  (Rows of K values one after the
// other made each load touch sixteen half cache lines; a workgroup streams all the weights
// through one CU, which is bound by the lines it can have in flight.)
__host__ __device__ inline size_t frag(int row, int k, int K) {
    return ((size_t)(row / 16) * (K / kKStep) + k / kKStep) * 512 + ((k % kKStep) / 8 * 16 + row % 16) * 8 + k % 8;
}

// Wave w of the workgroup computes the 32 x 32 block (m0, n0) as 2 x 2 MFMA tiles of
// 16 x 16; lane l supplies row l % 16 of each A tile and row l % 16 of each Bt tile,
// K values 8 (l / 16) .. 8 (l / 16) + 7 of the current K step, and receives
// C[4 (l / 16) + e][l % 16], e = 0..3, of each tile.
template <int EPI>
__global__ void __launch_bounds__(256) k_gemm(Gemm g) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m0 = blockIdx.y * kTile + (wave >> 1) * 32;
    const int n0 = blockIdx.x * kTile + (wave & 1) * 32;
    if (m0 >= g.M || n0 >= g.N) return;
    const int r = lane & 15, kq = (lane >> 4) * 8;
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16* pa0 = g.A + (size_t)(m0 + r) * g.lda + kq;
    const __bf16* pa1 = pa0 + (size_t)16 * g.lda;
    const __bf16* pb0 = g.Bt + (size_t)(n0 + r) * g.ldb + kq;
    const __bf16* pb1 = pb0 + (size_t)16 * g.ldb;
    for (int k = 0; k < g.K; k += kKStep) {
        const bf16x8 a0 = *(const bf16x8*)(pa0 + k), a1 = *(const bf16x8*)(pa1 + k);
        const bf16x8 b0 = *(const bf16x8*)(pb0 + k), b1 = *(const bf16x8*)(pb1 + k);
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc[1][1], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = n0 + 16 * j + r;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = m0 + 16 * i + (lane >> 4) * 4 + e;
                const float v = acc[i][j][e];
                if (EPI == E_HIDDEN) {
                    const float a = tanhf(v + g.bias[n]);
                    g.out32[(size_t)m * g.ld32 + n] = a;
                    g.outb[(size_t)m * g.ldob + n] = bf(a);
                    g.outbt[(size_t)n * g.ldobt + m] = bf(a);
                } else if (EPI == E_OUT) {
                    g.out32[(size_t)m * g.ld32 + n] = v + g.bias[n];
                } else if (EPI == E_DX) {
                    const float a = g.act[(size_t)m * g.ldact + n];
                    const float dz = v * (1.0f - a * a);
                    g.out32[(size_t)m * g.ld32 + n] = dz;
                    g.outb[(size_t)m * g.ldob + n] = bf(dz);
                    g.outbt[(size_t)n * g.ldobt + m] = bf(dz);
                } else {
                    if (m < g.mvalid) g.out32[(size_t)m * g.ld32 + n] = v;
                }
            }
        }
    }
}

// minibatch rows idx[it * B + b] of X [n][din] / T [n][dout] -> BF16 input in both
// layouts (zero padding columns) and the FP32 targets; it = *counter (or 0 with no idx:
// rows 0..B-1 in order)
__global__ void k_gather(const float* __restrict__ X, const float* __restrict__ T, const int* __restrict__ idx,
                         const int* __restrict__ counter, int B, int din, int dout, __bf16* ab, __bf16* abt,
                         float* tgt) {
    const int b = blockIdx.x;
    const int row = idx ? idx[(size_t)(*counter) * B + b] : b;
    for (int c = threadIdx.x; c < kInPad; c += blockDim.x) {
        const float x = c < din ? X[(size_t)row * din + c] : 0.f;
        ab[(size_t)b * kInPad + c] = bf(x);
        abt[(size_t)c * B + b] = bf(x);
    }
    if (T)
        for (int c = threadIdx.x; c < dout; c += blockDim.x) tgt[(size_t)b * dout + c] = T[(size_t)row * dout + c];
}

// dL/dy of L = sum (y - t)^2 / (B n) and the row sums of squared errors
__global__ void k_loss(const float* __restrict__ y, const float* __restrict__ t, int B, int n, float* dz32,
                       __bf16* dzb, __bf16* dzt, float* rowsum) {
    const int b = blockIdx.x;
    const float scale = 2.0f / ((float)B * (float)n);
    __shared__ float part[256];
    float s = 0.f;
    for (int c = threadIdx.x; c < n; c += blockDim.x) {
        const float d = y[(size_t)b * n + c] - t[(size_t)b * n + c];
        s += d * d;
        const float g = scale * d;
        dz32[(size_t)b * n + c] = g;
        dzb[(size_t)b * n + c] = bf(g);
        dzt[(size_t)c * B + b] = bf(g);
    }
    part[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = 0.f;
        for (unsigned i = 0; i < blockDim.x; i++) r += part[i];
        rowsum[b] = r;
    }
}

__global__ void k_loss_final(const float* __restrict__ rowsum, int B, int n, const int* __restrict__ counter,
                             float* hist, float* last) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double s = 0;
    for (int b = 0; b < B; b++) s += rowsum[b];
    const float L = (float)(s / ((double)B * (double)n));
    *last = L;
    if (hist) hist[*counter] = L;
}

// db[c] = sum over the batch of dz[b][c].  A 256-lane workgroup takes 64 columns: lane
// (c, k) sums rows k, k + 4, k + 8, ... with four independent accumulators (loads in
// flight instead of one dependent chain), and the four slices of a column are added in
// slice order through LDS, so the result does not depend on scheduling.
__global__ void __launch_bounds__(256) k_bias_grad(const float* __restrict__ dz, int B, int n, float* db) {
    __shared__ float part[4][64];
    const int cl = threadIdx.x & 63, k = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + cl;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    if (c < n) {
        int b = k;
        for (; b + 12 < B; b += 16) {
            s0 += dz[(size_t)b * n + c];
            s1 += dz[(size_t)(b + 4) * n + c];
            s2 += dz[(size_t)(b + 8) * n + c];
            s3 += dz[(size_t)(b + 12) * n + c];
        }
        for (; b < B; b += 4) s0 += dz[(size_t)b * n + c];
    }
    part[k][cl] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    if (k == 0 && c < n) db[c] = ((part[0][cl] + part[1][cl]) + part[2][cl]) + part[3][cl];
}

// Adam with bias correction; t = *counter + 1
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t n, float lr, float b1, float b2, float eps,
                       const int* __restrict__ counter) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float t = (float)(*counter + 1);
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / (1.f - powf(b1, t));
    const float vh = vi / (1.f - powf(b2, t));
    p[i] -= lr * mh / (sqrtf(vh) + eps);
}

// BF16 copies of layer weights W [din][dout] (FP32 master): Wb [dinp][dout] and
// Wbt [dout][dinp], zero rows for the input padding
__global__ void k_refresh(const float* __restrict__ W, int din, int dinp, int dout, __bf16* Wb, __bf16* Wbt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= dinp * dout) return;
    const int r = i / dout, c = i - r * dout;
    const __bf16 v = bf(r < din ? W[(size_t)r * dout + c] : 0.f);
    Wb[(size_t)r * dout + c] = v;
    Wbt[(size_t)c * dinp + r] = v;
}

// all layers' copies in one launch (training replays this once per iteration, where a
// launch per layer costs more than the copy): element i belongs to the layer l with
// start[l] <= i < start[l + 1]
constexpr int kRefreshLayers = 8;
struct RefreshAll {
    int L;
    int64_t start[kRefreshLayers + 1];
    const float* W[kRefreshLayers];
    int din[kRefreshLayers], dinp[kRefreshLayers], dout[kRefreshLayers];
    __bf16* Wb[kRefreshLayers];
    __bf16* Wbt[kRefreshLayers];
    int pieces;                        // operands in the two-launch path's order (frag)
};

__global__ void k_refresh_all(RefreshAll a) {
    const int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (g >= a.start[a.L]) return;
    int l = 0;
    while (g >= a.start[l + 1]) l++;
    const int i = (int)(g - a.start[l]), dout = a.dout[l], dinp = a.dinp[l];
    const int r = i / dout, c = i - r * dout;
    const __bf16 v = bf(r < a.din[l] ? a.W[l][(size_t)r * dout + c] : 0.f);
    a.Wb[l][a.pieces ? frag(r, c, dout) : (size_t)r * dout + c] = v;
    a.Wbt[l][a.pieces ? frag(c, r, dinp) : (size_t)c * dinp + r] = v;
}

__global__ void k_advance(int* counter) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *counter += 1;
}

// ---------------------------------------------------------------------------
// The network in two launches.  Every row of a batch goes through the layers on its own,
// so one workgroup takes 16 rows through the whole forward pass, the loss and the backward
// pass to the first layer (k_rows), activations and dL/dz staying in LDS; what couples the
// rows, the weight and bias gradients, follows in one launch over all layers with Adam and
// the refresh of the BF16 weight copies in its epilogue (k_weights).
//
// Bound: latency.  The products of a whole iteration (0.26 GFLOP at batch 256) are a
// fraction of a microsecond of the chip's matrix rate, but a row workgroup streams all the
// weights (0.6 MB of BF16) through one CU, layer after layer.  One launch per product, loss
// term, bias and update cost 21 launches of about 5 us, 131 us per iteration of the
// 9-256-256-256-128 network at batch 256; k_rows and k_weights take 19.1 and 7.1 us.  Each product
// accumulates its K values in ascending steps of 32 in one MFMA chain whatever the tile, so
// results equal the one-launch-per-product kernels' bit for bit.
constexpr int kNetLayers = 8;
constexpr int kRows = 16;              // rows of a workgroup of k_rows
constexpr int kRowThreads = 1024;      // 16 waves: one 16-column tile each of a 256-wide layer
constexpr int kHelpers = 8;            // helper workgroups per XCD (backward pass)
constexpr int kRowPad = 8;             // BF16 elements of padding per LDS row

struct Net {
    int L, B, rows;                    // rows: rows of X that exist (gather without idx)
    int w[kNetLayers + 1], wp[kNetLayers + 1];
    int wmax;                          // widest padded level
    const __bf16* Wb[kNetLayers];      // rows: inputs (frag)
    const __bf16* Wbt[kNetLayers];     // rows: outputs (frag)
    const float* bias[kNetLayers];
    const float* X;
    const float* T;
    const int* idx;
    int* counter;                      // [0] iteration of the next k_rows, [1] of the last one
    float* y;                          // forward only: all rows' outputs
    float* rowsum;
    __bf16* abt[kNetLayers];           // BF16 activations of levels 0..L-1, rows: channels (frag)
    __bf16* dzt[kNetLayers + 1];       // BF16 dL/dz of levels 1..L, rows: channels (frag)
    float* dz32[kNetLayers + 1];       // [B][w]
    // KEEP: the row-major copies mplb_mlp_tensor hands out, of the rows from keep0 on
    int keep0;
    float* ykeep;
    __bf16* ab[kNetLayers];
    float* a32[kNetLayers + 1];
    __bf16* dzb[kNetLayers + 1];
};

// LDS of k_rows in bytes: two operand buffers and, with the backward pass, the FP32
// activations of the hidden levels and the output
size_t rows_lds(int L, const int* w, const int* wp, bool bwd) {
    int wmax = 0, hidden = 0;
    for (int l = 0; l <= L; l++) wmax = wp[l] > wmax ? wp[l] : wmax;
    for (int l = 1; l < L; l++) hidden += w[l];
    return sizeof(__bf16) * 2 * kRows * (wmax + kRowPad) + sizeof(float) * kRows * (bwd ? hidden + w[L] + 1 : 0);
}

// K steps [k0, K) of one 16 x 16 tile, K in ascending steps of 32: a, this lane's row of a
// row-major operand, or (FRAG) its place in the tile's pieces; bt, its place in the other
// operand's pieces
template <bool FRAG>
__device__ inline f32x4 row_tile(const __bf16* a, const __bf16* bt, int k0, int K, f32x4 acc) {
#pragma unroll 8
    for (int k = k0; k < K; k += kKStep)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(a + (FRAG ? k / kKStep * 512 : k)),
                                                      *(const bf16x8*)(bt + k / kKStep * 512), acc, 0, 0, 0);
    return acc;
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// The workgroup meets with its LDS writes done; global loads and stores stay in flight
// (nothing of them is read by another wave).  A fence would wait for the transposed stores
// of the layer and for the next layer's weights.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// BWD: with loss and backward pass; KEEP: also the row-major intermediates.  A wave's first
// tile of a layer takes its weights from registers, loaded while the layer before it was
// finished (they do not depend on the rows).  At batch 256: 33.7 us with the weights loaded
// when a layer began, a fence per layer and the targets read at the loss, 30.7 us with all
// three ahead, 20.5 us with the operands in load order (frag), 19.1 us with the helper
// workgroups.
template <bool BWD, bool KEEP>
__global__ void __launch_bounds__(kRowThreads) k_rows(Net g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    if (BWD && (int)blockIdx.x >= g.B / kRows) {
        // helper workgroup: touches its slice of every layer's weights, in the order of use, so
        // that they are in this XCD's L2 when its row workgroups come to them (the update that
        // wrote them ran on all XCDs)
        const int part = ((int)blockIdx.x - g.B / kRows) / 8;
        unsigned seen = 0;
        for (int i = 0; i < 2 * g.L - 1; i++) {
            const int l = i < g.L ? i : 2 * g.L - 1 - i;
            const uint4* p = (const uint4*)(i < g.L ? g.Wbt[l] : g.Wb[l]);
            const int n = g.wp[l] * g.w[l + 1] / 8;
            for (int e = part * kRowThreads + threadIdx.x; e < n; e += kHelpers * kRowThreads) seen |= p[e].x;
        }
        asm volatile("" ::"v"(seen));
        return;
    }
    const int ld = g.wmax + kRowPad;
    __bf16* buf = (__bf16*)lds;                          // [2][kRows][ld]
    float* act = (float*)(buf + 2 * kRows * ld);         // hidden levels, [kRows][w] each, then [kRows][w_L + 1]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, kq = (lane >> 4) * 8, m0 = (lane >> 4) * 4;
    const int b0 = blockIdx.x * kRows, B = g.B;
    const int k0 = b0 - g.keep0;                         // first kept row (KEEP; below 0: none)
    const bool keep = KEEP && k0 >= 0;
    constexpr int kWaves = kRowThreads / 64, kHeld = 8, kTargets = 4;
    bf16x8 held[kHeld];
    float held_bias = 0.f;
    // weights (and bias) of this wave's first tile of a layer
    auto fetch = [&](const __bf16* bt, const float* bias, int N, int K) __attribute__((always_inline)) {
        if (wave >= N / 16) return;
        const __bf16* p = bt + (size_t)wave * 16 * K + lane * 8;
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i * kKStep < K) held[i] = *(const bf16x8*)(p + i * 512);
        if (bias) held_bias = bias[wave * 16 + r];
    };
    auto first_tile = [&](const __bf16* a, const __bf16* bt, int K) __attribute__((always_inline)) {
        f32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (i * kKStep < K)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(a + i * kKStep), held[i], acc, 0, 0, 0);
        return row_tile<false>(a, bt, kHeld * kKStep, K, acc);
    };
    fetch(g.Wbt[0], g.bias[0], g.w[1], g.wp[0]);
    const int* idx = g.idx ? g.idx + (size_t)g.counter[0] * B : nullptr;
    auto row_of = [&](int m) { return idx ? idx[b0 + m] : b0 + m; };
    const int nout = g.w[g.L];
    for (int e = threadIdx.x; e < kRows * kInPad; e += kRowThreads) {
        const int m = e / kInPad, c = e % kInPad, row = row_of(m);
        const float x = c < g.w[0] && row < g.rows ? g.X[(size_t)row * g.w[0] + c] : 0.f;
        buf[m * ld + c] = bf(x);
        if (BWD) g.abt[0][frag(c, b0 + m, B)] = bf(x);
        if (keep) g.ab[0][(size_t)(k0 + m) * kInPad + c] = bf(x);
    }
    float target[kTargets];
    if constexpr (BWD) {
#pragma unroll
        for (int j = 0; j < kTargets; j++) {
            const int e = threadIdx.x + j * kRowThreads;
            if (e < kRows * nout) target[j] = g.T[(size_t)row_of(e / nout) * nout + e % nout];
        }
    }
    lds_barrier();
    int cur = 0;
    float* level = act;                                  // FP32 activations of level l + 1
    for (int l = 0; l < g.L; l++) {
        const int N = g.w[l + 1], K = g.wp[l];
        const bool last = l == g.L - 1;
        const int stride = last ? N + 1 : N;             // (the output's rows are read by one lane each)
        const __bf16* a = buf + (cur * kRows + r) * ld + kq;
        __bf16* to = buf + (1 - cur) * kRows * ld;
        for (int nt = wave; nt < N / 16; nt += kWaves) {
            const int n = nt * 16 + r;
            const __bf16* bt = g.Wbt[l] + (size_t)nt * 16 * K + lane * 8;
            f32x4 acc{0.f, 0.f, 0.f, 0.f};
            float bias;
            if (nt == wave) {
                acc = first_tile(a, bt, K);
                bias = held_bias;
                if (!last) fetch(g.Wbt[l + 1], g.bias[l + 1], g.w[l + 2], g.wp[l + 1]);
                else if (BWD && l > 0) fetch(g.Wb[l], nullptr, g.wp[l], g.w[l + 1]);
            } else {
                acc = row_tile<false>(a, bt, 0, K, acc);
                bias = g.bias[l][n];
            }
            bf16x4 t;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = m0 + e;
                float v = acc[e] + bias;
                if (!last) {
                    v = tanhf(v);
                    t[e] = bf(v);
                    to[m * ld + n] = t[e];
                    if (keep) g.ab[l + 1][(size_t)(k0 + m) * N + n] = t[e];
                    if (keep) g.a32[l + 1][(size_t)(k0 + m) * N + n] = v;
                } else {
                    if (!BWD && b0 + m < B) g.y[(size_t)(b0 + m) * N + n] = v;
                    if (keep) g.ykeep[(size_t)(k0 + m) * N + n] = v;
                }
                if (BWD) level[m * stride + n] = v;
            }
            if (BWD && !last) *(bf16x4*)(g.abt[l + 1] + frag(n, b0 + m0, B)) = t;
        }
        // a wave without a tile in this layer may have one in the next
        if (wave >= N / 16) {
            if (!last) fetch(g.Wbt[l + 1], g.bias[l + 1], g.w[l + 2], g.wp[l + 1]);
            else if (BWD && l > 0) fetch(g.Wb[l], nullptr, g.wp[l], g.w[l + 1]);
        }
        cur = 1 - cur;
        if (BWD && !last) level += kRows * N;
        lds_barrier();
    }
    if constexpr (BWD) {
        // dL/dy of L = sum (y - t)^2 / (B n); level holds y, then the differences
        const int n = nout;
        const float scale = 2.0f / ((float)B * (float)n);
        __bf16* to = buf + cur * kRows * ld;
        auto loss_at = [&](int e, float t) __attribute__((always_inline)) {
            const int m = e / n, c = e - m * n;
            const float d = level[m * (n + 1) + c] - t;
            const float dz = scale * d;
            level[m * (n + 1) + c] = d;
            to[m * ld + c] = bf(dz);
            g.dz32[g.L][(size_t)(b0 + m) * n + c] = dz;
            if (keep) g.dzb[g.L][(size_t)(k0 + m) * n + c] = bf(dz);
        };
#pragma unroll
        for (int j = 0; j < kTargets; j++) {
            const int e = threadIdx.x + j * kRowThreads;
            if (e < kRows * n) loss_at(e, target[j]);
        }
        for (int e = threadIdx.x + kTargets * kRowThreads; e < kRows * n; e += kRowThreads)
            loss_at(e, g.T[(size_t)row_of(e / n) * n + e % n]);
        lds_barrier();
        for (int e = threadIdx.x; e < kRows * n; e += kRowThreads) {
            const int c = e / kRows, m = e % kRows;
            g.dzt[g.L][frag(c, b0 + m, B)] = to[m * ld + c];
        }
        // row sums of squared errors: 256 partial sums over every 256th column, added in
        // order, by one lane per row of the first wave after the backward pass (in which every
        // wave of a 256-wide layer has a tile to finish)
        const float* diff = level;
        for (int l = g.L - 1; l > 0; l--) {
            const int N = g.wp[l], K = g.w[l + 1];
            level -= kRows * N;
            const __bf16* a = buf + (cur * kRows + r) * ld + kq;
            __bf16* out = buf + (1 - cur) * kRows * ld;
            for (int nt = wave; nt < N / 16; nt += kWaves) {
                const int c = nt * 16 + r;
                const __bf16* bt = g.Wb[l] + (size_t)nt * 16 * K + lane * 8;
                f32x4 acc{0.f, 0.f, 0.f, 0.f};
                if (nt == wave) {
                    acc = first_tile(a, bt, K);
                    if (l > 1) fetch(g.Wb[l - 1], nullptr, g.wp[l - 1], g.w[l]);
                } else {
                    acc = row_tile<false>(a, bt, 0, K, acc);
                }
                bf16x4 t;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int m = m0 + e;
                    const float x = level[m * N + c];
                    const float dz = acc[e] * (1.0f - x * x);
                    t[e] = bf(dz);
                    out[m * ld + c] = t[e];
                    g.dz32[l][(size_t)(b0 + m) * N + c] = dz;
                    if (keep) g.dzb[l][(size_t)(k0 + m) * N + c] = t[e];
                }
                *(bf16x4*)(g.dzt[l] + frag(c, b0 + m0, B)) = t;
            }
            if (wave >= N / 16 && l > 1) fetch(g.Wb[l - 1], nullptr, g.wp[l - 1], g.w[l]);
            cur = 1 - cur;
            lds_barrier();
        }
        if (wave == 0 && lane < kRows) {
            const float* d = diff + lane * (n + 1);
            float sum = 0.f;
            if (n <= 256) {
#pragma unroll 16
                for (int i = 0; i < n; i++) sum += d[i] * d[i];
            } else {
                for (int i = 0; i < 256; i++) {
                    float s = 0.f;
                    for (int c = i; c < n; c += 256) s += d[c] * d[c];
                    sum += s;
                }
            }
            g.rowsum[b0 + lane] = sum;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0 && g.idx) g.counter[1] += 1;
    }
}

// one Adam update of parameter i with gradient gi (bias correction at step t)
struct Adam {
    float *p, *m, *v;
    float lr, b1, b2, eps;
};
__device__ inline float adam_update(const Adam& a, int64_t i, float gi, float t) {
    const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gi;
    const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    const float mh = mi / (1.f - powf(a.b1, t));
    const float vh = vi / (1.f - powf(a.b2, t));
    const float p = a.p[i] - a.lr * mh / (sqrtf(vh) + a.eps);
    a.p[i] = p;
    return p;
}

// Weight and bias gradients of every layer: blocks [0, 1) the loss, then per layer 64-column
// bias blocks, then 32 x 32 weight tiles (four waves of one 16 x 16 tile each).
struct Grads {
    int L, B;
    int w[kNetLayers + 1], wp[kNetLayers + 1];
    int bias0[kNetLayers + 1], tile0[kNetLayers + 1];    // first block of a layer's biases / tiles
    const __bf16* abt[kNetLayers];
    const __bf16* dzt[kNetLayers + 1];
    const float* dz32[kNetLayers + 1];
    __bf16* Wb[kNetLayers];
    __bf16* Wbt[kNetLayers];
    int64_t woff[kNetLayers], boff[kNetLayers];
    float* grad;                       // written when not training
    const float* rowsum;
    int* counter;
    float* hist;
    float* loss;
    Adam adam;
};

template <bool TRAIN>
__global__ void __launch_bounds__(256) k_weights(Grads g) {
    const int blk = blockIdx.x, B = g.B;
    const int it = TRAIN ? g.counter[1] : 0;
    const float t = (float)(it + 1);
    if (blk == 0) {
        __shared__ float rs[1024];
        double s = 0;
        for (int b1 = 0; b1 < B; b1 += 1024) {
            const int n = B - b1 < 1024 ? B - b1 : 1024;
            for (int i = threadIdx.x; i < n; i += 256) rs[i] = g.rowsum[b1 + i];
            __syncthreads();
            if (threadIdx.x == 0) {
#pragma unroll 8
                for (int i = 0; i < n; i++) s += rs[i];
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            const float L = (float)(s / ((double)B * (double)g.w[g.L]));
            *g.loss = L;
            if (g.hist) g.hist[it] = L;
            if (TRAIN) g.counter[0] += 1;
        }
        return;
    }
    if (blk < g.tile0[0]) {
        int l = 0;
        while (blk >= g.bias0[l + 1]) l++;
        // as k_bias_grad
        __shared__ float part[4][64];
        const float* dz = g.dz32[l + 1];
        const int n = g.w[l + 1], cl = threadIdx.x & 63, k = threadIdx.x >> 6;
        const int c = (blk - g.bias0[l]) * 64 + cl;
        float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
        if (c < n) {
            int b = k;
#pragma unroll 4
            for (; b + 12 < B; b += 16) {
                s0 += dz[(size_t)b * n + c];
                s1 += dz[(size_t)(b + 4) * n + c];
                s2 += dz[(size_t)(b + 8) * n + c];
                s3 += dz[(size_t)(b + 12) * n + c];
            }
            for (; b < B; b += 4) s0 += dz[(size_t)b * n + c];
        }
        part[k][cl] = (s0 + s1) + (s2 + s3);
        __syncthreads();
        if (k == 0 && c < n) {
            const float db = ((part[0][cl] + part[1][cl]) + part[2][cl]) + part[3][cl];
            if (TRAIN) adam_update(g.adam, g.boff[l] + c, db, t);
            else g.grad[g.boff[l] + c] = db;
        }
        return;
    }
    int l = 0;
    while (blk >= g.tile0[l + 1]) l++;
    const int dout = g.w[l + 1], dinp = g.wp[l], din = g.w[l];
    const int nt = dout / 32, tile = blk - g.tile0[l];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15;
    const int mt0 = tile / nt * 32 + (wave >> 1) * 16, n = tile % nt * 32 + (wave & 1) * 16 + r;
    const f32x4 acc = row_tile<true>(g.abt[l] + (size_t)mt0 * B + lane * 8, g.dzt[l + 1] + (size_t)(n - r) * B + lane * 8,
                                     0, B, f32x4{0.f, 0.f, 0.f, 0.f});
    const int m0 = mt0 + (lane >> 4) * 4;
    bf16x4 wt;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int m = m0 + e;
        if (TRAIN) {
            float p = 0.f;
            if (m < din) p = adam_update(g.adam, g.woff[l] + (int64_t)m * dout + n, acc[e], t);
            wt[e] = bf(p);
            g.Wb[l][frag(m, n, dout)] = wt[e];
        } else if (m < din) {
            g.grad[g.woff[l] + (int64_t)m * dout + n] = acc[e];
        }
    }
    if (TRAIN) *(bf16x4*)(g.Wbt[l] + frag(n, m0, dinp)) = wt;
}

__global__ void k_set_int(int* p, int v) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}

}  // namespace

struct mplb_mlp {
    std::string err;
    int dev = 0;
    hipStream_t stream = nullptr;
    int L = 0;                                  // layers
    std::vector<int> w;                         // level widths (w[0] = raw input width)
    std::vector<int> wp;                        // padded widths used on the device
    int B = 0;                                  // rows per product
    std::vector<int64_t> woff, boff;            // parameter offsets
    int64_t P = 0;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    std::vector<__bf16*> Wb, Wbt;               // per layer
    std::vector<__bf16*> ab, abt;               // per level 0..L-1
    std::vector<float*> a32;                    // per level 1..L-1 (index by level)
    float* y = nullptr;                         // [B][w[L]]
    float* tgt = nullptr;
    std::vector<float*> dz32;                   // per level 1..L
    std::vector<__bf16*> dzb, dzt;
    float* rowsum = nullptr;
    float* loss = nullptr;
    int* counter = nullptr;                     // [2]
    size_t lds_fwd = 0, lds_bwd = 0;            // LDS of k_rows; 0: one launch per product
    float* Y = nullptr;                         // outputs of a forward call
    size_t Y_cap = 0;
    std::vector<void*> owned;
    // training data resident on the device
    float *X = nullptr, *T = nullptr;
    int* idx = nullptr;
    size_t X_cap = 0, T_cap = 0, idx_cap = 0;
    float* hist = nullptr;
    size_t hist_cap = 0;
};

namespace {

int mfail(mplb_mlp* n, int code, const std::string& m) {
    if (n) n->err = m;
    return code;
}

#define MCHK(n, call)                                                                                           \
    do {                                                                                                        \
        hipError_t _e = (call);                                                                                 \
        if (_e != hipSuccess) return mfail((n), MPLB_E_HIP, std::string(#call) + ": " + hipGetErrorString(_e)); \
    } while (0)

template <typename T>
int alloc(mplb_mlp* n, T** ptr, size_t count) {
    void* q = nullptr;
    MCHK(n, hipMalloc(&q, sizeof(T) * (count ? count : 1)));
    MCHK(n, hipMemset(q, 0, sizeof(T) * (count ? count : 1)));
    n->owned.push_back(q);
    *ptr = (T*)q;
    return 0;
}

template <typename T>
int ensure(mplb_mlp* n, T** ptr, size_t* cap, size_t count) {
    if (count <= *cap) return 0;
    if (*ptr) MCHK(n, hipFree(*ptr));
    *ptr = nullptr;
    MCHK(n, hipMalloc((void**)ptr, sizeof(T) * count));
    *cap = count;
    return 0;
}

dim3 gemm_grid(int M, int N) { return dim3((unsigned)((N + kTile - 1) / kTile), (unsigned)((M + kTile - 1) / kTile)); }

void refresh(mplb_mlp* n) {
    if (n->L <= kRefreshLayers) {
        RefreshAll a{};
        a.L = n->L;
        a.pieces = n->lds_bwd != 0;
        for (int l = 0; l < n->L; l++) {
            a.start[l + 1] = a.start[l] + (int64_t)n->wp[l] * n->w[l + 1];
            a.W[l] = n->p + n->woff[l];
            a.din[l] = n->w[l];
            a.dinp[l] = n->wp[l];
            a.dout[l] = n->w[l + 1];
            a.Wb[l] = n->Wb[l];
            a.Wbt[l] = n->Wbt[l];
        }
        k_refresh_all<<<(unsigned)((a.start[n->L] + 255) / 256), 256, 0, n->stream>>>(a);
        return;
    }
    for (int l = 0; l < n->L; l++) {
        const int total = n->wp[l] * n->w[l + 1];
        k_refresh<<<(total + 255) / 256, 256, 0, n->stream>>>(n->p + n->woff[l], n->w[l], n->wp[l], n->w[l + 1],
                                                              n->Wb[l], n->Wbt[l]);
    }
}

void forward(mplb_mlp* n) {
    const int B = n->B;
    for (int l = 0; l < n->L; l++) {
        Gemm g{};
        g.A = n->ab[l];
        g.lda = n->wp[l];
        g.Bt = n->Wbt[l];
        g.ldb = n->wp[l];
        g.M = B;
        g.N = n->w[l + 1];
        g.K = n->wp[l];
        g.bias = n->p + n->boff[l];
        if (l < n->L - 1) {
            g.out32 = n->a32[l + 1];
            g.ld32 = g.N;
            g.outb = n->ab[l + 1];
            g.ldob = g.N;
            g.outbt = n->abt[l + 1];
            g.ldobt = B;
            k_gemm<E_HIDDEN><<<gemm_grid(g.M, g.N), 256, 0, n->stream>>>(g);
        } else {
            g.out32 = n->y;
            g.ld32 = g.N;
            k_gemm<E_OUT><<<gemm_grid(g.M, g.N), 256, 0, n->stream>>>(g);
        }
    }
}

void backward(mplb_mlp* n) {
    const int B = n->B, L = n->L;
    const int nout = n->w[L];
    k_loss<<<B, 256, 0, n->stream>>>(n->y, n->tgt, B, nout, n->dz32[L], n->dzb[L], n->dzt[L], n->rowsum);
    k_loss_final<<<1, 64, 0, n->stream>>>(n->rowsum, B, nout, n->counter, n->hist, n->loss);
    for (int l = L - 1; l >= 0; l--) {
        const int din = n->wp[l], dout = n->w[l + 1];
        Gemm gw{};
        gw.A = n->abt[l];
        gw.lda = B;
        gw.Bt = n->dzt[l + 1];
        gw.ldb = B;
        gw.M = din;
        gw.N = dout;
        gw.K = B;
        gw.out32 = n->g + n->woff[l];
        gw.ld32 = dout;
        gw.mvalid = n->w[l];
        k_gemm<E_DW><<<gemm_grid(gw.M, gw.N), 256, 0, n->stream>>>(gw);
        k_bias_grad<<<(dout + 63) / 64, 256, 0, n->stream>>>(n->dz32[l + 1], B, dout, n->g + n->boff[l]);
        if (l > 0) {
            Gemm gx{};
            gx.A = n->dzb[l + 1];
            gx.lda = dout;
            gx.Bt = n->Wb[l];
            gx.ldb = dout;
            gx.M = B;
            gx.N = din;
            gx.K = dout;
            gx.out32 = n->dz32[l];
            gx.ld32 = din;
            gx.outb = n->dzb[l];
            gx.ldob = din;
            gx.outbt = n->dzt[l];
            gx.ldobt = B;
            gx.act = n->a32[l];
            gx.ldact = din;
            k_gemm<E_DX><<<gemm_grid(gx.M, gx.N), 256, 0, n->stream>>>(gx);
        }
    }
}

// The two-launch path takes networks whose row workgroup fits its LDS; wider or deeper ones
// keep one launch per product.
constexpr size_t kRowsLds = 150 * 1024;

Net net_args(mplb_mlp* n) {
    Net g{};
    g.L = n->L;
    g.B = n->B;
    g.rows = n->B;
    for (int l = 0; l <= n->L; l++) {
        g.w[l] = n->w[l];
        g.wp[l] = n->wp[l];
        g.wmax = std::max(g.wmax, n->wp[l]);
        g.dzt[l] = n->dzt[l];
        g.dz32[l] = n->dz32[l];
        g.dzb[l] = n->dzb[l];
        g.a32[l] = n->a32[l];
    }
    for (int l = 0; l < n->L; l++) {
        g.Wb[l] = n->Wb[l];
        g.Wbt[l] = n->Wbt[l];
        g.bias[l] = n->p + n->boff[l];
        g.abt[l] = n->abt[l];
        g.ab[l] = n->ab[l];
    }
    g.X = n->X;
    g.T = n->T;
    g.counter = n->counter;
    g.ykeep = n->y;
    g.rowsum = n->rowsum;
    return g;
}

Grads grad_args(mplb_mlp* n, int* blocks) {
    Grads g{};
    g.L = n->L;
    g.B = n->B;
    for (int l = 0; l <= n->L; l++) {
        g.w[l] = n->w[l];
        g.wp[l] = n->wp[l];
        g.dzt[l] = n->dzt[l];
        g.dz32[l] = n->dz32[l];
    }
    int at = 1;
    for (int l = 0; l < n->L; l++) {
        g.abt[l] = n->abt[l];
        g.Wb[l] = n->Wb[l];
        g.Wbt[l] = n->Wbt[l];
        g.woff[l] = n->woff[l];
        g.boff[l] = n->boff[l];
        g.bias0[l] = at;
        at += (n->w[l + 1] + 63) / 64;
    }
    g.bias0[n->L] = at;
    for (int l = 0; l < n->L; l++) {
        g.tile0[l] = at;
        at += n->wp[l] / 32 * (n->w[l + 1] / 32);
    }
    g.tile0[n->L] = at;
    g.grad = n->g;
    g.rowsum = n->rowsum;
    g.counter = n->counter;
    g.loss = n->loss;
    *blocks = at;
    return g;
}

}  // namespace

extern "C" {

int mplb_mlp_create(int nlayers, const int* widths, int batch, int device, mplb_mlp** out) {
    if (!out) return MPLB_E_ARG;
    *out = nullptr;
    if (nlayers < 1 || !widths) return MPLB_E_ARG;
    mplb_mlp* n = new mplb_mlp();
    *out = n;
    n->L = nlayers;
    n->w.assign(widths, widths + nlayers + 1);
    if (n->w[0] < 1 || n->w[0] > kInPad) return mfail(n, MPLB_E_ARG, "input width must be in [1, 32]");
    for (int l = 1; l <= nlayers; l++)
        if (n->w[l] < 32 || n->w[l] % 32) return mfail(n, MPLB_E_ARG, "layer widths must be multiples of 32");
    if (batch < 32 || batch % 32) return mfail(n, MPLB_E_ARG, "batch must be a multiple of 32");
    n->B = batch;
    n->wp = n->w;
    n->wp[0] = kInPad;
    for (int l = 0; l < nlayers; l++) {
        n->woff.push_back(n->P);
        n->P += (int64_t)n->w[l] * n->w[l + 1];
        n->boff.push_back(n->P);
        n->P += n->w[l + 1];
    }
    n->dev = device;
    MCHK(n, hipSetDevice(device));
    MCHK(n, hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking));
    int rc = 0;
    rc |= alloc(n, &n->p, n->P);
    rc |= alloc(n, &n->g, n->P);
    rc |= alloc(n, &n->m, n->P);
    rc |= alloc(n, &n->v, n->P);
    n->Wb.resize(nlayers);
    n->Wbt.resize(nlayers);
    for (int l = 0; l < nlayers; l++) {
        rc |= alloc(n, &n->Wb[l], (size_t)n->wp[l] * n->w[l + 1]);
        rc |= alloc(n, &n->Wbt[l], (size_t)n->wp[l] * n->w[l + 1]);
    }
    n->ab.assign(nlayers, nullptr);
    n->abt.assign(nlayers, nullptr);
    n->a32.assign(nlayers + 1, nullptr);
    n->dz32.assign(nlayers + 1, nullptr);
    n->dzb.assign(nlayers + 1, nullptr);
    n->dzt.assign(nlayers + 1, nullptr);
    for (int j = 0; j < nlayers; j++) {
        rc |= alloc(n, &n->ab[j], (size_t)batch * n->wp[j]);
        rc |= alloc(n, &n->abt[j], (size_t)batch * n->wp[j]);
        if (j > 0) rc |= alloc(n, &n->a32[j], (size_t)batch * n->wp[j]);
    }
    for (int j = 1; j <= nlayers; j++) {
        rc |= alloc(n, &n->dz32[j], (size_t)batch * n->wp[j]);
        rc |= alloc(n, &n->dzb[j], (size_t)batch * n->wp[j]);
        rc |= alloc(n, &n->dzt[j], (size_t)batch * n->wp[j]);
    }
    rc |= alloc(n, &n->y, (size_t)batch * n->w[nlayers]);
    rc |= alloc(n, &n->tgt, (size_t)batch * n->w[nlayers]);
    rc |= alloc(n, &n->rowsum, (size_t)batch);
    rc |= alloc(n, &n->loss, 1);
    rc |= alloc(n, &n->counter, 2);
    if (rc) return MPLB_E_HIP;
    const size_t lds = rows_lds(nlayers, n->w.data(), n->wp.data(), true);
    if (nlayers <= kNetLayers && lds <= kRowsLds) {
        n->lds_bwd = lds;
        n->lds_fwd = rows_lds(nlayers, n->w.data(), n->wp.data(), false);
        MCHK(n, hipFuncSetAttribute((const void*)k_rows<false, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)kRowsLds));
        MCHK(n, hipFuncSetAttribute((const void*)k_rows<true, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)kRowsLds));
        MCHK(n, hipFuncSetAttribute((const void*)k_rows<true, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)kRowsLds));
    }
    return 0;
}

int mplb_mlp_close(mplb_mlp* n) {
    if (!n) return MPLB_E_ARG;
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    for (void* q : n->owned) (void)hipFree(q);
    void* extra[] = {n->X, n->T, n->idx, n->hist, n->Y};
    for (void* q : extra)
        if (q) (void)hipFree(q);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
    return 0;
}

const char* mplb_mlp_last_error(const mplb_mlp* n) { return n ? n->err.c_str() : "null network handle"; }

int64_t mplb_mlp_num_params(const mplb_mlp* n) { return n ? n->P : -1; }

int mplb_mlp_set_params(mplb_mlp* n, const float* params, size_t count) {
    if (!n || !params) return MPLB_E_ARG;
    if ((int64_t)count != n->P) return mfail(n, MPLB_E_ARG, "parameter count differs from the network's");
    MCHK(n, hipSetDevice(n->dev));
    MCHK(n, hipMemcpyAsync(n->p, params, sizeof(float) * count, hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(k_set_int, 1, 1, 0, n->stream, n->counter, 0);
    const size_t bytes = sizeof(float) * count;
    MCHK(n, hipMemsetAsync(n->m, 0, bytes, n->stream));
    MCHK(n, hipMemsetAsync(n->v, 0, bytes, n->stream));
    refresh(n);
    MCHK(n, hipGetLastError());
    MCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

int mplb_mlp_get_params(mplb_mlp* n, float* params, size_t count) {
    if (!n || !params) return MPLB_E_ARG;
    if ((int64_t)count != n->P) return mfail(n, MPLB_E_ARG, "parameter count differs from the network's");
    MCHK(n, hipSetDevice(n->dev));
    MCHK(n, hipMemcpyAsync(params, n->p, sizeof(float) * count, hipMemcpyDeviceToHost, n->stream));
    MCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

int mplb_mlp_forward(mplb_mlp* n, const float* x, int rows, float* y) {
    if (!n || !x || !y || rows < 0) return MPLB_E_ARG;
    MCHK(n, hipSetDevice(n->dev));
    const int din = n->w[0], dout = n->w[n->L], B = n->B;
    if (n->lds_bwd) {
        const int chunk = std::max(1, 65536 / B) * B;    // rows on the device at a time
        const size_t most = (size_t)std::min(rows, chunk);
        int rc = ensure(n, &n->X, &n->X_cap, most * din);
        if (!rc) rc = ensure(n, &n->Y, &n->Y_cap, most * dout);
        if (rc) return rc;
        Net g = net_args(n);
        g.y = n->Y;
        for (int r0 = 0; r0 < rows; r0 += chunk) {
            g.B = g.rows = std::min(chunk, rows - r0);
            // the last batch of rows stays for mplb_mlp_tensor, filled up with empty ones
            g.keep0 = (g.rows - 1) / B * B;
            MCHK(n, hipMemcpyAsync(n->X, x + (size_t)r0 * din, sizeof(float) * g.rows * din, hipMemcpyHostToDevice,
                                   n->stream));
            k_rows<false, true><<<(unsigned)((g.keep0 + B) / kRows), kRowThreads, n->lds_fwd, n->stream>>>(g);
            MCHK(n, hipGetLastError());
            MCHK(n, hipMemcpyAsync(y + (size_t)r0 * dout, n->Y, sizeof(float) * g.rows * dout, hipMemcpyDeviceToHost,
                                   n->stream));
            MCHK(n, hipStreamSynchronize(n->stream));
        }
        return 0;
    }
    int rc = ensure(n, &n->X, &n->X_cap, (size_t)B * din);
    if (rc) return rc;
    std::vector<float> xb((size_t)B * din), yb((size_t)B * dout);
    for (int r0 = 0; r0 < rows; r0 += B) {
        const int cnt = std::min(B, rows - r0);
        std::fill(xb.begin(), xb.end(), 0.f);
        std::memcpy(xb.data(), x + (size_t)r0 * din, sizeof(float) * cnt * din);
        MCHK(n, hipMemcpyAsync(n->X, xb.data(), sizeof(float) * xb.size(), hipMemcpyHostToDevice, n->stream));
        k_gather<<<B, 64, 0, n->stream>>>(n->X, nullptr, nullptr, nullptr, B, din, dout, n->ab[0], n->abt[0],
                                          nullptr);
        forward(n);
        MCHK(n, hipGetLastError());
        MCHK(n, hipMemcpyAsync(yb.data(), n->y, sizeof(float) * yb.size(), hipMemcpyDeviceToHost, n->stream));
        MCHK(n, hipStreamSynchronize(n->stream));
        std::memcpy(y + (size_t)r0 * dout, yb.data(), sizeof(float) * cnt * dout);
    }
    return 0;
}

int mplb_mlp_gradient(mplb_mlp* n, const float* x, const float* t, float* loss, float* grad, size_t ngrad) {
    if (!n || !x || !t) return MPLB_E_ARG;
    if (grad && (int64_t)ngrad != n->P) return mfail(n, MPLB_E_ARG, "gradient size differs from the parameter count");
    MCHK(n, hipSetDevice(n->dev));
    const int din = n->w[0], dout = n->w[n->L], B = n->B;
    int rc = ensure(n, &n->X, &n->X_cap, (size_t)B * din);
    if (!rc) rc = ensure(n, &n->T, &n->T_cap, (size_t)B * dout);
    if (rc) return rc;
    MCHK(n, hipMemcpyAsync(n->X, x, sizeof(float) * B * din, hipMemcpyHostToDevice, n->stream));
    MCHK(n, hipMemcpyAsync(n->T, t, sizeof(float) * B * dout, hipMemcpyHostToDevice, n->stream));
    if (n->lds_bwd) {
        int blocks = 0;
        const Grads g = grad_args(n, &blocks);
        k_rows<true, true><<<(unsigned)(B / kRows + 8 * kHelpers), kRowThreads, n->lds_bwd, n->stream>>>(net_args(n));
        k_weights<false><<<(unsigned)blocks, 256, 0, n->stream>>>(g);
    } else {
        k_gather<<<B, 64, 0, n->stream>>>(n->X, n->T, nullptr, nullptr, B, din, dout, n->ab[0], n->abt[0], n->tgt);
        float* keep = n->hist;
        n->hist = nullptr;
        forward(n);
        backward(n);
        n->hist = keep;
    }
    MCHK(n, hipGetLastError());
    if (loss) MCHK(n, hipMemcpyAsync(loss, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->stream));
    if (grad) MCHK(n, hipMemcpyAsync(grad, n->g, sizeof(float) * ngrad, hipMemcpyDeviceToHost, n->stream));
    MCHK(n, hipStreamSynchronize(n->stream));
    return 0;
}

int mplb_mlp_train(mplb_mlp* n, const float* X, const float* T, int nsamples, const int32_t* idx, int iters,
                   float lr, float beta1, float beta2, float eps, float* loss_hist) {
    if (!n || !X || !T || !idx || nsamples <= 0 || iters <= 0) return MPLB_E_ARG;
    MCHK(n, hipSetDevice(n->dev));
    const int din = n->w[0], dout = n->w[n->L], B = n->B;
    for (int64_t i = 0; i < (int64_t)iters * B; i++)
        if (idx[i] < 0 || idx[i] >= nsamples) return mfail(n, MPLB_E_ARG, "minibatch index out of range");
    int rc = ensure(n, &n->X, &n->X_cap, (size_t)nsamples * din);
    if (!rc) rc = ensure(n, &n->T, &n->T_cap, (size_t)nsamples * dout);
    if (!rc) rc = ensure(n, &n->idx, &n->idx_cap, (size_t)iters * B);
    if (!rc) rc = ensure(n, &n->hist, &n->hist_cap, (size_t)iters);
    if (rc) return rc;
    MCHK(n, hipMemcpyAsync(n->X, X, sizeof(float) * nsamples * din, hipMemcpyHostToDevice, n->stream));
    MCHK(n, hipMemcpyAsync(n->T, T, sizeof(float) * nsamples * dout, hipMemcpyHostToDevice, n->stream));
    MCHK(n, hipMemcpyAsync(n->idx, idx, sizeof(int32_t) * iters * B, hipMemcpyHostToDevice, n->stream));
    // every call is a fresh Adam run: the iteration counter (index table, loss history,
    // bias-correction step count) restarts and the first and second moments are zeroed
    hipLaunchKernelGGL(k_set_int, 1, 1, 0, n->stream, n->counter, 0);
    hipLaunchKernelGGL(k_set_int, 1, 1, 0, n->stream, n->counter + 1, -1);
    MCHK(n, hipMemsetAsync(n->m, 0, sizeof(float) * n->P, n->stream));
    MCHK(n, hipMemsetAsync(n->v, 0, sizeof(float) * n->P, n->stream));
    MCHK(n, hipStreamSynchronize(n->stream));
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    MCHK(n, hipStreamBeginCapture(n->stream, hipStreamCaptureModeThreadLocal));
    // the last iteration of the two-launch path also leaves its tensors for mplb_mlp_tensor
    auto rows_and_weights = [&](bool keep) {
        int blocks = 0;
        Grads gr = grad_args(n, &blocks);
        gr.hist = n->hist;
        gr.adam = Adam{n->p, n->m, n->v, lr, beta1, beta2, eps};
        Net g = net_args(n);
        g.idx = n->idx;
        g.rows = nsamples;
        const unsigned row_blocks = (unsigned)(B / kRows + 8 * kHelpers);
        if (keep) k_rows<true, true><<<row_blocks, kRowThreads, n->lds_bwd, n->stream>>>(g);
        else k_rows<true, false><<<row_blocks, kRowThreads, n->lds_bwd, n->stream>>>(g);
        k_weights<true><<<(unsigned)blocks, 256, 0, n->stream>>>(gr);
    };
    if (n->lds_bwd) {
        rows_and_weights(false);
    } else {
        k_gather<<<B, 64, 0, n->stream>>>(n->X, n->T, n->idx, n->counter, B, din, dout, n->ab[0], n->abt[0], n->tgt);
        forward(n);
        backward(n);
        k_adam<<<(unsigned)((n->P + 255) / 256), 256, 0, n->stream>>>(n->p, n->g, n->m, n->v, n->P, lr, beta1, beta2,
                                                                       eps, n->counter);
        refresh(n);
        k_advance<<<1, 64, 0, n->stream>>>(n->counter);
    }
    MCHK(n, hipStreamEndCapture(n->stream, &graph));
    MCHK(n, hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    for (int it = n->lds_bwd ? 1 : 0; it < iters; it++) MCHK(n, hipGraphLaunch(exec, n->stream));
    if (n->lds_bwd) {
        rows_and_weights(true);
        MCHK(n, hipGetLastError());
    }
    MCHK(n, hipStreamSynchronize(n->stream));
    MCHK(n, hipGraphExecDestroy(exec));
    MCHK(n, hipGraphDestroy(graph));
    if (loss_hist) MCHK(n, hipMemcpy(loss_hist, n->hist, sizeof(float) * iters, hipMemcpyDeviceToHost));
    return 0;
}

// Intermediate tensors of the last forward, gradient or training call (its last batch), as FP32 (BF16 ones widened):
// "x" level-0 BF16 input [B][32]; "a" level j BF16 activation [B][w_j] (j = 0..L-1);
// "a32" FP32 activation (1..L-1); "y" output [B][w_L]; "dz" FP32 dL/dz of level j
// (1..L); "dzb" its BF16 copy; "wb" BF16 weights of layer j [32 or w_j][w_j+1].
int mplb_mlp_tensor(mplb_mlp* n, const char* name, int j, float* out, size_t count) {
    if (!n || !name || !out) return MPLB_E_ARG;
    MCHK(n, hipSetDevice(n->dev));
    const int B = n->B, L = n->L;
    const void* src = nullptr;
    bool is_bf = false;
    size_t want = 0;
    if (!std::strcmp(name, "a") && j >= 0 && j < L) {
        src = n->ab[j];
        is_bf = true;
        want = (size_t)B * n->wp[j];
    } else if (!std::strcmp(name, "a32") && j >= 1 && j < L) {
        src = n->a32[j];
        want = (size_t)B * n->wp[j];
    } else if (!std::strcmp(name, "y")) {
        src = n->y;
        want = (size_t)B * n->w[L];
    } else if (!std::strcmp(name, "dz") && j >= 1 && j <= L) {
        src = n->dz32[j];
        want = (size_t)B * n->wp[j];
    } else if (!std::strcmp(name, "dzb") && j >= 1 && j <= L) {
        src = n->dzb[j];
        is_bf = true;
        want = (size_t)B * n->wp[j];
    } else if (!std::strcmp(name, "wb") && j >= 0 && j < L) {
        src = n->Wb[j];
        is_bf = true;
        want = (size_t)n->wp[j] * n->w[j + 1];
    } else {
        return mfail(n, MPLB_E_ARG, std::string("unknown tensor ") + name);
    }
    if (count != want) return mfail(n, MPLB_E_ARG, "tensor size mismatch");
    if (is_bf) {
        std::vector<uint16_t> h(count);
        MCHK(n, hipMemcpy(h.data(), src, 2 * count, hipMemcpyDeviceToHost));
        const int cols = !std::strcmp(name, "wb") ? n->w[j + 1] : 0;
        for (size_t i = 0; i < count; i++) {
            const size_t at = n->lds_bwd && cols ? frag((int)(i / cols), (int)(i % cols), cols) : i;
            const uint32_t u = (uint32_t)h[at] << 16;
            std::memcpy(&out[i], &u, 4);
        }
    } else {
        MCHK(n, hipMemcpy(out, src, 4 * count, hipMemcpyDeviceToHost));
    }
    return 0;
}

}  // extern "C"
