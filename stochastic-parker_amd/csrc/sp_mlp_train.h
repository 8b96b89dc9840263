// sp_mlp_train.h -- one AdamW step of the surrogate network in two launches.
// Included by sp_mlp.hip after its device helpers.
//
// Layer by layer a step is 37 dependent launches of 4096 x 256 x 256 work, each
// of 2-12 us: 210 us for 5.3 GFLOP.  The rows of a batch meet only in the
// weight gradients, so a step is
//   train_rows_kernel     each block takes 32 rows through the whole forward
//                         and backward chain: activations in LDS, the
//                         pre-activations of the rows in registers, weights
//                         streamed from L2 as MFMA fragments;
//   train_update_kernel   each block owns a 32 x 32 tile of one weight matrix
//                         (or 32 biases): its gradient over all rows, AdamW,
//                         and the BF16 copies that the next step reads.
// 32-row blocks give 128 blocks at the batch size of 4096 and keep every
// accumulation a chain of 32x32x16 MFMAs in the order of the layer-by-layer
// kernels, whose split-K and column-sum orders the update kernel follows too:
// parameters and losses are the same bits.  Batch 4096, 256 x 4 hidden: 210 ->
// 38 us per step, 21 + 14: a hidden layer takes the first kernel about 3700
// cycles, the time of each CU's 128 KiB of weights from L2 (35 B per clock) and
// of the BF16 activations' way to memory; the second reads 512 KiB of operands
// per CU at 27 B per clock (43 % of its requests hit L2: blocks on all dies wrote
// them).  Neither dealing the layers to the dies, nor
// streaming stores, nor other places for the fragments changed the sum of both.
#pragma once

namespace sp {
namespace mlp {

constexpr int kTrainRows = 32;        // rows per block
constexpr int kTrainMaxHidden = 5;    // pre-activations of more layers would spill
constexpr int kLossParts = 256;       // partial sums of the squared error (mse_kernel's blocks)
constexpr int kUpdateBlock = 1024;
constexpr int kUpdateSplits = 32;     // row ranges of a weight gradient, at most

// Activations X_l and pre-activation gradients G_l go to memory as operands of
// the weight gradient, rows along k: per 32-feature tile and 16-row step the 64
// lanes' 8-element operands of one MFMA in 1 KiB (as frag_index with rows for
// k).  `rs` row steps cover the batch padded to 32 rows, zeros past its end.
struct RowFrags {
    int rs, nlh;                      // row steps; hidden features / 32
    __host__ __device__ long long x(int l) const { return 512ll * rs * (l == 0 ? 0 : 1 + (l - 1) * nlh); }
    __host__ __device__ long long g(int l) const { return 512ll * rs * l * nlh; }
};

struct RowsArgs {
    const float* xd;                  // data set
    const float* td;
    uint32_t nd, step, k0, k1;        // its rows, step of the loop, Philox key
    int rows, nin, nout;
    RowFrags fr;
    const uint16_t* wf;               // fragment-ordered weights, forward
    const uint16_t* wb;               // and transposed, for the layers 1 ..
    const float* p;
    long long boff[kTrainMaxHidden + 1];
    uint16_t* xf;
    uint16_t* gf;
    float* sq;                        // squared errors, rows x nout
    float scale;                      // 1 / (rows nout)
    float* adam;                      // lr, c1, c2 of this step, for the update kernel
    uint32_t t, nsteps;               // AdamW steps taken; length of the loop
    float lr0, lr_min, b1, b2;
};

// acc += W-fragments (wq, KS k-steps) x the rows in LDS; slot ks of wq is
// refilled from `next` (NEXT fragments) as soon as it is consumed, so the next
// layer's weights are in flight through the epilogue and the barrier.
template <int LD, int KS, int NEXT, int NQ>
__device__ __forceinline__ void rows_mma(const uint16_t* act, v8bf (&wq)[NQ], v16f& acc,
                                         const v8bf* next, int lane) {
    const uint16_t* row = act + (lane & 31) * LD + 8 * (lane >> 5);
    constexpr int PF = KS < 4 ? KS : 4;
    v8bf b[PF];
#pragma unroll
    for (int i = 0; i < PF; ++i) b[i] = *reinterpret_cast<const v8bf*>(row + 16 * i);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wq[ks], b[ks % PF], acc, 0, 0, 0);
        if (ks + PF < KS) b[ks % PF] = *reinterpret_cast<const v8bf*>(row + 16 * (ks + PF));
        if (ks < NEXT) wq[ks] = next[ks * 64 + lane];
    }
}

// The wave's 32 features x 32 rows (v[4 g + q]: feature 8 g + 4 (lane / 32) + q
// of row lane % 32) as BF16 into the LDS rows; rows past the batch (mask 0)
// as zeros.
template <int LD>
__device__ __forceinline__ void rows_put(uint16_t* act, const float v[16], uint32_t mask, int tile, int lane) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint2 u;
        u.x = bf16x2_rne(v[4 * g], v[4 * g + 1]) & mask;
        u.y = bf16x2_rne(v[4 * g + 2], v[4 * g + 3]) & mask;
        *reinterpret_cast<uint2*>(&act[(lane & 31) * LD + 32 * tile + 8 * g + 4 * (lane >> 5)]) = u;
    }
}

// The same 32 x 32 values from the LDS rows, transposed: the lane's operands of
// the two row fragments of feature tile `tile`, and their store.  The reads
// come behind the barrier that follows rows_put, in the gaps of the next
// layer's MFMA chain; the stores behind that chain's weight loads, since loads
// and stores complete in order and the next layer would wait for the stores.
template <int LD>
__device__ __forceinline__ void frag_read(const uint16_t* act, uint32_t (&u)[8], int tile, int lane) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint16_t* col = act + (16 * h + 8 * (lane >> 5)) * LD + 32 * tile + (lane & 31);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            u[4 * h + i] = (uint32_t)col[2 * i * LD] | ((uint32_t)col[(2 * i + 1) * LD] << 16);
    }
}

__device__ __forceinline__ void frag_store(uint16_t* frag, const uint32_t (&u)[8], int tile, int rs, int lane) {
    __builtin_amdgcn_sched_barrier(0);
    uint4* f = reinterpret_cast<uint4*>(frag) + tile * (long long)rs * 64 + lane;
    const int st = 2 * (int)blockIdx.x;
    f[st * 64] = uint4{u[0], u[1], u[2], u[3]};
    f[(st + 1) * 64] = uint4{u[4], u[5], u[6], u[7]};
}

// NL hidden layers of H features; H / 32 waves, each 32 features of every
// layer.  Linear layer l maps X_l to Z_l: X_0 the input, X_{l+1} = silu(Z_l),
// Z_NL the output.
template <int H, int NL>
__global__ void __launch_bounds__(2 * H) train_rows_kernel(RowsArgs a) {
    constexpr int LD = H + 8, KSH = H / 16;
    __shared__ __align__(16) uint16_t act[2][kTrainRows * LD];
    __shared__ __align__(16) float sb[NL * H + H];
    __shared__ uint32_t src[kTrainRows];
    // the wave index as a scalar: weight and fragment addresses then are
    // scalar bases plus a lane offset
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int r0 = blockIdx.x * kTrainRows;
    const bool valid = r0 + (lane & 31) < a.rows;
    const uint32_t mask = valid ? 0xFFFFFFFFu : 0u;
    const v8bf* wf = reinterpret_cast<const v8bf*>(a.wf);
    const v8bf* wb = reinterpret_cast<const v8bf*>(a.wb);
    // fragment (64 lanes x 8 elements) index of a layer's first fragment for
    // this wave's tile
    auto fwd = [&](int l, int tile) -> const v8bf* {
        return l == 0 ? wf + tile * 64
                      : wf + (H * kFusedKin + (long long)(l - 1) * H * H) / 8 + (long long)tile * KSH * 64;
    };
    auto bwd = [&](int l, int nsteps) -> const v8bf* {
        return wb + (long long)(l - 1) * H * H / 8 + (long long)w * nsteps * 64;
    };
    const int T = a.nout / 32;            // output tiles, at most W
    v8bf w0[1] = {fwd(0, w)[lane]}, wq[KSH];
    if (NL > 1 || w < T) {
        const v8bf* f = fwd(1, w);
#pragma unroll
        for (int i = 0; i < KSH; ++i) wq[i] = f[i * 64 + lane];
    }
    for (int i = threadIdx.x; i < NL * H + a.nout; i += 2 * H) sb[i] = a.p[a.boff[i / H] + i % H];
    // the rows drawn for this step (batch_index_dev_kernel)
    if (threadIdx.x < kTrainRows) {
        const U4 u = philox4x32_10((uint32_t)(r0 + threadIdx.x), a.step, 0x6d6c70u, 0u, a.k0, a.k1);
        src[threadIdx.x] = (uint32_t)(((unsigned long long)u.a * a.nd) >> 32);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kTrainRows * 32; i += 2 * H) {
        const int r = i >> 5, c = i & 31;
        float v = 0.0f;
        if (r0 + r < a.rows && c < a.nin) v = a.xd[(long long)src[r] * a.nin + c];
        act[0][r * LD + c] = bf16_rne(v);
    }
    __syncthreads();
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        // the step's learning rate and bias corrections (adamw_dev_kernel)
        const float f = a.nsteps > 1 ? (float)a.step / (float)(a.nsteps - 1) : 0.0f;
        const float tt = (float)(a.t + 1);
        a.adam[0] = a.lr_min + 0.5f * (a.lr0 - a.lr_min) * (1.0f + cosf(3.14159265358979f * f));
        a.adam[1] = 1.0f - powf(a.b1, tt);
        a.adam[2] = 1.0f - powf(a.b2, tt);
    }
    if (w < 2) {                          // X_0, 16 rows per wave
        uint32_t u[4];
        const uint16_t* col = act[0] + (16 * w + 8 * (lane >> 5)) * LD + (lane & 31);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            u[i] = (uint32_t)col[2 * i * LD] | ((uint32_t)col[(2 * i + 1) * LD] << 16);
        *reinterpret_cast<uint4*>(a.xf + ((2 * (int)blockIdx.x + w) * 64ll + lane) * 8) = uint4{u[0], u[1], u[2], u[3]};
    }
    float dz[NL][16];                     // silu'(Z_l) of the wave's features and rows
    int cur = 0;
    auto bias = [&](int l, v16f& acc) {
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = sb[l * H + 32 * w + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3)];
    };
    // ---- forward through the hidden layers ----
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        v16f z;
        bias(l, z);
        if (l == 0) {
            rows_mma<LD, 1, 0>(act[cur], w0, z, (const v8bf*)nullptr, lane);
        } else {
            uint32_t u[8];
            frag_read<LD>(act[cur], u, w, lane);
            // next: a hidden layer, or the output layer's tile for each of the
            // first T waves (the others read tile 0 and drop it)
            rows_mma<LD, KSH, KSH>(act[cur], wq, z, l + 1 < NL ? fwd(l + 1, w) : fwd(NL, w < T ? w : 0), lane);
            frag_store(a.xf + a.fr.x(l), u, w, a.fr.rs, lane);
        }
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float s = sigmoid(z[j]);
            v[j] = z[j] * s;
            dz[l][j] = s * (1.0f + z[j] * (1.0f - s));
        }
        rows_put<LD>(act[cur ^ 1], v, mask, w, lane);
        cur ^= 1;
        __syncthreads();
    }
    uint32_t u[8];
    frag_read<LD>(act[cur], u, w, lane);
    // ---- output layer, error and its gradient (mse_kernel) ----
    const int oks = a.nout / 16;
    if (w < T) {
        v16f y;
        bias(NL, y);
        rows_mma<LD, KSH, 0>(act[cur], wq, y, (const v8bf*)nullptr, lane);
        float v[16];
        const long long trow = (long long)src[lane & 31] * a.nout;
        const long long orow = (long long)(r0 + (lane & 31)) * a.nout;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int c = 32 * w + 8 * g + 4 * (lane >> 5);
            float4 t = float4{0.0f, 0.0f, 0.0f, 0.0f}, q;
            if (valid) t = *reinterpret_cast<const float4*>(a.td + trow + c);
            const float e0 = y[4 * g] - t.x, e1 = y[4 * g + 1] - t.y;
            const float e2 = y[4 * g + 2] - t.z, e3 = y[4 * g + 3] - t.w;
            q = float4{e0 * e0, e1 * e1, e2 * e2, e3 * e3};
            if (valid) *reinterpret_cast<float4*>(a.sq + orow + c) = q;
            v[4 * g] = 2.0f * e0 * a.scale;
            v[4 * g + 1] = 2.0f * e1 * a.scale;
            v[4 * g + 2] = 2.0f * e2 * a.scale;
            v[4 * g + 3] = 2.0f * e3 * a.scale;
        }
        rows_put<LD>(act[cur ^ 1], v, mask, w, lane);
    }
    // slots 0 .. 7: the output layer's fragments (K = nout <= 128), the others
    // already layer NL - 1's
    {
        const v8bf *f = bwd(NL, oks), *f1 = bwd(NL > 1 ? NL - 1 : 1, KSH);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < oks) wq[i] = f[i * 64 + lane];
#pragma unroll
        for (int i = 8; i < KSH; ++i)
            if (NL > 1) wq[i] = f1[i * 64 + lane];
    }
    frag_store(a.xf + a.fr.x(NL), u, w, a.fr.rs, lane);
    cur ^= 1;
    __syncthreads();
    // ---- backward: G_l = (G_{l+1} W_{l+1}^T) silu'(Z_l) ----
#pragma unroll
    for (int l = NL - 1; l >= 0; --l) {
        v16f acc;
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
        if (l == NL - 1) {
            if (w < T) frag_read<LD>(act[cur], u, w, lane);
            const uint16_t* row = act[cur] + (lane & 31) * LD + 8 * (lane >> 5);
#pragma unroll
            for (int ks = 0; ks < 8; ++ks)
                if (ks < oks)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        wq[ks], *reinterpret_cast<const v8bf*>(row + 16 * ks), acc, 0, 0, 0);
            if (NL > 1) {
                const v8bf* f1 = bwd(NL - 1, KSH);
#pragma unroll
                for (int i = 0; i < 8; ++i) wq[i] = f1[i * 64 + lane];
            }
            if (w < T) frag_store(a.gf + a.fr.g(NL), u, w, a.fr.rs, lane);
        } else {
            frag_read<LD>(act[cur], u, w, lane);
            if (l > 0) rows_mma<LD, KSH, KSH>(act[cur], wq, acc, bwd(l, KSH), lane);
            else rows_mma<LD, KSH, 0>(act[cur], wq, acc, (const v8bf*)nullptr, lane);
            frag_store(a.gf + a.fr.g(l + 1), u, w, a.fr.rs, lane);
        }
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = acc[j] * dz[l][j];
        rows_put<LD>(act[cur ^ 1], v, mask, w, lane);
        cur ^= 1;
        __syncthreads();
    }
    frag_read<LD>(act[cur], u, w, lane);
    frag_store(a.gf + a.fr.g(0), u, w, a.fr.rs, lane);
}

struct UpdateArgs {
    int rows, nin, hidden, nl, nout;
    RowFrags fr;
    const uint16_t* xf;
    const uint16_t* gf;
    const float* sq;
    float *p, *m, *v;
    uint16_t *pb, *wf, *wb;
    long long woff[kTrainMaxHidden + 1], boff[kTrainMaxHidden + 1];
    int kchunk[kTrainMaxHidden + 1];   // rows per split of each layer's weight gradient
    float* loss_parts;                 // kLossParts sums of this step
    const float* adam;                 // lr, c1, c2 (train_rows_kernel)
    float b1, b2, eps, wd;
};

// One parameter with its AdamW moments, and the update of adamw_dev_kernel.
struct Param {
    float p, m, v;
};
__device__ __forceinline__ Param load_param(const UpdateArgs& a, long long i) {
    return Param{a.p[i], a.m[i], a.v[i]};
}
__device__ __forceinline__ uint16_t update_param(const UpdateArgs& a, long long i, const Param& o, float g) {
    const float lr = a.adam[0], c1 = a.adam[1], c2 = a.adam[2];
    const float mi = a.b1 * o.m + (1.0f - a.b1) * g;
    const float vi = a.b2 * o.v + (1.0f - a.b2) * g * g;
    a.m[i] = mi;
    a.v[i] = vi;
    const float upd = (mi / c1) / (sqrtf(vi / c2) + a.eps);
    const float pi = o.p - lr * (upd + a.wd * o.p);
    const uint16_t h = bf16_rne(pi);
    a.p[i] = pi;
    a.pb[i] = h;
    return h;
}

// Loss partial vb of kLossParts: the strided sum and the tree of mse_kernel's
// block vb, by the first 256 threads; `red` holds 256 floats.  Two barriers.
__device__ __forceinline__ void loss_part(const UpdateArgs& a, int vb, float* red) {
    const int t = threadIdx.x;
    const long long count = (long long)a.rows * a.nout;
    __syncthreads();
    if (t < 256) {
        float acc = 0.0f;
#pragma unroll 4
        for (long long i = (long long)vb * 256 + t; i < count; i += kLossParts * 256) acc += a.sq[i];
        red[t] = acc;
    }
    __syncthreads();
    if (t < 64) {
        float x = (red[t] + red[t + 128]) + (red[t + 64] + red[t + 192]);
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) x += __shfl_down(x, s);
        if (t == 0) a.loss_parts[vb] = x;
    }
}

// Blocks, in order: the 32 x 32 tiles of every weight matrix, the 32-column
// tiles of every bias vector; every block also takes its share of the loss
// partials (a few blocks of their own took three times as long as a tile).
// LDS holds a tile's (at most 32) partial products, summed in the order of the splits.
__global__ void __launch_bounds__(kUpdateBlock) train_update_kernel(UpdateArgs a) {
    __shared__ float part[kUpdateSplits][1024];
    __shared__ uint16_t wt[32][34];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rs = a.fr.rs;
    int b = (int)blockIdx.x;
    for (int vb = b; vb < kLossParts; vb += (int)gridDim.x) loss_part(a, vb, part[0]);
    __syncthreads();
    for (int l = 0; l <= a.nl; ++l) {
        const int K = l == 0 ? 32 : a.hidden, N = l == a.nl ? a.nout : a.hidden;
        const int tiles = (K / 32) * (N / 32);
        if (b >= tiles) { b -= tiles; continue; }
        const int kt = b / (N / 32), nt = b % (N / 32);
        const v8bf* A = reinterpret_cast<const v8bf*>(a.xf + a.fr.x(l)) + (long long)kt * rs * 64 + lane;
        const v8bf* B = reinterpret_cast<const v8bf*>(a.gf + a.fr.g(l)) + (long long)nt * rs * 64 + lane;
        const int kk = 8 * (w >> 2) + 4 * (lane >> 5) + (w & 3), k = 32 * kt + kk;
        const int n = 32 * nt + (lane & 31);
        const long long pi = a.woff[l] + (long long)k * N + n;
        const bool real = l > 0 || k < a.nin;
        Param old{0.0f, 0.0f, 0.0f};
        if (real) old = load_param(a, pi);
        const int per = a.kchunk[l] / 16, splits = (rs + per - 1) / per;
        for (int s = w; s < splits; s += kUpdateBlock / 64) {
            v16f acc;
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
            const int e = min(rs, (s + 1) * per);
#pragma unroll 8
            for (int q = s * per; q < e; ++q)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[q * 64], B[q * 64], acc, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 16; ++j) part[s][64 * j + lane] = acc[j];
        }
        __syncthreads();
        float g = 0.0f;
        for (int s = 0; s < splits; ++s) g += part[s][t];
        uint16_t h = 0;
        if (real) h = update_param(a, pi, old, g);
        wt[kk][lane & 31] = h;
        __syncthreads();
        // the fragment copies: 16 bytes of eight k (forward) or eight n (backward)
        const int half = (t >> 6) & 1, c = lane & 31, o = 16 * half + 8 * (lane >> 5);
        uint32_t u[4];
        if (w < 2 && (l > 0 || half == 0)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = (uint32_t)wt[o + 2 * i][c] | ((uint32_t)wt[o + 2 * i + 1][c] << 16);
            const int Ks = l == 0 ? kFusedKin / 16 : K / 16;
            const long long off = l == 0 ? 0 : (long long)a.hidden * kFusedKin + (long long)(l - 1) * a.hidden * a.hidden;
            *reinterpret_cast<uint4*>(a.wf + off + (((long long)nt * Ks + 2 * kt + half) * 64 + lane) * 8) =
                uint4{u[0], u[1], u[2], u[3]};
        } else if (w >= 2 && w < 4 && l > 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = (uint32_t)wt[c][o + 2 * i] | ((uint32_t)wt[c][o + 2 * i + 1] << 16);
            const long long off = (long long)(l - 1) * a.hidden * a.hidden;
            *reinterpret_cast<uint4*>(a.wb + off + (((long long)kt * (N / 16) + 2 * nt + half) * 64 + lane) * 8) =
                uint4{u[0], u[1], u[2], u[3]};
        }
        return;
    }
    for (int l = 0; l <= a.nl; ++l) {
        // bias gradients: kColParts row chunks, in each 32 row phases
        // (colsum_part_kernel), both summed in order
        const int N = l == a.nl ? a.nout : a.hidden;
        if (b >= N / 32) { b -= N / 32; continue; }
        const uint16_t* G = a.gf + a.fr.g(l) + (long long)b * rs * 512;
        const int chunk = (a.rows + kColParts - 1) / kColParts;
        static_assert(2 * kColParts <= kUpdateSplits, "each row chunk's 32 x 32 phase sums take two rows of part");
        static_assert(kColParts * 32 <= kUpdateBlock, "one thread per chunk and column");
        if (chunk % 32 == 0) {
            // whole 32-row groups (zeros past the batch): eight phases per load
            for (int i = t; i < kColParts * 128; i += kUpdateBlock) {
                const int c = i & 31, q = (i >> 5) & 3, pt = i >> 7;
                float s[8] = {};
#pragma unroll 4
                for (int j = 0; j < min(chunk / 32, (16 * rs - pt * chunk) / 32); ++j) {
                    const int st = (pt * chunk + 32 * j) / 16 + (q >> 1);
                    const uint4 u = *reinterpret_cast<const uint4*>(G + ((long long)st * 64 + c + 32 * (q & 1)) * 8);
                    const uint32_t x[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        s[2 * k] += __uint_as_float(x[k] << 16);
                        s[2 * k + 1] += __uint_as_float(x[k] & 0xFFFF0000u);
                    }
                }
#pragma unroll
                for (int k = 0; k < 8; ++k) part[2 * pt + (q >> 1)][((q & 1) * 8 + k) * 32 + c] = s[k];
            }
        } else {
            const int c = t & 31, ph = t >> 5;
            for (int pt = 0; pt < kColParts; ++pt) {
                float s = 0.0f;
                const int r1 = min(a.rows, (pt + 1) * chunk);
                for (int r = pt * chunk + ph; r < r1; r += 256) {
                    float x[8];   // eight loads in flight; zeros past the chunk
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const int q = r + 32 * k;
                        x[k] = q < r1 ? bf16_to_f(G[((long long)(q >> 4) * 64 + c + 32 * ((q >> 3) & 1)) * 8 + (q & 7)]) : 0.0f;
                    }
#pragma unroll
                    for (int k = 0; k < 8; ++k) s += x[k];
                }
                part[2 * pt + (ph >> 4)][(ph & 15) * 32 + c] = s;
            }
        }
        __syncthreads();
        float s = 0.0f;
        if (t < kColParts * 32)
            for (int ph = 0; ph < 32; ++ph) s += part[2 * (t >> 5) + (ph >> 4)][(ph & 15) * 32 + (t & 31)];
        __syncthreads();
        if (t < kColParts * 32) part[0][t] = s;
        __syncthreads();
        if (t < 32) {
            float g = 0.0f;
            for (int pt = 0; pt < kColParts; ++pt) g += part[0][32 * pt + t];
            const long long pi = a.boff[l] + 32 * b + t;
            update_param(a, pi, load_param(a, pi), g);
        }
        return;
    }
}

// losses[s] = scale * sum of step s's partials (loss_dev_kernel), one block per step.
__global__ void __launch_bounds__(256) train_loss_kernel(const float* parts, float scale, float* losses) {
    __shared__ float red[256];
    red[threadIdx.x] = parts[(long long)blockIdx.x * kLossParts + threadIdx.x];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) losses[blockIdx.x] = red[0] * scale;
}

// out = W (K x N row-major BF16) transposed in fragment order: per 32-row tile
// of k and 16-column step, lane k % 32 + 32 ((n / 8) % 2) holds n .. n + 7.
__global__ void frag_back_kernel(const uint16_t* w, int K, int N, uint16_t* out) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)K * N) return;
    const int k = (int)(i / N), n = (int)(i % N);
    out[frag_index(n, k, N)] = w[i];
}

}  // namespace mlp
}  // namespace sp
