// sp_mlp_query.h -- ensemble spectra of few rows in one launch.
// Included by sp_mlp.hip after sp_mlp_train.h.
//
// A query of eight rows took two launches and three copies, 69 us, 18.5 of them
// in an inference kernel whose blocks are built for 128 rows.  Here a block
// takes 32 rows through all members at once, 2 H threads per member (its waves
// as in train_rows_kernel: 32 features each, the next layer's weight fragments
// in flight through the epilogue), and turns their outputs, left in LDS, into
// mean spectrum and spread.  Inputs and results may lie in pinned host memory:
// each member's threads read the rows once and each result is written once.
// Every accumulation and rounding is that of mlp_infer_kernel and ensemble_kernel.
#pragma once

namespace sp {
namespace mlp {

constexpr int kQueryRows = 32;         // rows per block
constexpr int kQueryThreads = 1024;    // threads of a block at most
constexpr int kQueryMembers = 4;       // members at H = 128 (two at 256)

struct QueryArgs {
    FusedArgs f;                       // y unused
    int members, nout;
    float floor;
    float* spec;
    float* spread;
};

// Rows in several pinned slots (x, spec and spread then unused), of `per` blocks
// each: their spectra, spreads and inputs one after the other.  Arguments of a
// kernel of its own, which other queries do not wait for (0.5 us).
struct QueryPieces : QueryArgs {
    int per;
    char* slot[PinnedSlots::kMax];
};

template <int H, class Args>
__global__ void __launch_bounds__(kQueryThreads) mlp_query_kernel(Args a) {
    constexpr int M = kQueryThreads / (2 * H), LD = H + 8, KSH = H / 16, LY = 128 + 4;
    static_assert(M <= kQueryMembers, "members of a block");
    __shared__ __align__(16) uint16_t act[M][2][kQueryRows * LD];
    __shared__ __align__(16) float y[M][kQueryRows * LY];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = wv / (H / 32), w = wv % (H / 32);       // member, wave of the member
    const int tid = threadIdx.x - g * 2 * H;
    const int left = a.f.rows - (int)blockIdx.x * kQueryRows;   // rows from this block's first on
    const float* x = a.f.x;
    float *spec = a.spec, *spread = a.spread;
    long long r0 = (long long)blockIdx.x * kQueryRows;          // first row in those arrays
    if constexpr (std::is_same_v<Args, QueryPieces>) {
        const int rows = a.per * kQueryRows;
        spec = reinterpret_cast<float*>(a.slot[blockIdx.x / a.per]);
        spread = spec + (long long)rows * a.nout;
        x = spread + rows;
        r0 = (long long)(blockIdx.x % a.per) * kQueryRows;
    }
    const uint32_t mask = (lane & 31) < left ? 0xFFFFFFFFu : 0u;
    const float* p = a.f.p[g];
    const v8bf* wf = reinterpret_cast<const v8bf*>(a.f.wf[g]);
    const int T = a.nout / 32, nl = a.f.nhh + 1;          // output tiles, hidden layers
    // first fragment of a layer's tile; layer nl is the output layer
    auto frags = [&](int l, int tile) -> const v8bf* {
        return wf + (H * kFusedKin + (long long)(l - 1) * H * H) / 8 + (long long)tile * KSH * 64;
    };
    v8bf w0[1] = {wf[w * 64 + lane]}, wq[KSH];
    const v8bf* next = frags(1, nl > 1 || w < T ? w : 0);
#pragma unroll
    for (int i = 0; i < KSH; ++i) wq[i] = next[i * 64 + lane];
    for (int i = tid; i < kQueryRows * kFusedKin; i += 2 * H) {
        const int r = i / kFusedKin, c = i % kFusedKin;
        const float v = (r < left && c < a.f.nin) ? x[(r0 + r) * a.f.nin + c] : 0.0f;
        act[g][0][r * LD + c] = bf16_rne(v);
    }
    v16f z;
    auto bias = [&](int l) {
#pragma unroll
        for (int j = 0; j < 16; ++j) z[j] = p[a.f.boff[l] + 32 * w + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3)];
    };
    auto put = [&](uint16_t* to) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = silu(z[j]);
        rows_put<LD>(to, v, mask, w, lane);
    };
    bias(0);
    __syncthreads();
    rows_mma<LD, 1, 0>(act[g][0], w0, z, (const v8bf*)nullptr, lane);
    put(act[g][1]);
    int cur = 1;
    for (int l = 1; l < nl; ++l) {
        bias(l);
        __syncthreads();
        rows_mma<LD, KSH, KSH>(act[g][cur], wq, z, frags(l + 1, l + 1 < nl || w < T ? w : 0), lane);
        put(act[g][cur ^ 1]);
        cur ^= 1;
    }
    if (w < T) bias(nl);
    __syncthreads();
    if (w < T) {
        rows_mma<LD, KSH, 0>(act[g][cur], wq, z, (const v8bf*)nullptr, lane);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(&y[g][(lane & 31) * LY + 32 * w + 8 * q + 4 * (lane >> 5)]) =
                float4{z[4 * q], z[4 * q + 1], z[4 * q + 2], z[4 * q + 3]};
    }
    __syncthreads();
    // ensemble_kernel on the outputs in LDS: 16 lanes per row
    const int l16 = threadIdx.x & 15;
    const float inv = 1.0f / (float)a.members;
    for (int r = threadIdx.x >> 4; r < kQueryRows && r < left; r += blockDim.x >> 4) {
        float dist = 0.0f;
        for (int c = 4 * l16; c < a.nout; c += 64) {
            float4 yv[M];
#pragma unroll
            for (int i = 0; i < M; ++i)
                if (i < a.members) yv[i] = *reinterpret_cast<const float4*>(&y[i][r * LY + c]);
            *reinterpret_cast<float4*>(spec + (r0 + r) * a.nout + c) = ensemble_columns<M>(yv, a.members, a.floor, inv, dist);
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) dist += __shfl_xor(dist, o, 16);
        if (l16 == 0) spread[r0 + r] = dist * inv;
    }
}

}  // namespace mlp
}  // namespace sp
