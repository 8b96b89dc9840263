// sp_sort.hip -- spatial ordering of the particle arrays.
//
// The mover hands out particles in array order, so the particles in flight at
// any moment are a window of consecutive indices.  Ordering the arrays by a
// Morton key of coarse grid blocks makes that window a compact region of the
// grid whose field records stay resident in L2/MALL, instead of random cells
// all over the snapshot.  The order never changes a result: every particle's
// increments are keyed on its own identity.
//
// Stable LSD radix sort of (key, index) pairs, 6-bit digits: per-tile digit
// histograms, one scan of each digit's row of the tile table, and a stable
// scatter in which each wave ranks equal digits of its 512 particles by
// ballots.  The permutation then moves whole particles: the arrays are first
// packed, in the old order, into rows in the spare buffer set (64 + 40 + 2
// bytes, as much as the arrays take), and the rows are read in the new order
// and spread over the arrays.  A particle's 106 bytes then come from three
// places; gathered array by array they came from 18, and of a freshly injected
// population, whose order is random in space, each 8 bytes cost a 64-byte
// sector (2e7 particles: 8.2 ms, now 1.0 + 1.6 ms; the whole sort 9.2 -> 3.1).
#include "sp_device.h"
#include "sp_particles.h"

namespace sp {

namespace {

constexpr int kBlock = 256;
constexpr int kTile = kBlock * kTileItems;
constexpr int kWaveItems = kTile / (kBlock / kWave);   // consecutive particles of one wave
constexpr int kDigits = 1 << kSortDigitBits;
static_assert(kDigits == kWave, "one lane per digit");
constexpr int kScanBlock = 1024;

__device__ __forceinline__ uint32_t spread2(uint32_t v) {  // 16 bits -> even bits
    v &= 0xFFFFu;
    v = (v | (v << 8)) & 0x00FF00FFu;
    v = (v | (v << 4)) & 0x0F0F0F0Fu;
    v = (v | (v << 2)) & 0x33333333u;
    v = (v | (v << 1)) & 0x55555555u;
    return v;
}

__device__ __forceinline__ uint32_t spread3(uint32_t v) {  // 10 bits -> every third bit
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t block_of(double pos, double lo, double inv_d, int ncell, int shift) {
    double c = floor((pos - lo) * inv_d);
    c = fmin(fmax(c, 0.0), (double)(ncell - 1));
    return (uint32_t)c >> shift;
}

__device__ __forceinline__ uint32_t sort_key(const SortArgs& sa, double x, double y, double z, double rdt) {
    const uint32_t bx = block_of(x, sa.xmin, sa.idx, sa.nx, sa.shift);
    const uint32_t by = block_of(y, sa.ymin, sa.idy, sa.ny, sa.shift);
    uint32_t k;
    if (sa.ndim == 3) {
        const uint32_t bz = block_of(z, sa.zmin, sa.idz, sa.nz, sa.shift);
        k = spread3(bx) | (spread3(by) << 1) | (spread3(bz) << 2);
    } else {
        k = spread2(bx) | (spread2(by) << 1);
    }
    if (sa.done_bit >= 0 && !(rdt > 0.0)) k |= 1u << sa.done_bit;
    return k;
}

// Particle rows in a spare buffer set of capacity cap: 64 bytes (x, y, z, p,
// v, mu, w, t), 40 bytes (dt, rdt and the six 32-bit members) and 2 bytes
// (split_times, count_flag) per particle, each kind contiguous.
struct Rows {
    char* base;
    long long cap;
    __device__ double2* a(long long i) const { return reinterpret_cast<double2*>(base + 64 * i); }
    __device__ uint2* b(long long i) const { return reinterpret_cast<uint2*>(base + 64 * cap + 40 * i); }
    __device__ uint16_t* c(long long i) const { return reinterpret_cast<uint16_t*>(base + 104 * cap + 2 * i); }
};

// Adds this block's digit counts of one pass to LDS and writes them to its
// tile's column of the digit-major table.
__device__ __forceinline__ void store_counts(const unsigned* h, long long ntiles, unsigned* hist) {
    if (threadIdx.x < kDigits) hist[(long long)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// Keys, the counts of the first digit, and the particle rows.
__global__ void __launch_bounds__(kBlock) pack_rows_kernel(Ptl P, long long n, SortArgs sa, Rows R,
                                                           uint32_t* key, long long ntiles,
                                                           unsigned* hist) {
    __shared__ unsigned h[kDigits];
    if (threadIdx.x < kDigits) h[threadIdx.x] = 0;
    __syncthreads();
    const long long t0 = (long long)blockIdx.x * kTile;
#pragma unroll 2
    for (int it = 0; it < kTileItems; ++it) {
        const long long i = t0 + (long long)it * kBlock + threadIdx.x;
        if (i >= n) break;
        const PtlRow r = load_row(P, i);
        const uint32_t k = sort_key(sa, r.x, r.y, r.z, r.rdt);
        key[i] = k;
        atomicAdd(&h[k & (kDigits - 1)], 1u);
        double2* a = R.a(i);
        a[0] = make_double2(r.x, r.y);
        a[1] = make_double2(r.z, r.p);
        a[2] = make_double2(r.v, r.mu);
        a[3] = make_double2(r.w, r.t);
        uint2* b = R.b(i);
        reinterpret_cast<double*>(b)[0] = r.dt;
        reinterpret_cast<double*>(b)[1] = r.rdt;
        b[2] = make_uint2((uint32_t)r.origin, (uint32_t)r.nsteps_tracked);
        b[3] = make_uint2((uint32_t)r.nsteps_pushed, (uint32_t)r.tag_injected);
        b[4] = make_uint2((uint32_t)r.tag_splitted, r.rng_step);
        *R.c(i) = (uint16_t)((uint8_t)r.split_times | ((uint32_t)(uint8_t)r.count_flag << 8));
    }
    __syncthreads();
    store_counts(h, ntiles, hist);
}

__global__ void __launch_bounds__(kBlock) digit_count_kernel(const uint32_t* key, long long n, int shift,
                                                             long long ntiles, unsigned* hist) {
    __shared__ unsigned h[kDigits];
    if (threadIdx.x < kDigits) h[threadIdx.x] = 0;
    __syncthreads();
    const long long t0 = (long long)blockIdx.x * kTile;
#pragma unroll
    for (int it = 0; it < kTileItems; ++it) {
        const long long i = t0 + (long long)it * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[(key[i] >> shift) & (kDigits - 1)], 1u);
    }
    __syncthreads();
    store_counts(h, ntiles, hist);
}

// Exclusive scan of each digit's row of tile counts (one block per digit) and
// the rows' totals; the scatter adds the totals of the lower digits.
__global__ void __launch_bounds__(kScanBlock) digit_scan_kernel(unsigned* hist, long long ntiles,
                                                                unsigned* totals) {
    constexpr int kItems = 4;
    __shared__ unsigned wsum[kScanBlock / kWave];
    unsigned* row = hist + (long long)blockIdx.x * ntiles;
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    unsigned carry = 0;
    for (long long b = 0; b < ntiles; b += kScanBlock * kItems) {
        const long long i = b + (long long)threadIdx.x * kItems;
        unsigned v[kItems], sum = 0;
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            v[k] = i + k < ntiles ? row[i + k] : 0u;
            sum += v[k];
        }
        unsigned x = sum;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const unsigned y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        if (lane == kWave - 1) wsum[wv] = x;
        __syncthreads();
        unsigned o = carry + x - sum;
#pragma unroll
        for (int k = 0; k < kScanBlock / kWave; ++k) {
            const unsigned t = wsum[k];
            if (k < wv) o += t;
            carry += t;
        }
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            if (i + k < ntiles) row[i + k] = o;
            o += v[k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Stable scatter of one digit.  iin is the identity in the first pass
// (nullptr); the last pass writes no keys (kout nullptr).
__global__ void __launch_bounds__(kBlock) digit_scatter_kernel(const uint32_t* kin, const uint32_t* iin,
                                                               uint32_t* kout, uint32_t* iout,
                                                               long long n, int shift,
                                                               long long ntiles, const unsigned* off,
                                                               const unsigned* totals) {
    __shared__ unsigned run[kBlock / kWave][kDigits];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    run[wv][lane] = 0;
    __syncthreads();
    const long long i0 = (long long)blockIdx.x * kTile + wv * kWaveItems + lane;
    uint32_t key[kTileItems];
#pragma unroll
    for (int it = 0; it < kTileItems; ++it) {
        const long long i = i0 + it * kWave;
        key[it] = i < n ? kin[i] : 0u;
        if (i < n) atomicAdd(&run[wv][(key[it] >> shift) & (kDigits - 1)], 1u);
    }
    __syncthreads();
    // lane d of every wave: where the wave's particles of digit d begin
    unsigned tot = totals[lane], x = tot;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    unsigned base = x - tot + off[(long long)lane * ntiles + blockIdx.x];
    for (int q = 0; q < wv; ++q) base += run[q][lane];
    __syncthreads();
    run[wv][lane] = base;
    const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int it = 0; it < kTileItems; ++it) {
        const long long i = i0 + it * kWave;
        const bool valid = i < n;
        const int d = (int)((key[it] >> shift) & (kDigits - 1));
        unsigned long long same = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kSortDigitBits; ++b) {
            const unsigned long long m = __ballot((d >> b) & 1);
            same &= ((d >> b) & 1) ? m : ~m;
        }
        // the wave's own counters: its LDS accesses are executed in order
        asm volatile("" ::: "memory");
        const unsigned o = run[wv][d] + (unsigned)__popcll(same & lt);
        asm volatile("" ::: "memory");
        if (valid) {
            if ((same & lt) == 0ull) run[wv][d] = o + (unsigned)__popcll(same);
            if (kout) kout[o] = key[it];
            iout[o] = iin ? iin[i] : (uint32_t)i;
        }
    }
}

// Arrays from the rows, in the order of perm.
__global__ void __launch_bounds__(kBlock) unpack_rows_kernel(Rows R, Ptl D, long long n, const uint32_t* perm) {
    const long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const long long i = perm[j];
    const double2* a = R.a(i);
    const uint2* b = R.b(i);
    const double2 a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
    const double dt = reinterpret_cast<const double*>(b)[0], rdt = reinterpret_cast<const double*>(b)[1];
    const uint2 b2 = b[2], b3 = b[3], b4 = b[4];
    const uint16_t c = *R.c(i);
    const PtlRow r{a0.x, a0.y, a1.x, a1.y, a2.x, a2.y, a3.x, a3.y, dt, rdt,
                   (int8_t)(c & 0xFF), (int8_t)(c >> 8), (int32_t)b2.x, (int32_t)b2.y, (int32_t)b3.x,
                   (int32_t)b3.y, (int32_t)b4.x, b4.y};
    store_row<true>(D, j, r);
}

}  // namespace

hipError_t launch_digit_order(const uint32_t* digit, long long n, uint32_t* order, unsigned* hist,
                              hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const long long ntiles = num_tiles(n);
    unsigned* totals = hist + kDigits * ntiles;
    hipLaunchKernelGGL(digit_count_kernel, dim3((unsigned)ntiles), dim3(kBlock), 0, s, digit, n, 0, ntiles, hist);
    hipLaunchKernelGGL(digit_scan_kernel, dim3(kDigits), dim3(kScanBlock), 0, s, hist, ntiles, totals);
    hipLaunchKernelGGL(digit_scatter_kernel, dim3((unsigned)ntiles), dim3(kBlock), 0, s, digit,
                       (const uint32_t*)nullptr, (uint32_t*)nullptr, order, n, 0, ntiles, hist, totals);
    return hipGetLastError();
}

hipError_t launch_spatial_sort(const Ptl& P, const PtlBase& spare, long long n, const SortArgs& sa,
                               uint32_t* keyA, uint32_t* idxA, uint32_t* keyB, uint32_t* idxB,
                               unsigned* hist, hipStream_t s) {
    if (n <= 1) return hipSuccess;
    const unsigned grid = (unsigned)((n + kBlock - 1) / kBlock);
    const long long ntiles = num_tiles(n);
    unsigned* totals = hist + kDigits * ntiles;
    const Rows rows{spare.base, spare.cap};
    hipLaunchKernelGGL(pack_rows_kernel, dim3((unsigned)ntiles), dim3(kBlock), 0, s, P, n, sa, rows, keyA,
                       ntiles, hist);
    for (int pass = 0; pass < sa.passes; ++pass) {
        const int shift = kSortDigitBits * pass;
        if (pass > 0)
            hipLaunchKernelGGL(digit_count_kernel, dim3((unsigned)ntiles), dim3(kBlock), 0, s, keyA, n,
                               shift, ntiles, hist);
        hipLaunchKernelGGL(digit_scan_kernel, dim3(kDigits), dim3(kScanBlock), 0, s, hist, ntiles, totals);
        hipLaunchKernelGGL(digit_scatter_kernel, dim3((unsigned)ntiles), dim3(kBlock), 0, s, keyA,
                           pass > 0 ? idxA : nullptr, pass + 1 < sa.passes ? keyB : nullptr, idxB, n, shift,
                           ntiles, hist, totals);
        uint32_t* t = keyA; keyA = keyB; keyB = t;
        t = idxA; idxA = idxB; idxB = t;
    }
    hipLaunchKernelGGL(unpack_rows_kernel, dim3(grid), dim3(kBlock), 0, s, rows, P, n, idxA);
    return hipGetLastError();
}

}  // namespace sp
