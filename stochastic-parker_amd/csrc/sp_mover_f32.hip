// sp_mover_f32.hip -- mover and single-step kernels with FP32 gather and
// coefficients, FP64 position / momentum / time accumulators.
#include "sp_mover_impl.h"
#include "sp_phys_f32.h"

namespace sp {

// FP32 gather and coefficients; one or two particles per lane, each with its
// own copy of the per-particle diffusion parameters (KF).  Steps without
// momentum diffusion gather from compact records (2D: FP32 cell coefficient
// records, or FP16-gradient x-pair records when HALF; 3D: bricked node
// records, FP16 values when HALF), those with it from the node records that
// carry its slots.  Configurations marked FX_LEAN get their own kernels.
template <bool HALF>
struct PolicyF32Base {
    static constexpr int kMaxPPL = 2;
    static constexpr bool kThreeWave2D = true;
    static constexpr bool kLean = true;
    using Var = f32::KF;
    __device__ __forceinline__ static Var var_of(const MoverParams& m) { return f32::kf_of(m); }
    __device__ __forceinline__ static void set_var(MoverParams&, Var& v, const KappaVar& kv) {
        v = f32::kf_of(kv);
    }
    // Whether a wave skips the momentum floor's selects by a branch, and whether a
    // lane keeps the particle's Philox words or its tags alone: what a branch and
    // two registers cost differs with how full the kernel's registers are.
    // Mover time of an interval (4e6 particles on 1024^2, 1.5e6 on 96^3) with the
    // branch / without: 2D FP32 7.45 / 7.53 ms, with acceleration region 7.95 / 8.23,
    // two frames 14.38 / 14.57, two particles a lane 14.5 / 14.9 (FP16 gradients 10.4 /
    // 11.6); with kappa's B dependence 9.62 / 9.44, two frames 17.1 / 16.96, NLGC 29.7 /
    // 28.8; FP16 gradients one frame 7.0 / 6.84, with B dependence 9.5 / 9.16; 3D 41.8 /
    // 41.0, with momentum diffusion 842 / 877.  The words / the tags: 2D FP32 7.45 / 7.50,
    // NLGC 28.8 / 27.65; FP16 gradients one frame 6.84 / 6.77 (1e5 particles on 512^2,
    // eleven intervals 32.3 / 30.2), with B dependence 9.16 / 9.31, NLGC 29.9 / 30.7.
    template <int NDIM, bool TI, int FX, int PPL>
    static constexpr bool kFloorBranch =
        (FX & FX_DPP) != 0 || (NDIM == 2 && (FX & (FX_LEAN | FX_NLGC)) == FX_LEAN && !(HALF && !TI && PPL == 1));
    template <int NDIM, bool TI, int FX>
    static constexpr bool kTags = NDIM == 2 && !TI &&
                                  (HALF ? (FX & (FX_LEAN | FX_NLGC)) == FX_LEAN : (FX & FX_NLGC) != 0);
    template <int NDIM, bool TI, int FX>
    using Rng = std::conditional_t<kTags<NDIM, TI, FX>, PhiloxTags, PhiloxPtl>;
    template <int NDIM, bool TI, int FX, int PPL>
    using Cache = f32::GatherCache<NDIM, TI, HALF, (FX & FX_DPP) != 0, PPL>;
    template <int NDIM, bool TI, int FX, class GC>
    __device__ __forceinline__ static void step(const MoverParams& m, const Var& kf, State& s,
                                                bool fixed, const Rng<NDIM, TI, FX>& rng, uint32_t rstep,
                                                double d[4], GC& gc) {
        float r[4];
        f32::step_rands(m, rng, rstep, r);
        f32::gather_kappa_push<NDIM, TI, FX, HALF, kFloorBranch<NDIM, TI, FX, 1>>(m, kf, s, fixed, r, d, gc);
    }
    // PPL particles: the Philox blocks, the gathers and the steps of all
    // slots in one block, for the scheduler to interleave
    template <int NDIM, bool TI, int FX, int PPL>
    __device__ __forceinline__ static void step_n(const MoverParams& m, const Var* kf, State* s,
                                                  const bool* fixed, const Slot<Rng<NDIM, TI, FX>>* sl,
                                                  double (*d)[4]) {
        float r[PPL][4];
#pragma unroll
        for (int k = 0; k < PPL; ++k) f32::step_rands(m, sl[k].rng, sl[k].rstep, r[k]);
        Cache<NDIM, TI, FX, PPL> none;   // no records kept across steps at PPL > 1
#pragma unroll
        for (int k = 0; k < PPL; ++k)
            f32::gather_kappa_push<NDIM, TI, FX, HALF, kFloorBranch<NDIM, TI, FX, PPL>>(m, kf[k], s[k], fixed[k], r[k], d[k], none);
    }
    template <int NDIM, bool TI, int FX>
    __device__ __forceinline__ static void step_given(const MoverParams& m, const Var& kf,
                                                      State& s, bool fixed, const double* r,
                                                      double d[4]) {
        const float rf[4] = {(float)r[0], (float)r[1], (float)r[2], (float)r[3]};
        Cache<NDIM, TI, FX, 2> none;   // one step: nothing to keep
        f32::gather_kappa_push<NDIM, TI, FX, HALF, false>(m, kf, s, fixed, rf, d, none);
    }
};

// FP32 arithmetic on FP32 records.
struct PolicyF32 : PolicyF32Base<false> {
    static constexpr bool kWaits = true;
    static constexpr bool kOnly3D = false;
    static constexpr bool kDpp = true;
};

// FP32 arithmetic on x-pair records with FP16 gradients.
struct PolicyF32H : PolicyF32Base<true> {
    static constexpr bool kWaits = false;   // 3 % slower
    static constexpr bool kOnly3D = false;
    static constexpr bool kDpp = false;   // no momentum-diffusion slots in these records
};

int mover_blocks_per_cu_f32h(int ndim, bool ti, int fx, int ppl) {
    return mover_occupancy<PolicyF32H>(ndim, ti, fx, ppl);
}

hipError_t launch_mover_f32h(const MoverParams& m, bool ti, int fx, int ndim, int ppl, int grid,
                             hipStream_t s) {
    return launch_mover<PolicyF32H>(m, ti, fx, ndim, ppl, grid, s);
}

hipError_t launch_step_once_f32h(const MoverParams& m, bool ti, int fx, int ndim, const StepRows& r,
                                 hipStream_t s) {
    return launch_step_once<PolicyF32H>(m, ti, fx, ndim, r, s);
}

int mover_blocks_per_cu_f32(int ndim, bool ti, int fx, int ppl) {
    return mover_occupancy<PolicyF32>(ndim, ti, fx, ppl);
}

hipError_t launch_mover_f32(const MoverParams& m, bool ti, int fx, int ndim, int ppl, int grid,
                            hipStream_t s) {
    return launch_mover<PolicyF32>(m, ti, fx, ndim, ppl, grid, s);
}

hipError_t launch_step_once_f32(const MoverParams& m, bool ti, int fx, int ndim, const StepRows& r,
                                hipStream_t s) {
    return launch_step_once<PolicyF32>(m, ti, fx, ndim, r, s);
}

hipError_t launch_order_f32(const MoverParams& m, bool ti, int fx, int ndim, uint32_t* digit, float* counts,
                            hipStream_t s) {
    return launch_order<PolicyF32>(m, ti, fx, ndim, digit, counts, s);
}

hipError_t launch_order_f32h(const MoverParams& m, bool ti, int fx, int ndim, uint32_t* digit, float* counts,
                            hipStream_t s) {
    return launch_order<PolicyF32H>(m, ti, fx, ndim, digit, counts, s);
}

}  // namespace sp
