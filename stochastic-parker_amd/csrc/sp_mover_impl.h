// sp_mover_impl.h -- the persistent particle-mover kernel.
//
// One lane owns one particle at a time and walks it through the reference's
// per-particle interval loop (particle_mover_one_cycle,
// particle_module.f90:1561-1830): the fine-step loop, the adaptive steps, the
// interval-end undo + fixed-dt redo, the slack-bound boundary checks and,
// when the particle is done, particle_mover's exact-bounds pass
// (:1959-1968).  Each loop iteration is one particle-step for every lane
// that has one to take; a lane whose particle finished takes the next
// particle index from a global counter (one atomic per wave and refill), so
// differing step counts never idle a wave.  Random increments come from
// Philox keyed on the particle's (tag_injected, tag_splitted, rng_step), so
// results do not depend on which lane or wave pushes a particle.
//
// The reference loop is flattened into a per-lane action chosen at the top of
// each iteration, so the boundary check, the step and the store each appear
// once in the kernel body:
//   pending PRE   after a load: safety check, finish if out of the box
//   inner loop    t - t0 < target: boundary check, then an adaptive step
//   overshoot     t - t0 > target: undo the last step, fixed-dt redo step;
//                 the redo's boundary check and the advance of the target run
//                 at the top of the next iteration (pending REDO)
//   otherwise     advance the target (next fine step, or done)
//
// With a step budget, a particle that has taken that many steps in this
// launch stops at the top of its inner loop (before the boundary check of its
// next step): its state and interval target are stored and the launch counts
// it as paused.  The next launch resumes it at the same point; the increments
// depend only on the particle's counter, so pausing never changes a result.
#pragma once

#include "sp_device.h"

#include <type_traits>

namespace sp {

enum : int { PEND_NONE = 0, PEND_PRE = 1, PEND_REDO = 2 };
enum : int { ACT_NONE = 0, ACT_PRE = 1, ACT_PUSH = 2, ACT_PUSH_FIXED = 3, ACT_ADVANCE = 4,
              ACT_PAUSE = 5 };

// Keeps a uniform floating-point value in vector registers: the hot loop
// reads dozens of FP64/FP32 constants, more than the scalar register file
// holds, and constants spilled from scalar registers cost one v_readlane per
// 32-bit half at every use.  An operand already in a VGPR costs nothing.
template <class T>
__device__ __forceinline__ void pin_vgpr(T& v) {
    asm volatile("" : "+v"(v));
}

__device__ __forceinline__ void pin_constants(MoverParams& m) {
    pin_vgpr(m.t0); pin_vgpr(m.dtf); pin_vgpr(m.dt_fine); pin_vgpr(m.dt_limit);
    pin_vgpr(m.xmin); pin_vgpr(m.ymin); pin_vgpr(m.zmin);
    pin_vgpr(m.dx); pin_vgpr(m.dy); pin_vgpr(m.dz);
    pin_vgpr(m.idx); pin_vgpr(m.idy); pin_vgpr(m.idz);
    for (int k = 0; k < 3; ++k) {
        pin_vgpr(m.slo[k]); pin_vgpr(m.shi[k]); pin_vgpr(m.elo[k]); pin_vgpr(m.ehi[k]);
    }
    pin_vgpr(m.p0); pin_vgpr(m.p_floor);
    pin_vgpr(m.kpara0); pin_vgpr(m.kret); pin_vgpr(m.pindex); pin_vgpr(m.gamma_m2);
    pin_vgpr(m.vdp_pre); pin_vgpr(m.d1p0); pin_vgpr(m.d2p02);
    pin_vgpr(m.half_min); pin_vgpr(m.inv_dtf);
    pin_vgpr(m.dt_min); pin_vgpr(m.dt_max);
    pin_vgpr(m.f_kpara0); pin_vgpr(m.f_kret); pin_vgpr(m.f_pindex); pin_vgpr(m.f_gm2);
    pin_vgpr(m.f_vdp_pre); pin_vgpr(m.f_d1p0); pin_vgpr(m.f_d2p02);
    pin_vgpr(m.f_half_dx); pin_vgpr(m.f_half_dy); pin_vgpr(m.f_half_dz);
    pin_vgpr(m.f_dt_min); pin_vgpr(m.f_dt_max);
    pin_vgpr(m.inv_p0);
    for (int k = 0; k < 6; ++k) pin_vgpr(m.acc_region[k]);
    pin_vgpr(m.lx); pin_vgpr(m.ly); pin_vgpr(m.lz);
}

// Per-slot state of the particle a lane is pushing.
template <class Rng>
struct Slot {
    long long idx;                // particle index (-1: none)
    State s;
    double w, dtarget, dt_old;
    double dl[4];                 // the last step's increments (for the undo)
    int cf, nsp, pending;
    Rng rng;
    uint32_t rstep;
    unsigned ksteps;              // steps of this particle in this launch
    bool resumed;
};

// At most two resident waves per SIMD: the mover runs one or two 256-lane
// blocks per CU (fewer particles in flight keep their field records in L2),
// so the compiler may spend registers on keeping the gather's loads in flight
// rather than on a higher occupancy that is never used (3D: +13 %).
//
// PPL particles per lane: each lane carries PPL independent particles
// ("slots") through the loop above.  Their steps are computed in one
// straight-line block (every slot steps, a slot that has no step to take
// discards its result), so the compiler can interleave two particles' loads,
// Philox rounds and arithmetic and fill the latency one particle alone leaves
// idle.  Every slot draws its increments from its own particle's counter, so
// the particles per lane never change a result.  Two 2D particles per lane
// fit the two-wave register budget (233 VGPRs) once the constants are left to
// the compiler; two 3D particles need the one-wave budget.
template <int NDIM, int PPL>
constexpr bool kTwoWavePair = NDIM == 2 && PPL == 2;
// The one-frame 2D step of the FP32 movers with one particle per lane runs
// three waves per SIMD (129-168 VGPRs, the constants left to the compiler):
// with most gathers served by the register cache, a third wave hides more of
// the step's latency than pinning every constant saves (-9 % kernel time
// against two pinned waves).  Two-frame steps would spill at that budget.
template <class Pol, int NDIM, bool TINTERP, int PPL>
constexpr bool kThreeWave = Pol::kThreeWave2D && NDIM == 2 && !TINTERP && PPL == 1;

// ORDER: the parts hand out particles in the order of m.order (a kernel of its
// own: the test and the pointer in the other kernels cost them 2-3 %).
// WAIT: the wave's other work (taking a particle, landing on a target time,
// leaving) comes to one lane in most iterations and costs the whole wave its
// instructions.  So these lanes wait until together they have lost kServeLanes
// iterations, or are an eighth of the lanes that step (64 variants, 3.8e6
// particles on 512^2, two intervals: at once 25.4 ms, 2 lane-iterations 23.5, 4
// 22.7, 8 22.0, 16 21.6).  A kernel of its own, for lanes that take many
// particles in turn: where they take a few, the last ones' chains of steps are
// drawn out (-15 %), and the votes alone cost 5 %.
constexpr int kServeLanes = 16;
template <class Pol, int NDIM, bool TINTERP, int FX, int PPL, bool ORDER = false, bool WAIT = false>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(kThreeWave<Pol, NDIM, TINTERP, PPL> ? 3 : (kTwoWavePair<NDIM, PPL> ? 2 : 1),
                                   kThreeWave<Pol, NDIM, TINTERP, PPL> ? 3 : 2)))
mover_kernel(MoverParams m0) {
    static_assert(PPL >= 1 && PPL <= Pol::kMaxPPL, "particles per lane of this policy");
    constexpr int kServe = WAIT ? kServeLanes : 0;
    static_assert(!WAIT || PPL == 1, "one slot waits");
    MoverParams m = m0;
    // within the two-wave register budget the constants fit in VGPRs for 2D
    // and 3D alike (2D: +5 %, 3D: +1 %)
    if constexpr (!kTwoWavePair<NDIM, PPL> && !kThreeWave<Pol, NDIM, TINTERP, PPL>) pin_constants(m);
    // at three waves only the FP64 constants of every iteration fit (interval
    // times, the interpolation origin and scale, the slack bounds): -6 to -9 %
    // kernel time; the acceleration-gated NLGC step has no room for them
    constexpr bool kPinHot = kThreeWave<Pol, NDIM, TINTERP, PPL> &&
                             !((FX & FX_ACC) != 0 && (FX & FX_NLGC) != 0);
    if constexpr (kPinHot) {
        pin_vgpr(m.t0); pin_vgpr(m.dt_fine); pin_vgpr(m.dt_limit);
        pin_vgpr(m.xmin); pin_vgpr(m.ymin); pin_vgpr(m.idx); pin_vgpr(m.idy);
        pin_vgpr(m.slo[0]); pin_vgpr(m.slo[1]); pin_vgpr(m.shi[0]); pin_vgpr(m.shi[1]);
    }
    const int lane = threadIdx.x & (kWave - 1);
    double* const px = m.P.d(PD_X);
    double* const py = m.P.d(PD_Y);
    double* const pz = m.P.d(PD_Z);
    double* const pp = m.P.d(PD_P);
    double* const pt = m.P.d(PD_T);
    double* const pdt = m.P.d(PD_DT);
    int8_t* const pflag = m.P.b(PB_FLAG);
    int32_t* const ppushed = m.P.i(PI_PUSHED);
    uint32_t* const prstep = reinterpret_cast<uint32_t*>(m.P.i(PI_RSTEP));
    double* const prdt = m.P.d(PD_RDT);

    bool exhausted = false;
    // start on this die's part of the range, then help the other parts
    int part = (int)(xcc_id() % (unsigned)kParts), parts_done = 0;
    using Rng = typename Pol::template Rng<NDIM, TINTERP, FX>;
    Slot<Rng> sl[PPL];
    typename Pol::Var var[PPL];
    typename Pol::template Cache<NDIM, TINTERP, FX, PPL> gc;   // slot 0's last records
    gc.invalidate();
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
        sl[k].idx = -1;
        sl[k].s = State{0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        sl[k].w = sl[k].dtarget = sl[k].dt_old = 0.0;
        sl[k].dl[0] = sl[k].dl[1] = sl[k].dl[2] = sl[k].dl[3] = 0.0;
        sl[k].cf = sl[k].nsp = 0;
        sl[k].pending = PEND_NONE;
        sl[k].rng = Rng{};
        sl[k].rstep = 0u;
        sl[k].ksteps = 0u;
        sl[k].resumed = false;
        var[k] = Pol::var_of(m);
    }
    unsigned long long my_steps = 0, my_paused = 0;
    bool serve = true;            // this iteration does the wave's other work (kServeLanes)
    int waited = 0;               // lane-iterations lost since it was last done

    while (true) {
        // ---- refill idle slots (wave-aggregated work fetch, one slot index at a time) ----
#pragma unroll
        for (int k = 0; k < PPL; ++k) {
            if (kServe > 0 && !serve) break;
            Slot<Rng>& q = sl[k];
            const bool need = q.idx < 0 && !exhausted;
            const unsigned long long need_mask = __builtin_amdgcn_ballot_w64(need);
            if (!need_mask) continue;
            const int leader = __ffsll((unsigned long long)need_mask) - 1;
            const unsigned long long cnt = (unsigned long long)__popcll(need_mask);
            unsigned long long base = 0;
            if (lane == leader) base = atomicAdd(&m.ctr->part[part * kPartStride], cnt);
            base = __shfl(base, leader);
            const long long pb = (long long)part * m.part_len;
            const long long pe = pb + m.part_len < m.n ? pb + m.part_len : m.n;
            if (pb + (long long)(base + cnt) >= pe) {
                // this part is used up: move on; after all parts, stop fetching
                part = (part + 1) % kParts;
                if (++parts_done == kParts) exhausted = true;
            }
            if (need) {
                long long j =
                    pb + (long long)(base + (unsigned long long)__popcll(need_mask & ((1ull << lane) - 1ull)));
                if (j < pe) {
                    if constexpr (ORDER) j = m0.order[j];
                    q.idx = j;
                    if (k == 0) gc.invalidate();
                    q.s.x = px[j];
                    q.s.y = py[j];
                    q.s.z = pz[j];
                    q.s.p = pp[j];
                    q.s.t = pt[j];
                    q.s.dt = pdt[j];
                    if constexpr ((FX & FX_NLGC) != 0) q.s.mu = m.P.d(PD_MU)[j];
                    q.w = m.P.d(PD_W)[j];
                    q.cf = pflag[j];
                    q.nsp = ppushed[j];
                    if (m0.nvar > 0) {
                        // this particle's variant: its diffusion parameters
                        int v = m.P.i(PI_ORIGIN)[j];
                        v = v < 0 ? 0 : (v >= m0.nvar ? m0.nvar - 1 : v);
                        Pol::set_var(m, var[k], m0.var[v]);
                    }
                    philox_take(q.rng, (uint32_t)m.P.i(PI_TAGI)[j], (uint32_t)m.P.i(PI_TAGS)[j], m.stream,
                                m.key0, m.key1);
                    q.rstep = prstep[j];
                    q.dl[0] = q.dl[1] = q.dl[2] = q.dl[3] = 0.0;
                    q.ksteps = 0;
                    const double rd = prdt[j];
                    q.resumed = rd > 0.0;
                    if (q.resumed) {
                        // paused at the top of the inner loop by an earlier launch
                        q.dtarget = rd;
                        q.pending = PEND_NONE;
                    } else {
                        // target time from the particle's own time stamp (:1570-1578)
                        const double stp = ceil((q.s.t - m.t0) / m.dt_fine);
                        if (stp <= 0.0) q.dtarget = m.dt_fine; else q.dtarget = stp * m.dt_fine;
                        if (q.dtarget > m.dtf) q.dtarget = m.dtf;
                        q.pending = PEND_PRE;
                    }
                }
            }
        }
        bool busy = false;
#pragma unroll
        for (int k = 0; k < PPL; ++k) busy = busy || sl[k].idx >= 0;
        if (__builtin_amdgcn_ballot_w64(busy || !exhausted) == 0ull) break;

        bool do_push[PPL], fixed[PPL];
#pragma unroll
        for (int k = 0; k < PPL; ++k) {
            Slot<Rng>& q = sl[k];
            do_push[k] = false;
            fixed[k] = false;
            if (q.idx < 0) continue;
            // ---- the common case: an inner-loop step of a particle inside the
            // slack bounds with a non-negative momentum, for which the action
            // choice, the check and the transitions below reduce to "push"
            // with nothing changed.  Tested with the same comparisons the
            // check makes, so NaN positions take this path as they pass there.
            {
                bool inside = !(q.s.p < 0.0) && !(q.s.x < m.slo[0]) && !(q.s.x > m.shi[0]) &&
                              !(q.s.y < m.slo[1]) && !(q.s.y > m.shi[1]);
                if (NDIM == 3) inside = inside && !(q.s.z < m.slo[2]) && !(q.s.z > m.shi[2]);
                const bool running = q.pending == PEND_NONE && (q.s.t - m.t0) < q.dtarget &&
                                     q.cf == SP_COUNT_FLAG_INBOX &&
                                     !(m.step_budget != 0u && q.ksteps >= m.step_budget);
                if (running && inside) {
                    do_push[k] = true;
                    continue;
                }
            }
            if (kServe > 0 && !serve) continue;
            // ---- choose this slot's action ----
            int act = ACT_NONE;
            bool need_bc = false;
            if (q.pending == PEND_PRE) {
                need_bc = true;  // safety check before the loop (:1581-1592)
                act = ACT_PRE;
            } else if (q.pending == PEND_REDO) {
                q.s.dt = q.dt_old;  // the redo step is done; restore dt, check, advance (:1804-1826)
                need_bc = true;
                act = ACT_ADVANCE;
            } else if ((q.s.t - m.t0) < q.dtarget && q.cf == SP_COUNT_FLAG_INBOX) {
                if (m.step_budget != 0u && q.ksteps >= m.step_budget) {
                    act = ACT_PAUSE;
                } else {
                    need_bc = true;  // top of the inner loop (:1600-1612)
                    act = ACT_PUSH;
                }
            } else if ((q.s.t - m.t0) > q.dtarget && q.cf == SP_COUNT_FLAG_INBOX) {
                // land exactly on the target time (:1707-1720)
                q.s.x = q.s.x - q.dl[0];
                q.s.y = q.s.y - q.dl[1];
                q.s.z = q.s.z - q.dl[2];
                q.s.p = q.s.p - q.dl[3];
                q.s.t = q.s.t - q.s.dt;
                q.dt_old = q.s.dt;
                q.s.dt = m.t0 + q.dtarget - q.s.t;
                if (q.s.dt > 0) {
                    q.nsp = q.nsp - 1;
                    act = ACT_PUSH_FIXED;
                } else {
                    q.s.dt = q.dt_old;
                    need_bc = true;
                    act = ACT_ADVANCE;
                }
            } else {
                act = ACT_ADVANCE;
            }
            q.pending = PEND_NONE;

            // ---- the slack-bound check: momentum sign first, then the faces ----
            if (need_bc) {
                if (q.s.p < 0.0 && q.cf == SP_COUNT_FLAG_INBOX) {
                    q.cf = SP_COUNT_FLAG_OTHERS;
                    atomicAdd(&m.ctr->negp_fx, weight_fx(q.w));
                } else {
                    const double lk = boundary_condition<NDIM>(m.flags, q.s.x, q.s.y, q.s.z, q.cf,
                                                               q.w, m.slo[0], m.slo[1], m.slo[2],
                                                               m.shi[0], m.shi[1], m.shi[2]);
                    if (lk != 0.0) atomicAdd(&m.ctr->leak_fx, weight_fx(lk));
                }
            }

            // ---- transitions ----
            bool fin = false;
            if (act == ACT_PUSH) {
                if (q.cf == SP_COUNT_FLAG_INBOX) do_push[k] = true;
                else fin = true;  // the inner loop exits and the outer loop ends on count_flag
            } else if (act == ACT_PUSH_FIXED) {
                do_push[k] = true;
                fixed[k] = true;
                q.pending = PEND_REDO;
            } else if (act == ACT_ADVANCE) {
                q.dtarget = q.dtarget + m.dt_fine;
                fin = !(q.dtarget < m.dt_limit) || q.cf != SP_COUNT_FLAG_INBOX;
            } else if (act == ACT_PRE) {
                fin = q.cf != SP_COUNT_FLAG_INBOX || !(q.dtarget < m.dt_limit);
            }
            const bool pause = act == ACT_PAUSE;
            if (fin || pause) {
                if (fin && q.cf == SP_COUNT_FLAG_INBOX) {
                    const double lk = boundary_condition<NDIM>(m.flags, q.s.x, q.s.y, q.s.z, q.cf,
                                                               q.w, m.elo[0], m.elo[1], m.elo[2],
                                                               m.ehi[0], m.ehi[1], m.ehi[2]);
                    if (lk != 0.0) atomicAdd(&m.ctr->leak_fx, weight_fx(lk));
                }
                const long long j = q.idx;
                if (pause) {
                    prdt[j] = q.dtarget;
                    ++my_paused;
                } else if (q.resumed) {
                    prdt[j] = 0.0;
                }
                px[j] = q.s.x;
                py[j] = q.s.y;
                pz[j] = q.s.z;
                pp[j] = q.s.p;
                pt[j] = q.s.t;
                pdt[j] = q.s.dt;
                pflag[j] = (int8_t)q.cf;
                ppushed[j] = q.nsp;
                prstep[j] = q.rstep;
                my_steps += q.ksteps;
                q.idx = -1;
            }
        }

        if constexpr (kServe > 0) {
            const unsigned long long wm = __builtin_amdgcn_ballot_w64(sl[0].idx >= 0 ? !do_push[0] : !exhausted);
            const unsigned long long pm = __builtin_amdgcn_ballot_w64(do_push[0]);
            if (serve) {
                waited = 0;
                serve = pm == 0ull;
            } else {
                waited += __popcll(wm);
                serve = waited >= kServe || __popcll(wm) * 8 >= __popcll(pm);
            }
        }

        // ---- one particle-step for every slot that takes one ----
        bool any_push = false;
#pragma unroll
        for (int k = 0; k < PPL; ++k) any_push = any_push || do_push[k];
        if (any_push) {
            if constexpr (PPL == 1) {
                Pol::template step<NDIM, TINTERP, FX>(m, var[0], sl[0].s, fixed[0], sl[0].rng,
                                                      sl[0].rstep, sl[0].dl, gc);
            } else {
                // every slot steps (one straight-line block); a slot without a
                // step to take keeps its state
                State ns[PPL];
                double nd[PPL][4];
#pragma unroll
                for (int k = 0; k < PPL; ++k) ns[k] = sl[k].s;
                Pol::template step_n<NDIM, TINTERP, FX, PPL>(m, var, ns, fixed, sl, nd);
#pragma unroll
                for (int k = 0; k < PPL; ++k) {
                    if (do_push[k]) {
                        sl[k].s = ns[k];
                        sl[k].dl[0] = nd[k][0];
                        sl[k].dl[1] = nd[k][1];
                        sl[k].dl[2] = nd[k][2];
                        sl[k].dl[3] = nd[k][3];
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < PPL; ++k) {
                if (!do_push[k]) continue;
                Slot<Rng>& q = sl[k];
                q.rstep += 1u;
                int v = q.nsp + 1;  // mod(nsteps_pushed + 1, nsteps_interval)
                if ((unsigned)v >= (unsigned)m.nsteps_interval) v %= m.nsteps_interval;
                q.nsp = v;
                ++q.ksteps;
            }
        }
    }

    // ---- per-wave step and pause totals: one atomic each per wave ----
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        my_steps += __shfl_xor(my_steps, off);
        my_paused += __shfl_xor(my_paused, off);
    }
    if (lane == 0 && my_steps) atomicAdd(&m.ctr->steps, my_steps);
    if (lane == 0 && my_paused) atomicAdd(&m.ctr->paused, my_paused);
}

// Single-step kernel: caller-supplied states and increments, rows of 6 and 4
// doubles, 64 rows per block, blockIdx.y the piece.  The rows pass through LDS so that each block
// reads and writes them in 16-byte pieces in order, once: they may lie in
// pinned host memory, where every piece is a transfer over PCIe.
constexpr int kStepRows = 64;
template <class Pol, int NDIM, bool TINTERP, int FX>
__global__ void __launch_bounds__(kStepRows) step_once_kernel(MoverParams m, StepRows sr) {
    __shared__ double2 st2[kStepRows * 3], rd2[kStepRows * 2];
    double* const st = reinterpret_cast<double*>(st2);
    double* const rd = reinterpret_cast<double*>(rd2);
    const long long i0 = (long long)blockIdx.x * kStepRows, i = i0 + threadIdx.x;
    const int pc = blockIdx.y;
    const long long left = sr.n[pc] - i0;
    if (left <= 0) return;
    const int rows = (int)(left < kStepRows ? left : kStepRows);
    double2* const gs = reinterpret_cast<double2*>(sr.state[pc] + 6 * i0);
    double2* const gd = reinterpret_cast<double2*>(sr.deltas[pc] + 4 * i0);
    const double2* const gr = reinterpret_cast<const double2*>(sr.rands[pc] + 4 * i0);
    const bool on = (int)threadIdx.x < rows;
    const int8_t fx = on ? sr.fixed[pc][i] : (int8_t)0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int q = k * kStepRows + threadIdx.x;
        if (q < 3 * rows) st2[q] = gs[q];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int q = k * kStepRows + threadIdx.x;
        if (q < 2 * rows) rd2[q] = gr[q];
    }
    __syncthreads();
    if (on) {
        double* const row = st + 6 * threadIdx.x;
        double* const r = rd + 4 * threadIdx.x;
        State s{row[0], row[1], row[2], row[3], row[4], row[5], 0.0};
        if constexpr ((FX & FX_NLGC) != 0) s.mu = m.P.d(PD_MU)[sr.row0[pc] + i];
        double d[4] = {0.0, 0.0, 0.0, 0.0};
        const double rr[4] = {r[0], r[1], r[2], r[3]};
        Pol::template step_given<NDIM, TINTERP, FX>(m, Pol::var_of(m), s, fx != 0, rr, d);
        row[0] = s.x;
        row[1] = s.y;
        row[2] = s.z;
        row[3] = s.p;
        row[4] = s.t;
        row[5] = s.dt;
        for (int c = 0; c < 4; ++c) r[c] = d[c];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int q = k * kStepRows + threadIdx.x;
        if (q < 3 * rows) gs[q] = st2[q];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int q = k * kStepRows + threadIdx.x;
        if (q < 2 * rows) gd[q] = rd2[q];
    }
}

// dt that particle i's first step would take, by a step with zero increments.
template <class Pol, int NDIM, bool TINTERP, int FX>
__device__ __forceinline__ double first_dt(MoverParams& m, long long i) {
    State s{m.P.d(PD_X)[i], m.P.d(PD_Y)[i], m.P.d(PD_Z)[i], m.P.d(PD_P)[i], m.P.d(PD_T)[i], m.P.d(PD_DT)[i], 0.0};
    if constexpr ((FX & FX_NLGC) != 0) s.mu = m.P.d(PD_MU)[i];
    typename Pol::Var var = Pol::var_of(m);
    if (m.nvar > 0) {
        const int v = m.P.i(PI_ORIGIN)[i];
        Pol::set_var(m, var, m.var[v < 0 ? 0 : (v >= m.nvar ? m.nvar - 1 : v)]);
    }
    const double still[4] = {0.0, 0.0, 0.0, 0.0};
    double d[4];
    Pol::template step_given<NDIM, TINTERP, FX>(m, var, s, false, still, d);
    return s.dt;
}

// Part of each particle (m.part_len) and the class of the step count that its
// first step's dt predicts, the larger counts first: classes a factor of two
// apart from the smallest count, dtf / dt_max, up.  digit = part * 8 + class.
constexpr int kOrderClasses = 8;
template <class Pol, int NDIM, bool TINTERP, int FX>
__global__ void __launch_bounds__(256) order_digit_kernel(MoverParams m, uint32_t* digit) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m.n) return;
    const double dt = first_dt<Pol, NDIM, TINTERP, FX>(m, i);
    const float c = __builtin_amdgcn_logf((float)m.dt_max / (float)dt);   // log2; a NaN goes last
    const int few = c > 0.0f ? (int)fminf(c, (float)(kOrderClasses - 1)) : 0;
    digit[i] = (uint32_t)(i / m.part_len) * kOrderClasses + (uint32_t)(kOrderClasses - 1 - few);
}

// Predicted step counts of kOrderSample particles spread over the population
// (at least as many), into pinned memory.
template <class Pol, int NDIM, bool TINTERP, int FX>
__global__ void __launch_bounds__(256) order_sample_kernel(MoverParams m, float* counts) {
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const double dt = first_dt<Pol, NDIM, TINTERP, FX>(m, t * (m.n / kOrderSample));
    counts[t] = (float)(m.dtf / dt);
}

template <int N, bool T, int X>
struct Variant {
    static constexpr int ndim = N;
    static constexpr bool ti = T;
    static constexpr int fx = X;
};

template <bool DPP, int N, int BASE, class F>
auto dispatch_acc(bool ti, int fx, F&& f) {
    const bool with_acc = (fx & FX_ACC) != 0;
    if (ti) return with_acc ? f(Variant<N, true, BASE | FX_ACC>{}) : f(Variant<N, true, BASE>{});
    return with_acc ? f(Variant<N, false, BASE | FX_ACC>{}) : f(Variant<N, false, BASE>{});
}

template <bool DPP, int N, int LEAN, class F>
auto dispatch_fx_base(bool ti, int fx, F&& f) {
    if constexpr (DPP) {
        if (fx & FX_DPP) {
            if (fx & FX_NLGC) return dispatch_acc<DPP, N, LEAN | FX_DPP | FX_NLGC>(ti, fx, f);
            return dispatch_acc<DPP, N, LEAN | FX_DPP>(ti, fx, f);
        }
    }
    if (fx & FX_NLGC) return dispatch_acc<DPP, N, LEAN | FX_NLGC>(ti, fx, f);
    return dispatch_acc<DPP, N, LEAN>(ti, fx, f);
}

template <bool DPP, bool LEAN, int N, class F>
auto dispatch_fx(bool ti, int fx, F&& f) {
    if constexpr (LEAN) {
        if (fx & FX_LEAN) return dispatch_fx_base<DPP, N, FX_LEAN>(ti, fx, f);
    }
    return dispatch_fx_base<DPP, N, 0>(ti, fx, f);
}

// Calls f(Variant<...>{}) for the runtime (ndim, time_interp, step features)
// combination; a policy with kOnly3D builds (and serves) 3D variants only, one
// without kDpp no momentum-diffusion variants, one without kLean ignores
// FX_LEAN.
template <class Pol, class F>
auto dispatch_variant(int ndim, bool ti, int fx, F&& f) {
    if constexpr (!Pol::kOnly3D) {
        if (ndim == 2) return dispatch_fx<Pol::kDpp, Pol::kLean, 2>(ti, fx, f);
    }
    return dispatch_fx<Pol::kDpp, Pol::kLean, 3>(ti, fx, f);
}

// Calls f(v, std::integral_constant<int, PPL>{}) for the runtime particles
// per lane: 1, or 2 where the policy supports it and the step gathers one
// frame (two frames per particle and two particles spill registers).
template <class Pol, class V, class F>
auto dispatch_ppl(int ppl, V v, F&& f) {
    if constexpr (Pol::kMaxPPL >= 2 && !V::ti) {
        if (ppl == 2) return f(v, std::integral_constant<int, 2>{});
    }
    return f(v, std::integral_constant<int, 1>{});
}

template <class Pol>
int mover_occupancy(int ndim, bool ti, int fx, int ppl) {
    return dispatch_variant<Pol>(ndim, ti, fx, [&](auto v) {
        return dispatch_ppl<Pol>(ppl, v, [](auto vv, auto pc) {
            using V = decltype(vv);
            int nb = 0;
            hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &nb, mover_kernel<Pol, V::ndim, V::ti, V::fx, decltype(pc)::value>, 256, 0);
            return e == hipSuccess ? nb : 1;
        });
    });
}

// Whether the mover and the digits for a work order are built: one-frame 2D
// steps without acceleration region, momentum diffusion or NLGC.
template <class V>
constexpr bool kOrdered = V::ndim == 2 && !V::ti && (V::fx & ~FX_LEAN) == 0;

template <class Pol>
hipError_t launch_mover(const MoverParams& m, bool ti, int fx, int ndim, int ppl, int grid,
                        hipStream_t st) {
    const int built = dispatch_variant<Pol>(ndim, ti, fx, [&](auto v) {
        return dispatch_ppl<Pol>(ppl, v, [&](auto vv, auto pc) {
            using V = decltype(vv);
            constexpr int kPpl = decltype(pc)::value;
            if (m.order) {
                if constexpr (kOrdered<V> && kPpl == 1) {
                    if constexpr (Pol::kWaits) {
                        if (m.flags & MF_WAIT) {
                            hipLaunchKernelGGL((mover_kernel<Pol, V::ndim, V::ti, V::fx, 1, true, true>),
                                               dim3(grid), dim3(256), 0, st, m);
                            return 1;
                        }
                    }
                    hipLaunchKernelGGL((mover_kernel<Pol, V::ndim, V::ti, V::fx, 1, true>), dim3(grid),
                                       dim3(256), 0, st, m);
                    return 1;
                }
                return 0;
            }
            hipLaunchKernelGGL((mover_kernel<Pol, V::ndim, V::ti, V::fx, kPpl>), dim3(grid), dim3(256), 0, st,
                               m);
            return 1;
        });
    });
    return built ? hipGetLastError() : hipErrorInvalidValue;
}

template <class Pol>
hipError_t launch_order(const MoverParams& m, bool ti, int fx, int ndim, uint32_t* digit, float* counts,
                        hipStream_t st) {
    static_assert(kOrderSample % 256 == 0, "whole blocks");
    if (m.n < (counts ? kOrderSample : 1)) return hipErrorInvalidValue;
    const int grid = counts ? kOrderSample / 256 : (int)((m.n + 255) / 256);
    const int built = dispatch_variant<Pol>(ndim, ti, fx, [&](auto v) {
        using V = decltype(v);
        if constexpr (kOrdered<V>) {
            if (counts)
                hipLaunchKernelGGL((order_sample_kernel<Pol, V::ndim, V::ti, V::fx>), dim3(grid), dim3(256), 0,
                                   st, m, counts);
            else
                hipLaunchKernelGGL((order_digit_kernel<Pol, V::ndim, V::ti, V::fx>), dim3(grid), dim3(256), 0,
                                   st, m, digit);
        }
        return kOrdered<V> ? 1 : 0;
    });
    return built ? hipGetLastError() : hipErrorInvalidValue;
}

template <class Pol>
hipError_t launch_step_once(const MoverParams& m, bool ti, int fx, int ndim, const StepRows& r,
                            hipStream_t st) {
    long long n = 0;
    for (int k = 0; k < r.pieces; ++k) n = r.n[k] > n ? r.n[k] : n;
    if (n <= 0) return hipSuccess;
    const unsigned grid = (unsigned)((n + kStepRows - 1) / kStepRows);
    dispatch_variant<Pol>(ndim, ti, fx, [&](auto v) {
        using V = decltype(v);
        hipLaunchKernelGGL((step_once_kernel<Pol, V::ndim, V::ti, V::fx>), dim3(grid, (unsigned)r.pieces),
                           dim3(kStepRows), 0, st, m, r);
        return 0;
    });
    return hipGetLastError();
}

}  // namespace sp
