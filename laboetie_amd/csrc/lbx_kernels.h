// Device code of liblbx shared by the single-lattice path (lbx.hip) and the
// multi-instance batch path (lbx_batch.hip): the control block, neighbour
// lookup, the LB work of one block of nodes (lb_step_tile, parameterised by
// the block size), the VACF reduction and the small kernels both paths launch
// (moment propagation itself: lbx_mp.h).  A lattice's nodes are a range of
// the packed fluid-node list; both paths run the same per-node arithmetic, so
// an instance gives the same bits alone or in a batch.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "lbx_device.h"
#include "lbx_tables.h"

#pragma clang fp contract(off)

namespace {

using namespace lbx;


constexpr int kBlock = 256;          // one tile = 256 consecutive packed nodes
constexpr int kSlots = 64;           // striped l2err slots per step
constexpr int kRing = 1024;          // l2err ring slots (>= 2 chunks)
constexpr int kChunk = 256;          // LB steps launched between host checks
constexpr int kMpChunk = 512;        // MP steps per host check
constexpr uint32_t kSolidSlot = 0xFFFFFFFFu;
constexpr uint32_t kIndexMask = 0x7FFFFFFFu;
constexpr uint32_t kNodeInterfacial = 0x80000000u;

// Device-side control block.  Every field has a single writer per launch
// (block 0 of a step kernel, or the one-block reduction kernel), and is read
// by later launches on the same stream, so plain stores suffice.
struct Ctrl {
    int32_t stop;                // LB: a step kernel saw the previous step converge
    int32_t restpart;            // MP: a rest probability < eps (set by mp prep)
    int64_t exit_step;           // LB: that converged step
    int64_t negpop;              // LB: first step with a negative population (-1: none)
    int32_t mp_stop;             // MP: VACF convergence reached
    int32_t mp_divide;           // MP: densities or flows outside quotient()'s range (set by mp prep)
    int64_t mp_conv_step;
    int32_t floor_hit;           // LB (FP32-shift): the stop at exit_step was the l2err floor test
    int32_t pad2;
    double l2min[2];             // LB floor test: running minimum of l2err of the stage up to step s,
    int64_t l2min_step[2];       // the step that set it, in slot s & 1,
    double l2max[2];             // and the running maximum
    double vacf0[12];            // 3 per tracer (at most 4)
    double deff_s[12], deff_c[12]; // Neumaier running sums of the VACF integrals
};

// A value another block or an earlier launch wrote (control fields, l2err
// slots, VACF partials): a relaxed device-scope atomic load, which reads past
// this CU's L1 like a volatile one but, unlike it, does not wait for each load
// before issuing the next (a volatile load is followed by a full wait).
template <typename T>
__device__ __forceinline__ T vload(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A control flag as thread 0 of the block read it, the same for every wave:
// another block may write the flag while this block's waves read it, and a
// block whose waves disagreed would split at its next barrier.
__device__ __forceinline__ bool block_flag(bool v) {
    __shared__ int32_t flag;
    __syncthreads();  // the previous use of `flag` by this block is over
    if (threadIdx.x == 0) flag = v ? 1 : 0;
    __syncthreads();
    return flag != 0;
}

// packed indices of the 18 neighbours r + c_l (l = 1..18) of full-box node r
struct Neighbours {
    uint32_t q[kQ];
    __device__ __forceinline__ void load(const uint32_t* __restrict__ map, uint32_t r, const FastDiv& dlx,
                                         const FastDiv& dly, uint32_t lz) {
        Nbr nb;
        nb.init(r, dlx, dly, lz);
        static_for<1, kQ>([&](auto I) {
            constexpr int L = I;
            q[L] = ld(map, nb.at<kCX[L], kCY[L], kCZ[L]>());
        });
    }
};

// ---------------------------------------------------------------- LB kernels

// Populations are stored as E, the step's arithmetic, its flux and step
// constants are R: E = R = double for the FP64 form; E = float (deviations
// g = n - a0 rho0 from the rest state) with R = float for the FP32-shift form
// and R = double for the FP32-store form.
template <typename E, typename R = E>
struct StepArgs {
    const E* __restrict__ fin;
    E* __restrict__ fout;
    R* __restrict__ j;
    const uint32_t* __restrict__ nodes;
    const uint32_t* __restrict__ map;
    unsigned long long* slots;            // [3][kSlots] striped per-step max|dj| bit patterns
    double* l2ring;
    Ctrl* ctrl;
    FastDiv dlx, dly;
    uint32_t lz, Nf;
    uint64_t Np;
    R A, B, C;
    R fmx, fmy, fmz;   // F(t)/2, the force of step t in j(t) (equilibration.f90:293-295)
    R fcx, fcy, fcz;   // F(t+1), the force of the collision that opens step t+1
    R rho0;            // FP32 storage: the rest density of the deviations
    int64_t t;
    int64_t check_after;    // stop check on l2err(t-1) only when t-1 > check_after
    int64_t floor_window;   // > 0: also stop when l2err set no new minimum for this many steps
    double target;
    int32_t write_l2;       // 0 for a redo of a step whose l2err is already known
    int32_t have_prev;      // step t-1 ran in this run: reduce its l2err first
    // Steps whose l2err is measured (is_check): every step when check_every
    // is 1 (FP64, and stage 1 of the FP32 storage forms); else the steps
    // check_base + m check_every (check_every a power of two), where l2err is
    // max|j(t) - j(t - check_every)| / check_every and j is kept only there
    int32_t check_every = 1;
    int32_t pad_ = 0;
    int64_t check_base = 0;
    R check_inv = R(1);     // 1 / check_every
    // TAB steps: element of the populations that direction l of node i pulls, at [(l-1) Np + i]
    const uint32_t* pulls = nullptr;
    // non-NULL: each block writes the sum of j(t) over its nodes (3 doubles,
    // in a fixed order) to jpart[3 * tile ...] (the per-step total mass flux)
    double* jpart = nullptr;
};

// A = 1 - 1/tau and B = 1/tau rounded to FP32 with A + B = 1 exactly, so that
// the FP32 relaxation keeps the momentum (rounded one by one they can miss 1
// by an ulp, a spurious force like the one a1_f32 removes).  1 - B is exact
// for B in [1/2, 2]; for smaller B, B is re-derived from the rounded A, which
// is exact for A in [1/2, 1].
inline void fp32_relaxation(double tau, float* A, float* B) {
    float b = (float)(1.0 / tau);
    const float a = 1.0f - b;
    if (!(b >= 0.5f)) b = 1.0f - a;
    *A = a;
    *B = b;
}

// The number of steps between the l2err measurements of the FP32 storage
// forms' stage 2 (a power of two)
constexpr int32_t kCheckEvery = 64;

// In the FP32 storage forms, j(t) - j(t-1) at a node is of the order of the
// rounding of j itself once the flow is nearly steady, so the per-step max|dj|
// settles on a rounding floor well above what the flow's decay would give and
// a stage would end early on the floor test.  Over check_every steps the decay
// adds up while the rounding does not, so the difference divided by
// check_every follows the decay down by that factor more; it also leaves j out
// of the other steps' memory traffic.
__host__ __device__ __forceinline__ bool is_check(int64_t s, int64_t base, int32_t every) {
    return every <= 1 || (s - base) % every == 0;
}

// A negative population among a block's nodes is reported as +inf in place of
// its max|dj| (max over bit patterns of non-negative doubles = max of values).
constexpr unsigned long long kNegMark = 0x7FF0000000000000ull;

// the floor test needs l2err this far below the stage's maximum
constexpr double kFloorDrop = 1e-2;

// maximum over the 64 lanes of a wave, returned to every lane (all 64 lanes
// active): DPP row steps, then the four row maxima
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
    const auto step = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, C, 0xf, 0xf, false);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), C, 0xf, 0xf, false);
        const unsigned long long o = ((unsigned long long)hi << 32) | lo;
        v = o > v ? o : v;
    };
    step(std::integral_constant<int, 0xB1>{});
    step(std::integral_constant<int, 0x4E>{});
    step(std::integral_constant<int, 0x141>{});
    step(std::integral_constant<int, 0x140>{});
    unsigned long long m = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, 16 * r);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), 16 * r);
        const unsigned long long o = ((unsigned long long)hi << 32) | lo;
        m = o > m ? o : m;
    }
    return m;
}

// max over the kSlots slots of one step (called by the first wave of a block)
__device__ __forceinline__ unsigned long long slots_max(const unsigned long long* set) {
    return wave_max_u64(vload(&set[threadIdx.x & (kSlots - 1)]));
}

// Per-block sums of NV values in a fixed order, written to out[0 .. NV-1]
// (value a by thread a).
template <int NV, int BLOCK>
__device__ __forceinline__ void block_partial(const double (&v)[NV], double* out, double* lds /* [BLOCK/64*NV] */) {
    static_assert(NV <= BLOCK, "one thread per value");
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double s[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) s[a] = v[a];
    wave_sums<NV>(s);
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < NV; ++a) lds[w * NV + a] = s[a];
    __syncthreads();
    if (threadIdx.x < NV) {  // value a summed over the waves in wave order, by thread a
        const int a = threadIdx.x;
        double s = lds[a];
        for (int k = 1; k < BLOCK / 64; ++k) s = s + lds[k * NV + a];
        out[a] = s;
    }
    __syncthreads();
}

// Pull-streaming with half-way bounce-back (equilibration.f90:204-243): the
// population arriving at node i in direction L left r - c_L, or, when that
// node is solid, left i itself in direction inv(L).
// The two candidate sources differ only in the lane's element index, so one
// load per direction serves both.
template <int L>
__device__ __forceinline__ uint32_t pull_source(uint32_t Np, uint32_t i, const Neighbours& nb) {
    if constexpr (L == 0) {
        return i;
    } else {
        const uint32_t q = nb.q[kInv[L]];  // r - c_L = r + c_inv(L)
        return q != kSolidSlot ? (uint32_t)L * Np + q : (uint32_t)kInv[L] * Np + i;
    }
}
template <int L, bool Wide, typename E>
__device__ __forceinline__ E pull(const View<Wide, E>& fin, uint32_t Np, uint32_t i, const Neighbours& nb) {
    return fin.ld(pull_source<L>(Np, i, nb));
}

// the pull sources of every node (StepArgs::pulls)
__global__ __launch_bounds__(kBlock) void k_pull_table(uint32_t* __restrict__ pulls, const uint32_t* __restrict__ nodes,
                                                       const uint32_t* __restrict__ map, FastDiv dlx, FastDiv dly,
                                                       uint32_t lz, uint32_t Nf, uint32_t Np) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    Neighbours nb;
    nb.load(map, nodes[i] & kIndexMask, dlx, dly, lz);
    static_for<1, kQ>([&](auto I) { pulls[(uint64_t)(I - 1) * Np + i] = pull_source<I>(Np, i, nb); });
}

// One time step, fused: pull-streaming with bounce-back of the post-collision
// populations of step t, the negativity check (equilibration.f90:248),
// density (:254) and flux (:293-300), the l2err contribution (:339-344), then
// the collision that opens step t+1 (module_collision.f90:87-108).
// E = float: the FP32-shift form; the l2err is still a max of FP64 values.
#ifndef LBX_LB_WAVES
#define LBX_LB_WAVES 1
#endif
//
// lb_step_tile is one block's share: `tile` is the block's tile (BLOCK
// consecutive packed nodes, i = tile*BLOCK + lane, valid below a.Nf), `stripe`
// picks its l2err slot, and `first_block` is the one block of the lattice that
// writes the step's control fields and clears the next step's slots.
//
// TAB (small lattices, whose step is a chain of round trips to memory and not
// bytes): the pull sources come from a table in place of node word and map,
// and the stop flags are looked at after the populations have been asked for:
// two round trips instead of four.
template <int BLOCK, bool Wide, typename E, typename R = E, bool NT = false, bool TAB = false>
__device__ __forceinline__ void lb_step_tile(const StepArgs<E, R>& a, uint32_t tile, uint32_t stripe,
                                             bool first_block) {
    constexpr bool kShift = std::is_same<E, float>::value;  // deviations stored in FP32
    const uint32_t i = tile * BLOCK + threadIdx.x;
    // Each wave's work is a chain of dependent memory round trips, so
    // independent requests go out together: the node word, the stop flags
    // and the previous step's l2err slots (read whether or not a flag is set).
    const uint32_t node = !TAB && i < a.Nf ? ld(a.nodes, i) : 0u;
    __shared__ int32_t stop_flag;
    __shared__ unsigned long long prev_bits;
    __syncthreads();  // a previous step of this block (persistent launches) has read both
    bool stop = false;
    unsigned long long prev = 0ull;
    if (threadIdx.x < 64) {
        stop = ((int)(vload(&a.ctrl->stop) != 0) | (int)(vload(&a.ctrl->negpop) >= 0)) != 0;
        if (a.have_prev) prev = vload(a.slots + ((a.t - 1) % 3) * kSlots + (threadIdx.x & (kSlots - 1)));
    }
    E early[TAB ? kQ : 1];  // TAB: the populations and j_old
    R jearly[3] = {R(0), R(0), R(0)};
    if constexpr (TAB)
        if (i < a.Nf) {
            const uint32_t Np = (uint32_t)a.Np;
            const View<Wide, E> fin(a.fin, kQ * a.Np);
            uint32_t src[kQ];
            static_for<1, kQ>([&](auto I) { src[I] = ld(a.pulls, (I - 1) * Np + i); });
            if (a.write_l2 && is_check(a.t, a.check_base, a.check_every)) {
                const View<Wide, R> jv(a.j, 3 * a.Np);
                for (int c = 0; c < 3; ++c) jearly[c] = jv.ld(c * Np + i);
            }
            early[0] = fin.ld(i);
            static_for<1, kQ>([&](auto I) { early[I] = fin.ld(src[I]); });
        }
    if (threadIdx.x < 64) {
        const unsigned long long v = wave_max_u64(prev);
        if (threadIdx.x == 0) {
            stop_flag = stop ? 1 : 0;
            prev_bits = v;
        }
    }
    __syncthreads();
    if (stop_flag) return;
    if (a.have_prev) {
        // l2err of step t-1 (equilibration.f90:339-344) from its striped
        // slots, then the negativity (:248) and convergence (:346) verdicts
        const bool first = first_block && threadIdx.x == 0;
        if (prev_bits == kNegMark) {
            if (first) a.ctrl->negpop = a.t - 1;
            return;
        }
        // a step without a measurement (is_check false) records NaN and
        // takes no stop decision
        const bool chk = is_check(a.t - 1, a.check_base, a.check_every);
        const double prev = chk ? __longlong_as_double((long long)prev_bits) : __builtin_nan("");
        if (first) a.l2ring[(a.t - 1) % kRing] = prev;
        bool floor = false;
        if (a.floor_window > 0 && a.t - 1 > a.check_after) {
            // record of the stage up to step t-1 from the one up to t-2 (every
            // block derives the same record; block 0 stores it for step t+1)
            const int s0 = (int)((a.t - 2) & 1), s1 = (int)((a.t - 1) & 1);
            double m = vload(&a.ctrl->l2min[s0]), mx = vload(&a.ctrl->l2max[s0]);
            int64_t ms = vload(&a.ctrl->l2min_step[s0]);
            if (chk) {
                if (prev < m) {
                    m = prev;
                    ms = a.t - 1;
                }
                mx = fmax(mx, prev);
            }
            if (first) {
                a.ctrl->l2min[s1] = m;
                a.ctrl->l2min_step[s1] = ms;
                a.ctrl->l2max[s1] = mx;
            }
            // a floor: no new minimum for floor_window steps after l2err has
            // fallen 100-fold below the stage's largest value (a plateau of a
            // still-accelerating flow is not one)
            floor = chk && (a.t - 1) - ms >= a.floor_window && m <= kFloorDrop * mx;
        }
        if (chk && a.t - 1 > a.check_after && (prev <= a.target || floor)) {
            if (first) {
                a.ctrl->exit_step = a.t - 1;
                a.ctrl->floor_hit = prev <= a.target ? 0 : 1;
                a.ctrl->stop = 1;
            }
            return;
        }
    }
    // clear the slots of step t+1 (last used by step t-2, read by step t-1)
    if (a.write_l2 && first_block && threadIdx.x < kSlots) a.slots[((a.t + 1) % 3) * kSlots + threadIdx.x] = 0ull;
    double l2 = 0.0;
    bool neg = false;
    double jsum[3] = {0.0, 0.0, 0.0};  // this node's j(t), for the flux sums
    if (i < a.Nf) {
        const uint32_t Np = (uint32_t)a.Np;
        const View<Wide, E> fin(a.fin, kQ * a.Np), fout(a.fout, kQ * a.Np);
        const View<Wide, R> jv(a.j, 3 * a.Np);
        Neighbours nb;
        if constexpr (!TAB) nb.load(a.map, node & kIndexMask, a.dlx, a.dly, a.lz);
        // l2err of this step is measured: always in FP64; in the FP32 storage
        // forms only at the check steps, the only ones that read and keep j
        const bool chk = a.write_l2 && is_check(a.t, a.check_base, a.check_every);
        R jo[3] = {jearly[0], jearly[1], jearly[2]};
        if (!TAB && chk) {  // j_old, issued before the populations so its latency overlaps theirs
            jo[0] = jv.ld(i);
            jo[1] = jv.ld(Np + i);
            jo[2] = jv.ld(2 * Np + i);
        }
        R f[kQ];
        static_for<0, kQ>([&](auto I) {
            if constexpr (TAB) f[I] = (R)early[I]; else f[I] = (R)pull<I, Wide, E>(fin, Np, i, nb);
        });
        if constexpr (kShift)  // n < 0  <=>  g < -a0 rho0
            static_for<0, kQ>([&](auto I) { neg = neg || (f[I] < -((R)a0(I) * a.rho0)); });
        else
            static_for<0, kQ>([&](auto I) { neg = neg || (f[I] < 0.0); });
        R rho = f[0];  // FP32 storage: drho = rho - rho0
        static_for<1, kQ>([&](auto I) { rho = rho + f[I]; });
        R jx = a.fmx, jy = a.fmy, jz = a.fmz;
        static_for<0, kQ>([&](auto I) {
            constexpr int L = I;
            if constexpr (kCX[L] != 0) jx = jx + sgn<kCX[L]>(f[L]);
            if constexpr (kCY[L] != 0) jy = jy + sgn<kCY[L]>(f[L]);
            if constexpr (kCZ[L] != 0) jz = jz + sgn<kCZ[L]>(f[L]);
        });
        if (chk) {
            R dx = fabs(jx - jo[0]), dy = fabs(jy - jo[1]), dz = fabs(jz - jo[2]);
            if constexpr (kShift) {  // exact: check_inv is a power of two
                dx = dx * a.check_inv;
                dy = dy * a.check_inv;
                dz = dz * a.check_inv;
            }
            l2 = (double)fmax(fmax(dx, dy), dz);
        }
        if (!kShift || chk) {  // FP64: j of every step is the run's output flux
            jv.st(i, jx);
            jv.st(Np + i, jy);
            jv.st(2 * Np + i, jz);
        }
        jsum[0] = (double)jx;
        jsum[1] = (double)jy;
        jsum[2] = (double)jz;
        if constexpr (kShift) {
            const R drho = rho, full = a.rho0 + drho;
            R ux, uy, uz;
            shift_velocity<R>(jx, jy, jz, full, ux, uy, uz);
            static_for<0, kQ>([&](auto I) {
                constexpr int L = I;
                const E v = (E)collide_shift<L, R>(f[L], drho, jx, jy, jz, ux, uy, uz, a.fcx, a.fcy, a.fcz, a.A,
                                                   a.B, a.C);
                if constexpr (NT)
                    fout.stnt((uint32_t)L * Np + i, v);
                else
                    fout.st((uint32_t)L * Np + i, v);
            });
        } else {
            const double ux = jx / rho, uy = jy / rho, uz = jz / rho;
            static_for<0, kQ>([&](auto I) {
                constexpr int L = I;
                const double v = collide_pop<L>(f[L], rho, jx, jy, jz, ux, uy, uz, a.fcx, a.fcy, a.fcz, a.A, a.B, a.C);
                if constexpr (NT)
                    fout.stnt((uint32_t)L * Np + i, v);
                else
                    fout.st((uint32_t)L * Np + i, v);
            });
        }
    }
    if (a.write_l2) {
        __shared__ double lds[BLOCK / 64];
        l2 = wave_max(l2);
        const bool wneg = __ballot(neg) != 0ull;
        if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = wneg ? -1.0 : l2;
        __syncthreads();
        if (threadIdx.x == 0) {
            double m = lds[0];
            bool bneg = m < 0.0;
            for (int w = 1; w < BLOCK / 64; ++w) {
                bneg = bneg || lds[w] < 0.0;
                m = fmax(m, lds[w]);
            }
            if (bneg || m > 0.0)
                atomicMax(&a.slots[(a.t % 3) * kSlots + (stripe & (kSlots - 1))],
                          bneg ? kNegMark : (unsigned long long)__double_as_longlong(m));
        }
        if (a.jpart) {
            __shared__ double jl[BLOCK / 64 * 3];
            block_partial<3, BLOCK>(jsum, a.jpart + 3 * (uint64_t)tile, jl);
        }
    }
}

// The FP32-store step (FP32 storage, FP64 arithmetic) fits five waves per
// SIMD without spilling; the compiler's own choice leaves it at four.
template <typename E, typename R>
constexpr int kLbMinWaves = (std::is_same<E, float>::value && std::is_same<R, double>::value) ? 5 : LBX_LB_WAVES;

// NT: the outgoing populations are written with the streaming hint, for a
// lattice whose two population sets outgrow the last-level cache, where the
// next step's reads find none of them there anyway.
#ifndef LBX_NT_MIN_BYTES  // population footprint (both sets) above which LB stores stream
#define LBX_NT_MIN_BYTES (256ull << 20)
#endif
template <bool Wide, typename E, typename R = E, bool NT = false, bool TAB = false>
__global__ __launch_bounds__(kBlock, (TAB ? 2 : kLbMinWaves<E, R>)) void k_lb_step(StepArgs<E, R> a) {
    lb_step_tile<kBlock, Wide, E, R, NT, TAB>(a, xcd_tile(), blockIdx.x, blockIdx.x == 0);
}

// l2err of the last step of a launch run, which no later step kernel reads
// (called by one wave).
__device__ __forceinline__ void lb_finalize(const unsigned long long* slots, double* l2ring, Ctrl* ctrl, int64_t t,
                                            int64_t check_base, int32_t check_every) {
    if (vload(&ctrl->stop) || vload(&ctrl->negpop) >= 0) return;
    const unsigned long long v = slots_max(slots + (t % 3) * kSlots);
    if (threadIdx.x == 0) {
        if (v == kNegMark)
            ctrl->negpop = t;
        else
            l2ring[t % kRing] =
                is_check(t, check_base, check_every) ? __longlong_as_double((long long)v) : __builtin_nan("");
    }
}

__global__ __launch_bounds__(64) void k_lb_finalize(const unsigned long long* slots, double* l2ring, Ctrl* ctrl,
                                                    int64_t t, int64_t check_base, int32_t check_every) {
    lb_finalize(slots, l2ring, ctrl, t, check_base, check_every);
}

// A whole launch run of steps t0+1 .. t0+S (a.t = t0) in one launch of one
// block, for a lattice of at most kRunNodes nodes: one node a thread, the
// post-collision populations in LDS and j_old in registers, two barriers a
// step in place of a launch.  The last step's two population sets, the flags,
// l2err record and slots are left as the launches leave them; arithmetic and
// verdicts are lb_step_tile's.  One CU does the work of all, so it pays while
// few waves share its SIMDs: us per step launched / here, FP64 and FP32-shift,
// 60 nodes 4.8 / 1.5 and 4.7 / 1.5, 256 nodes 5.1 / 1.9 and 4.8 / 1.8, 512 nodes
// 5.3 / 3.1 and 5.2 / 2.8; a second node a thread would double the last.
constexpr uint32_t kRunNodes = 512;

template <typename E, typename R>
__global__ __launch_bounds__(kRunNodes) void k_lb_run(StepArgs<E, R> a, E* f0, E* f1, int64_t S) {
    constexpr bool kShift = std::is_same<E, float>::value;
    __shared__ E pop[kQ * kRunNodes];
    __shared__ double red[kRunNodes / 64];
    __shared__ unsigned long long first_bits;
    const uint32_t i = threadIdx.x, Np = (uint32_t)a.Np, nwaves = blockDim.x >> 6;
    const bool valid = i < a.Nf, first = i == 0;
    const int64_t t0 = a.t;
    if (block_flag((int)(vload(&a.ctrl->stop) != 0) | (int)(vload(&a.ctrl->negpop) >= 0))) return;
    // the record of the stage up to step t0 - 1, in every thread
    double lmin = a.ctrl->l2min[(t0 - 1) & 1], lmax = a.ctrl->l2max[(t0 - 1) & 1];
    int64_t lstep = a.ctrl->l2min_step[(t0 - 1) & 1];
    // the verdicts on step t, which step t+1 takes in lb_step_tile: true ends the run
    const auto ends = [&](int64_t t, unsigned long long bits) {
        if (bits == kNegMark) {
            if (first) a.ctrl->negpop = t;
            return true;
        }
        const bool chk = is_check(t, a.check_base, a.check_every);
        const double prev = chk ? __longlong_as_double((long long)bits) : __builtin_nan("");
        if (first) a.l2ring[t % kRing] = prev;
        bool floor = false;
        if (a.floor_window > 0 && t > a.check_after) {
            if (chk) {
                if (prev < lmin) {
                    lmin = prev;
                    lstep = t;
                }
                lmax = fmax(lmax, prev);
            }
            floor = chk && t - lstep >= a.floor_window && lmin <= kFloorDrop * lmax;
        }
        if (!(chk && t > a.check_after && (prev <= a.target || floor))) return false;
        if (first) {
            a.ctrl->exit_step = t;
            a.ctrl->floor_hit = prev <= a.target ? 0 : 1;
            a.ctrl->stop = 1;
        }
        return true;
    };
    if (t0 > 0) {
        if (i < 64) {
            const unsigned long long v = slots_max(a.slots + (t0 % 3) * kSlots);
            if (first) first_bits = v;
        }
        __syncthreads();
        if (ends(t0, first_bits)) return;
    }
    uint16_t src[kQ];
    R jo[3] = {R(0), R(0), R(0)};
    if (valid) {
        const E* fin = t0 & 1 ? f1 : f0;
        src[0] = (uint16_t)i;
        static_for<1, kQ>([&](auto I) {
            const uint32_t v = a.pulls[(uint64_t)(I - 1) * Np + i];
            src[I] = (uint16_t)(v / Np * kRunNodes + v % Np);
        });
        static_for<0, kQ>([&](auto I) { pop[I * kRunNodes + i] = fin[(uint64_t)I * Np + i]; });
        for (int c = 0; c < 3; ++c) jo[c] = a.j[c * (uint64_t)Np + i];
    }
    __syncthreads();
    for (int64_t t = t0 + 1;; ++t) {
        const bool chk = is_check(t, a.check_base, a.check_every);
        double l2 = 0.0;
        bool neg = false;
        E out[kQ];
        if (valid) {
            R f[kQ];
            static_for<0, kQ>([&](auto I) { f[I] = (R)pop[src[I]]; });
            if constexpr (kShift)
                static_for<0, kQ>([&](auto I) { neg = neg || (f[I] < -((R)a0(I) * a.rho0)); });
            else
                static_for<0, kQ>([&](auto I) { neg = neg || (f[I] < 0.0); });
            R rho = f[0];
            static_for<1, kQ>([&](auto I) { rho = rho + f[I]; });
            R jx = a.fmx, jy = a.fmy, jz = a.fmz;
            static_for<0, kQ>([&](auto I) {
                constexpr int L = I;
                if constexpr (kCX[L] != 0) jx = jx + sgn<kCX[L]>(f[L]);
                if constexpr (kCY[L] != 0) jy = jy + sgn<kCY[L]>(f[L]);
                if constexpr (kCZ[L] != 0) jz = jz + sgn<kCZ[L]>(f[L]);
            });
            if (chk) {
                R dx = fabs(jx - jo[0]), dy = fabs(jy - jo[1]), dz = fabs(jz - jo[2]);
                if constexpr (kShift) {
                    dx = dx * a.check_inv;
                    dy = dy * a.check_inv;
                    dz = dz * a.check_inv;
                }
                l2 = (double)fmax(fmax(dx, dy), dz);
            }
            if (!kShift || chk) {
                jo[0] = jx;
                jo[1] = jy;
                jo[2] = jz;
            }
            if constexpr (kShift) {
                const R drho = rho, full = a.rho0 + drho;
                R ux, uy, uz;
                shift_velocity<R>(jx, jy, jz, full, ux, uy, uz);
                static_for<0, kQ>([&](auto I) {
                    constexpr int L = I;
                    out[L] = (E)collide_shift<L, R>(f[L], drho, jx, jy, jz, ux, uy, uz, a.fcx, a.fcy, a.fcz, a.A, a.B,
                                                    a.C);
                });
            } else {
                const double ux = jx / rho, uy = jy / rho, uz = jz / rho;
                static_for<0, kQ>([&](auto I) {
                    constexpr int L = I;
                    out[L] = collide_pop<L>(f[L], rho, jx, jy, jz, ux, uy, uz, a.fcx, a.fcy, a.fcz, a.A, a.B, a.C);
                });
            }
        }
        l2 = wave_max(l2);
        const bool wneg = __ballot(neg) != 0ull;
        if ((i & 63u) == 0) red[i >> 6] = wneg ? -1.0 : l2;
        __syncthreads();  // every read of the populations is over
        double m = red[0];
        bool bneg = m < 0.0;
        for (uint32_t w = 1; w < nwaves; ++w) {
            bneg = bneg || red[w] < 0.0;
            m = fmax(m, red[w]);
        }
        const unsigned long long bits =
            bneg ? kNegMark : (m > 0.0 ? (unsigned long long)__double_as_longlong(m) : 0ull);
        if (t == t0 + S || ends(t, bits)) {
            if (valid) {
                E *fin = t & 1 ? f0 : f1, *fout = t & 1 ? f1 : f0;
                static_for<0, kQ>([&](auto I) {
                    fin[(uint64_t)I * Np + i] = pop[I * kRunNodes + i];
                    fout[(uint64_t)I * Np + i] = out[I];
                });
                for (int c = 0; c < 3; ++c) a.j[c * (uint64_t)Np + i] = jo[c];
            }
            if (i < kSlots) {
                a.slots[(t % 3) * kSlots + i] = i == 0 ? bits : 0ull;
                a.slots[((t + 1) % 3) * kSlots + i] = 0ull;
            }
            break;
        }
        if (valid) static_for<0, kQ>([&](auto I) { pop[I * kRunNodes + i] = out[I]; });
        __syncthreads();
    }
    if (first) {
        for (int k = 0; k < 2; ++k) {
            a.ctrl->l2min[k] = lmin;
            a.ctrl->l2min_step[k] = lstep;
            a.ctrl->l2max[k] = lmax;
        }
    }
}

// Streaming only: the post-streaming state f_s(t) of the step whose input is
// fin, and its density SUM(n,4) (equilibration.f90:254), of packed node i.
__device__ __forceinline__ void extract_node(const double* __restrict__ fin, double* __restrict__ nout,
                                             double* __restrict__ rho_out, const Neighbours& nb, uint32_t i,
                                             uint64_t Np) {
    const View<true> fv(fin, kQ * Np);
    double rho = 0.0;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const double v = pull<L, true>(fv, (uint32_t)Np, i, nb);
        nout[(uint64_t)L * Np + i] = v;
        rho = (L == 0) ? v : rho + v;
    });
    rho_out[i] = rho;
}

// The same for the FP32-shift form: the post-streaming deviations g into
// gout, and the FP64 density rho0 + sum g and flux F/2 + sum g c, summed in
// FP64 from the FP32 deviations (the flow that moment propagation reads).
__device__ __forceinline__ void extract_node_shift(const float* __restrict__ gin, float* __restrict__ gout,
                                                   double* __restrict__ rho_out, double* __restrict__ j_out,
                                                   const Neighbours& nb, uint32_t i, uint64_t Np, double rho0,
                                                   double fmx, double fmy, double fmz) {
    const View<true, float> gv(gin, kQ * Np);
    double drho = 0.0, jx = fmx, jy = fmy, jz = fmz;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const float v = pull<L, true>(gv, (uint32_t)Np, i, nb);
        gout[(uint64_t)L * Np + i] = v;
        const double d = v;
        drho = (L == 0) ? d : drho + d;
        if constexpr (kCX[L] != 0) jx = jx + sgn<kCX[L]>(d);
        if constexpr (kCY[L] != 0) jy = jy + sgn<kCY[L]>(d);
        if constexpr (kCZ[L] != 0) jz = jz + sgn<kCZ[L]>(d);
    });
    rho_out[i] = rho0 + drho;
    j_out[i] = jx;
    j_out[Np + i] = jy;
    j_out[2 * Np + i] = jz;
}

__global__ __launch_bounds__(kBlock) void k_extract(const double* __restrict__ fin, double* __restrict__ nout,
                                                    double* __restrict__ rho_out, const uint32_t* __restrict__ nodes,
                                                    const uint32_t* __restrict__ map, FastDiv dlx, FastDiv dly,
                                                    uint32_t lz, uint32_t Nf, uint64_t Np) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    Neighbours nb;
    nb.load(map, nodes[i] & kIndexMask, dlx, dly, lz);
    extract_node(fin, nout, rho_out, nb, i, Np);
}

__global__ __launch_bounds__(kBlock) void k_extract_shift(const float* __restrict__ gin, float* __restrict__ gout,
                                                          double* __restrict__ rho_out, double* __restrict__ j_out,
                                                          const uint32_t* __restrict__ nodes,
                                                          const uint32_t* __restrict__ map, FastDiv dlx, FastDiv dly,
                                                          uint32_t lz, uint32_t Nf, uint64_t Np, double rho0,
                                                          double fmx, double fmy, double fmz) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    Neighbours nb;
    nb.load(map, nodes[i] & kIndexMask, dlx, dly, lz);
    extract_node_shift(gin, gout, rho_out, j_out, nb, i, Np, rho0, fmx, fmy, fmz);
}

// The density SUM(n,4) (equilibration.f90:254) and flux F(t)/2 + sum n c
// (:293-300) of the post-streaming state of the step whose input is fin,
// without writing the populations (the run goes on from fin): out[0][Np] the
// density, out[1..3][Np] the flux.  The same sums in the same order as
// k_extract and the step kernel.
__global__ __launch_bounds__(kBlock) void k_flow(const double* __restrict__ fin, double* __restrict__ out,
                                                 const uint32_t* __restrict__ nodes, const uint32_t* __restrict__ map,
                                                 FastDiv dlx, FastDiv dly, uint32_t lz, uint32_t Nf, uint64_t Np,
                                                 double fmx, double fmy, double fmz) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    Neighbours nb;
    nb.load(map, nodes[i] & kIndexMask, dlx, dly, lz);
    const View<true> fv(fin, kQ * Np);
    double rho = 0.0, jx = fmx, jy = fmy, jz = fmz;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const double v = pull<L, true>(fv, (uint32_t)Np, i, nb);
        rho = (L == 0) ? v : rho + v;
        if constexpr (kCX[L] != 0) jx = jx + sgn<kCX[L]>(v);
        if constexpr (kCY[L] != 0) jy = jy + sgn<kCY[L]>(v);
        if constexpr (kCZ[L] != 0) jz = jz + sgn<kCZ[L]>(v);
    });
    out[i] = rho;
    out[Np + i] = jx;
    out[2 * Np + i] = jy;
    out[3 * Np + i] = jz;
}

// The same for the FP32 storage forms, as k_extract_shift sums them: FP64
// density rho0 + sum g and flux F(t)/2 + sum g c from the FP32 deviations.
__global__ __launch_bounds__(kBlock) void k_flow_shift(const float* __restrict__ gin, double* __restrict__ out,
                                                       const uint32_t* __restrict__ nodes,
                                                       const uint32_t* __restrict__ map, FastDiv dlx, FastDiv dly,
                                                       uint32_t lz, uint32_t Nf, uint64_t Np, double rho0,
                                                       double fmx, double fmy, double fmz) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    Neighbours nb;
    nb.load(map, nodes[i] & kIndexMask, dlx, dly, lz);
    const View<true, float> gv(gin, kQ * Np);
    double drho = 0.0, jx = fmx, jy = fmy, jz = fmz;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const double d = pull<L, true>(gv, (uint32_t)Np, i, nb);
        drho = (L == 0) ? d : drho + d;
        if constexpr (kCX[L] != 0) jx = jx + sgn<kCX[L]>(d);
        if constexpr (kCY[L] != 0) jy = jy + sgn<kCY[L]>(d);
        if constexpr (kCZ[L] != 0) jz = jz + sgn<kCZ[L]>(d);
    });
    out[i] = rho0 + drho;
    out[Np + i] = jx;
    out[2 * Np + i] = jy;
    out[3 * Np + i] = jz;
}

// The collision on packed fields with a uniform force (the opening collision
// of a run), in place: module_collision.f90:87-108.
__global__ __launch_bounds__(kBlock) void k_collide_packed(double* f, const double* __restrict__ rho,
                                                           const double* __restrict__ j, double fx, double fy,
                                                           double fz, uint32_t Nf, uint64_t Np, double A, double B,
                                                           double C) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    const double d = rho[i], jx = j[i], jy = j[Np + i], jz = j[2 * Np + i];
    const double ux = jx / d, uy = jy / d, uz = jz / d;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const double v = f[(uint64_t)L * Np + i];
        f[(uint64_t)L * Np + i] = collide_pop<L>(v, d, jx, jy, jz, ux, uy, uz, fx, fy, fz, A, B, C);
    });
}

// The same for the FP32 storage forms: the FP64 density and flux of the state
// become the step's drho = rho - rho0 and j (type R: float for FP32-shift,
// double for FP32-store) of the collision and j_old of the first step
// (jold may be j itself in the FP32-store form).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_collide_packed_shift(float* g, const double* __restrict__ rho,
                                                                 const double* j, R* jold, R fx, R fy, R fz,
                                                                 uint32_t Nf, uint64_t Np, R A, R B, R C,
                                                                 double rho0) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    const R drho = (R)(rho[i] - rho0), full = (R)rho0 + drho;
    const R jx = (R)j[i], jy = (R)j[Np + i], jz = (R)j[2 * Np + i];
    jold[i] = jx;  // j_old of the first step
    jold[Np + i] = jy;
    jold[2 * Np + i] = jz;
    R ux, uy, uz;
    shift_velocity<R>(jx, jy, jz, full, ux, uy, uz);
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const R v = g[(uint64_t)L * Np + i];
        g[(uint64_t)L * Np + i] = (float)collide_shift<L, R>(v, drho, jx, jy, jz, ux, uy, uz, fx, fy, fz, A, B, C);
    });
}

// collide() on whole full-box fields with per-node forces, in place
// (module_collision.f90:15-130, fluid nodes only): the stateless entry point.
__global__ __launch_bounds__(kBlock) void k_collide_box(double* f, const double* __restrict__ rho,
                                                        const double* __restrict__ j,
                                                        const double* __restrict__ F,
                                                        const int8_t* __restrict__ nature, uint32_t N, double A,
                                                        double B, double C) {
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= N || nature[r] != 0) return;
    const uint64_t n = N;
    const double d = rho[r], jx = j[r], jy = j[n + r], jz = j[2 * n + r];
    const double fx = F[r], fy = F[n + r], fz = F[2 * n + r];
    const double ux = jx / d, uy = jy / d, uz = jz / d;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        const double v = f[(uint64_t)L * n + r];
        f[(uint64_t)L * n + r] = collide_pop<L>(v, d, jx, jy, jz, ux, uy, uz, fx, fy, fz, A, B, C);
    });
}

// Rest state, init_simu.f90:31-39: n = rho0*a0 at fluid nodes, j = 0; in the
// FP32-shift form (g != NULL) the deviations g = 0 and the FP32 flux j32 = 0.
__global__ __launch_bounds__(kBlock) void k_init_rest(double* __restrict__ f, float* __restrict__ g,
                                                      float* __restrict__ j32, double* __restrict__ rho,
                                                      double* __restrict__ j, uint32_t Nf, uint64_t Np,
                                                      double rho0) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= Nf) return;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        if (f) f[(uint64_t)L * Np + i] = rho0 * a0(L);
        if (g) g[(uint64_t)L * Np + i] = 0.0f;
    });
    rho[i] = rho0;
    for (int c = 0; c < 3; ++c) {
        j[c * Np + i] = 0.0;
        if (j32) j32[c * Np + i] = 0.0f;
    }
}

// ---------------------------------------------------------------- MP kernels

// Several tracers that share the flow and Db (so the scattering
// probabilities, rem and u*) but differ in ka, kd can be propagated in one
// pass: the shared coefficients are read once per node for all of them.  The
// arithmetic of each tracer is exactly that of a single-tracer run.

constexpr int kMaxTracers = 4;

// VACF of one moment-propagation step (NV = 3 per tracer) from the per-block
// partial sums, in a fixed order that does not depend on which kernel runs it
// (so every run gives the same bits), then the running D_eff sums and,
// optionally, the convergence test of module_moment_propagation.f90:284-288
// (all NV components below both limits).  Called by all BLOCK threads of one
// block.  mode 0: VACF(0) of mp init; mode 1: VACF(it) of a step.
// Component a is summed over the waves and kept by thread a, whose loads of the
// running sums go out with the partials: one thread doing all components paid
// a memory round trip for each (a 3-tracer step of 2 000 nodes: 11.9 us).
template <int NV, int BLOCK>
__device__ __forceinline__ void mp_reduce_block(const double* part, uint32_t nparts, double* vtrace, Ctrl* ctrl,
                                                int32_t mode, int64_t it, int32_t check_conv, double lim1,
                                                double lim2, double* lds /* [BLOCK/64*NV] */) {
    static_assert(NV <= 64, "one wave keeps the components");
    const int me = threadIdx.x;
    double run_s = 0.0, run_c = 0.0;
    if (mode != 0 && me < NV) {
        run_s = ctrl->deff_s[me];
        run_c = ctrl->deff_c[me];
    }
    double s[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) s[a] = 0.0;
    for (uint32_t k = threadIdx.x; k < nparts; k += BLOCK)
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            const double x = vload(&part[(uint64_t)NV * k + a]);
            s[a] = (k == threadIdx.x) ? x : s[a] + x;
        }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    wave_sums<NV>(s);
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < NV; ++a) lds[w * NV + a] = s[a];
    __syncthreads();
    if (w == 0) {
        bool below = true;
        if (me < NV) {
            double t = lds[me];
            for (int k = 1; k < BLOCK / 64; ++k) t = t + lds[k * NV + me];
            if (mode == 0) {
                ctrl->vacf0[me] = t;
                ctrl->deff_s[me] = 0.5 * t;
                ctrl->deff_c[me] = 0.0;
            } else {
                vtrace[me] = t;
                // Neumaier update of D = VACF(0)/2 + sum VACF(t)
                const double u = run_s + t;
                ctrl->deff_c[me] = run_c + ((fabs(run_s) >= fabs(t)) ? (run_s - u) + t : (t - u) + run_s);
                ctrl->deff_s[me] = u;
            }
            below = fabs(t) < lim1 && fabs(t) < lim2;
        }
        if (mode != 0 && check_conv && it > 2 && __all(below) && me == 0) {
            ctrl->mp_conv_step = it;
            ctrl->mp_stop = 1;
        }
    }
    __syncthreads();
}

template <int NV>
__global__ __launch_bounds__(kBlock) void k_mp_reduce(const double* __restrict__ part, uint32_t nparts,
                                                      double* vtrace, Ctrl* ctrl, int32_t mode, int64_t it,
                                                      int32_t check_conv, double lim1, double lim2) {
    __shared__ double lds[kBlock / 64 * NV];
    if (mode == 1 && vload(&ctrl->mp_stop)) return;
    mp_reduce_block<NV, kBlock>(part, nparts, vtrace, ctrl, mode, it, check_conv, lim1, lim2, lds);
}

struct TracerParams {
    double bw[kMaxTracers];    // 1/Pstat (module_moment_propagation.f90:97,108)
    double ka[kMaxTracers], kd[kMaxTracers], one_minus_kd[kMaxTracers];
    int32_t ads[kMaxTracers];  // adsorption on (K = ka/kd > eps, :46-56)
};

// W is the type the scattering probabilities and u* are rounded to (and, where
// they are kept, stored in): double, or float in the FP32-shift form.  There each probability is rounded
// to FP32 once, and every quantity built from it (the rest probability
// rem = 1 - sum s, which stays FP64, u*, P(r,1), VACF(0)) uses the rounded
// value, so the propagator still conserves sum_r P exactly up to FP64 rounding.
template <typename W>
__device__ __forceinline__ double as_coef(double v) {
    return (double)(W)v;
}

// The scattering probability s(r', l') = n_l'/rho - w_l' + lambda w_l' / 2
// (module_moment_propagation.f90:218-228,331-346) of a node r' with density
// rho and flow v = j + f, from its tracer population n_l' = a0 rho + a1 c.v
// (drop_tracers.f90:97-100), rounded as the coefficients are kept (W).  The
// set-up and the recomputing step kernel call this one function, so they get
// the same bits.
template <int L, typename W>
__device__ __forceinline__ double scatter_prob(double rho, double vx, double vy, double vz, double lambda) {
    constexpr int cx = kCX[L], cy = kCY[L], cz = kCZ[L];
    const double nt = a0(L) * rho + a1(L) * dot3<cx, cy, cz>(vx, vy, vz);
    return as_coef<W>(nt / rho - a0(L) + lambda * a0(L) * 0.5);
}

// x / y rounded correctly from r = 1/y rounded correctly (y shared by many
// quotients, so its division is done once): after one correction q is within
// an ulp of x/y, and then q + r (x - y q), its remainder exact in one fused
// multiply-add, rounds to x/y rounded correctly (Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", IBM J. Res.
// Dev. 34, 1990, theorem on the last step of a division).  For y in [2^-400,
// 2^400] and x = 0 or in [2^-900, 2^900] nothing over- or underflows on the way.
__device__ __forceinline__ double quotient(double x, double y, double r) {
    double q = x * r;
    q = __builtin_fma(__builtin_fma(-y, q, x), r, q);
    return __builtin_fma(__builtin_fma(-y, q, x), r, q);
}

// scatter_prob with 1/rho given: the same bits
template <int L, typename W>
__device__ __forceinline__ double scatter_prob(double rho, double rinv, double vx, double vy, double vz, double lambda) {
    constexpr int cx = kCX[L], cy = kCY[L], cz = kCZ[L];
    const double nt = a0(L) * rho + a1(L) * dot3<cx, cy, cz>(vx, vy, vz);
    return as_coef<W>(quotient(nt, rho, rinv) - a0(L) + lambda * a0(L) * 0.5);
}

// Plain streaming copy (16 B per lane per iteration, grid-stride): the
// measured ceiling that the roofline fractions are read against, and the
// known-size kernel that calibrates the HBM traffic counters.
__global__ __launch_bounds__(kBlock) void k_copy(const double2* __restrict__ a, double2* __restrict__ b, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock)
        b[i] = a[i];
}

// The LB step's streams without its gathers: S FP64 planes of n nodes read
// and S written, one node per lane, every load issued before the first store
// (the order of the step's pulls and writes).  Its rate is the ceiling of the
// structure-of-arrays layout itself, below the plain copy's.
template <int S>
__global__ __launch_bounds__(kBlock) void k_planes(const double* __restrict__ in, double* __restrict__ out, uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    double v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = in[(uint64_t)s * n + i];
#pragma unroll
    for (int s = 0; s < S; ++s) out[(uint64_t)s * n + i] = v[s];
}

}  // namespace
