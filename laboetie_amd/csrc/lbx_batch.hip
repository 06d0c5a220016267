// liblbx batch engine: many independent lattices ("instances") resident in
// HBM at once and advanced together, for batched and served solves.
//
// Layout.  All instances share one packed fluid-node list: instance b owns the
// node range [node_off, node_end) (node_off a multiple of 256, so every 128-
// or 256-node tile belongs to one instance) and a range of a shared full-box
// map array.  Populations, flux and density are the single-lattice arrays over
// the whole list (plane stride = the node capacity).  tile_inst[] maps each
// 256-node tile to its instance, and a device table of BInst entries holds
// every instance's geometry, physics and the work of the current round.
// Moment propagation runs on its own tiles (lbx_mp.h), laid out when an
// instance enters it: an instance whose nodes take n tiles of the list from
// tile t on has the 2n tiles from 2t on to itself (a layout never needs more).
//
// One LB launch advances every instance in the LB phase by one step, one MP
// launch every instance in the MP phase; the blocks of other instances leave
// at once.  The per-block work is lb_step_tile / mp_step_tile, the functions
// the single-lattice kernels run, on a per-instance view (its own step index,
// control block, l2err slots, VACF partials), so an instance's results are
// bit-identical to a single-lattice run of the same input.
//
// Phases (host-driven between rounds, as the single-lattice host loop does):
// LB stage 1 -> (redo of the switch step with the force on) -> LB stage 2 ->
// extract + MP prep -> MP steps -> done.
#include <hip/hip_cooperative_groups.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <map>
#include <new>
#include <vector>

#include "../../include/lbx.h"
#include "lbx_block.h"
#include "lbx_device.h"
#include "lbx_kernels.h"
#include "lbx_mp.h"
#include "lbx_nodes.h"
#include "lbx_tables.h"

#pragma clang fp contract(off)

using namespace lbx;

namespace {

constexpr int kTile = 256;                 // allocation unit (nodes) of an instance's range
constexpr uint32_t kNoInst = 0xFFFFFFFFu;
constexpr int kRoundMax = 1024;            // launches per phase per round (vtrace rows)
constexpr size_t kStage = 1u << 20;
constexpr size_t kGraphCacheMax = 64;      // captured round graphs kept at once

struct BInst {
    // geometry (set when the instance is added)
    uint32_t node_off, node_end;  // packed range
    uint32_t tile_first, ntiles;  // 256-node tiles
    uint32_t map_off, lz;
    FastDiv dlx, dly;
    double A, B, C, rho0, target;
    // this round's LB work
    int32_t lb_on, lb_redo;       // takes part; the launch is the redo of step lb_t0 (force switch)
    int64_t lb_t0, lb_n;          // launch k runs step lb_t0 + k while k < lb_n
    int64_t check_after, floor_window;
    int64_t check_base;           // l2err measured at check_base + m check_every (StepArgs)
    int32_t check_every, pad2_;
    double check_inv;             // 1 / check_every
    double fm[3], fc[3];          // F(t)/2 and the collision force (the stage's)
    // this round's MP work
    int32_t mp_on, any_ads;
    int64_t mp_it0, mp_n;         // launch k runs MP step mp_it0 + k + 1 while k < mp_n
    int32_t mp_repeat;            // every launch recomputes step mp_it0 + 1 (timing)
    uint32_t mp_tile0, mp_ntiles; // its MP tiles
    int32_t mp_general;           // its MP steps need the general kernel (lbx_mp.h)
    double lambda;
    TracerParams tp;
    // set-up of its moment propagation: the end of its LB phase (step, F/2), lb.in's f_ext
    int64_t end_t;
    double end_fm[3], F[3];
};

// the control block of an instance at the start of a stage or phase
__device__ __forceinline__ void reset_ctrl(Ctrl* c, int64_t check_after) {
    Ctrl h{};
    h.negpop = -1;
    for (int k = 0; k < 2; ++k) {
        h.l2min[k] = HUGE_VAL;
        h.l2min_step[k] = check_after;
    }
    *c = h;
}

template <typename E, typename R = E>
struct BatchView {
    const BInst* insts;
    const uint32_t* tile_inst;
    const uint32_t* act;          // the 256-node tiles of the instances in the phase, ascending
    E* f0;
    E* f1;
    R* j;                         // the step's flux (FP32-shift: j32)
    const uint32_t* nodes;
    const uint32_t* maps;
    unsigned long long* slots;    // [inst][3][kSlots]
    double* l2ring;               // [inst][kRing]
    Ctrl* ctrl;                   // [inst]
    uint64_t Np;
};

// A launch covers only the tiles of the instances in its phase: logical
// block l of the launch is BLOCK-node tile `active_tile(act, l)`, in the
// 256-node tile act[l / (256/BLOCK)] (instances in the other phase, or done,
// cost no blocks).
template <int BLOCK>
__device__ __forceinline__ uint32_t active_tile(const uint32_t* act, uint32_t l) {
    constexpr uint32_t per = kTile / BLOCK;
    return act[l / per] * per + l % per;
}

// LB launch k of a round on one BLOCK-node tile (a redo repeats step lb_t0);
// NT: population stores with the streaming hint
template <int BLOCK, bool Wide, typename E, typename R = E, bool NT = false>
__device__ __forceinline__ void kb_lb_tile(const BatchView<E, R>& v, uint32_t tile, int64_t k) {
    const uint32_t id = v.tile_inst[tile / (kTile / BLOCK)];
    if (id == kNoInst) return;
    const BInst& in = v.insts[id];
    if (!in.lb_on || k >= in.lb_n) return;
    const int64_t t = in.lb_t0 + (in.lb_redo ? 0 : k);
    StepArgs<E, R> a;
    a.fin = (t - 1) & 1 ? v.f1 : v.f0;
    a.fout = t & 1 ? v.f1 : v.f0;
    a.j = v.j;
    a.nodes = v.nodes;
    a.map = v.maps + in.map_off;
    a.slots = v.slots + (uint64_t)id * 3 * kSlots;
    a.l2ring = v.l2ring + (uint64_t)id * kRing;
    a.ctrl = v.ctrl + id;
    a.dlx = in.dlx;
    a.dly = in.dly;
    a.lz = in.lz;
    a.Nf = in.node_end;
    a.Np = v.Np;
    a.A = (R)in.A;
    a.B = (R)in.B;
    a.C = (R)in.C;
    a.fmx = (R)in.fm[0];
    a.fmy = (R)in.fm[1];
    a.fmz = (R)in.fm[2];
    a.fcx = (R)in.fc[0];
    a.fcy = (R)in.fc[1];
    a.fcz = (R)in.fc[2];
    a.rho0 = (R)in.rho0;
    a.t = t;
    a.check_after = in.check_after;
    a.floor_window = in.floor_window;
    a.target = in.target;
    a.write_l2 = in.lb_redo ? 0 : 1;
    a.have_prev = (!in.lb_redo && t > 1) ? 1 : 0;
    a.check_every = in.check_every;
    a.check_base = in.check_base;
    a.check_inv = (R)in.check_inv;
    const uint32_t first = in.tile_first * (kTile / BLOCK);
    lb_step_tile<BLOCK, Wide, E, R, NT>(a, tile, tile - first, tile == first);
}

template <int BLOCK, bool Wide, typename E, typename R = E, bool NT = false>
__global__ __launch_bounds__(BLOCK, (kLbMinWaves<E, R>)) void kb_lb_step(BatchView<E, R> v, int64_t k) {
    kb_lb_tile<BLOCK, Wide, E, R, NT>(v, active_tile<BLOCK>(v.act, xcd_tile()), k);
}

// l2err of each LB instance's last step of the round (one wave per instance slot)
// (called by the first wave of a block)
__device__ __forceinline__ void kb_lb_finalize_inst(const BInst* insts, unsigned long long* slots, double* l2ring,
                                                    Ctrl* ctrl, uint32_t id) {
    const BInst& in = insts[id];
    if (!in.lb_on || in.lb_redo || in.lb_n <= 0) return;
    lb_finalize(slots + (uint64_t)id * 3 * kSlots, l2ring + (uint64_t)id * kRing, ctrl + id, in.lb_t0 + in.lb_n - 1,
                in.check_base, in.check_every);
}

__global__ __launch_bounds__(64) void kb_lb_finalize(const BInst* insts, unsigned long long* slots, double* l2ring,
                                                     Ctrl* ctrl) {
    kb_lb_finalize_inst(insts, slots, l2ring, ctrl, blockIdx.x);
}

template <typename W>
struct BatchMpView {
    const BInst* insts;
    const uint32_t* tile_inst;    // of each MP tile
    const uint32_t* act;          // the MP tiles of the instances in the phase, the general ones last, each ascending
    MpTiles t;
    MpFields<W> f;
    const uint32_t* nodes;
    const uint32_t* maps;
    double* part[2];              // VACF partials by step parity, 3 per MP tile
    double* vtrace;               // [k][inst][3]
    uint32_t vt_stride;           // instance slots per vtrace row
    Ctrl* ctrl;
};

// MP launch k of a round on one MP tile (mp_repeat: every launch recomputes
// step mp_it0 + 1, for timing).  FP64 recomputes the incoming probabilities,
// the FP32 forms keep them.
template <typename W, bool GEN>
__device__ __forceinline__ void kb_mp_tile(const BatchMpView<W>& v, uint32_t tile, int64_t k, int32_t reduce_prev) {
    const uint32_t id = v.tile_inst[tile];
    if (id == kNoInst) return;
    const BInst& in = v.insts[id];
    if (!in.mp_on || k >= in.mp_n) return;
    const int64_t it = in.mp_it0 + (in.mp_repeat ? 0 : k) + 1;  // P(it) -> P(it+1); P(m) lives in buffer (m-1)&1
    MpStepArgs<W> a;
    a.t = v.t;
    a.fields(v.f, ((it - 1) & 1) != 0);
    a.any_ads = in.any_ads;
    a.partials = it & 1 ? v.part[1] : v.part[0];
    a.prev_partials = (reduce_prev && !in.mp_repeat && k > 0)
                          ? ((it - 1) & 1 ? v.part[1] : v.part[0]) + 3 * (uint64_t)in.mp_tile0
                          : nullptr;
    a.prev_vtrace = v.vtrace + ((uint64_t)(k - 1) * v.vt_stride + id) * 3;
    a.it = it;
    a.lambda = in.lambda;
    a.ctrl = v.ctrl + id;
    a.tp = in.tp;
    a.nodes = v.nodes;
    a.map = v.maps + in.map_off;
    a.dlx = in.dlx;
    a.dly = in.dly;
    a.lz = in.lz;
    if (tile == in.mp_tile0) mp_reduce_prev<1, W>(a, in.mp_ntiles);
    mp_step_tile<1, W, std::is_same<W, double>::value, GEN>(a, tile);
}

template <typename W, bool GEN>
__global__ __launch_bounds__(kBlock, (GEN ? 2 : 4)) void kb_mp_step(BatchMpView<W> v, int64_t k, int32_t reduce_prev) {
    kb_mp_tile<W, GEN>(v, v.act[xcd_tile()], k, reduce_prev);
}

// VACF of an MP instance's last step of the round (one block)
template <typename W>
__device__ __forceinline__ void kb_mp_reduce_inst(const BatchMpView<W>& v, uint32_t id) {
    __shared__ double lds[kBlock / 64 * 3];
    const BInst& in = v.insts[id];
    if (!in.mp_on || in.mp_n <= 0 || in.mp_repeat) return;
    const int64_t it = in.mp_it0 + in.mp_n;
    const double* part = (it & 1 ? v.part[1] : v.part[0]) + 3 * (uint64_t)in.mp_tile0;
    mp_reduce_block<3, kBlock>(part, in.mp_ntiles, v.vtrace + ((uint64_t)(in.mp_n - 1) * v.vt_stride + id) * 3,
                               v.ctrl + id, 1, it, 0, 0.0, 0.0, lds);
}

// (one block per instance slot)
template <typename W>
__global__ __launch_bounds__(kBlock) void kb_mp_reduce_last(BatchMpView<W> v) {
    kb_mp_reduce_inst(v, blockIdx.x);
}

// Admission of one instance in one launch: its nodes at rest and through the
// opening collision of step 1 (k_init_rest, k_collide_packed*: the same
// operations), its tiles' owner, and (first block) its control block, l2err
// slots and ring.
template <typename E, typename R>
__global__ __launch_bounds__(kBlock) void kb_admit(E* f, R* jold, double* __restrict__ rho, double* __restrict__ j,
                                                   BInst in, uint32_t id, uint32_t* __restrict__ tile_inst,
                                                   unsigned long long* __restrict__ slots, double* __restrict__ l2ring,
                                                   Ctrl* ctrl, uint64_t Np, const int8_t* __restrict__ nature,
                                                   uint32_t N, const uint32_t* __restrict__ counts,
                                                   uint32_t* __restrict__ nodes, uint32_t* __restrict__ maps,
                                                   uint32_t* nfi) {
    static_assert(kBlock == kNodeThreads, "one block size");
    if (blockIdx.x * kNodeChunk < N)
        node_chunk(nature, N, counts, blockIdx.x, in.node_off, nodes, maps + in.map_off, nfi + id, in.dlx, in.dly,
                   in.lz);
    if (blockIdx.x >= in.ntiles) return;
    if (threadIdx.x == 0) tile_inst[in.tile_first + blockIdx.x] = id;
    if (blockIdx.x == 0) {
        for (uint32_t k = threadIdx.x; k < 3 * kSlots; k += kBlock) slots[(uint64_t)id * 3 * kSlots + k] = 0ull;
        for (uint32_t k = threadIdx.x; k < (uint32_t)kRing; k += kBlock) l2ring[(uint64_t)id * kRing + k] = 0.0;
        if (threadIdx.x == 0) reset_ctrl(ctrl + id, 2);
    }
    const uint32_t i = in.node_off + blockIdx.x * kBlock + threadIdx.x;
    if (i >= in.node_end) return;
    const R z = R(0);
    rho[i] = in.rho0;
    for (int c = 0; c < 3; ++c) {
        j[c * Np + i] = 0.0;
        jold[c * Np + i] = z;
    }
    const R A = (R)in.A, B = (R)in.B, C = (R)in.C;
    static_for<0, kQ>([&](auto I) {
        constexpr int L = I;
        if constexpr (std::is_same<E, float>::value) {
            const R drho = (R)(in.rho0 - in.rho0), full = (R)in.rho0 + drho;
            R ux, uy, uz;
            shift_velocity<R>(z, z, z, full, ux, uy, uz);
            f[(uint64_t)L * Np + i] = (float)collide_shift<L, R>(z, drho, z, z, z, ux, uy, uz, z, z, z, A, B, C);
        } else {
            const double d = in.rho0, u = 0.0 / d;
            f[(uint64_t)L * Np + i] = collide_pop<L>(d * a0(L), d, 0.0, 0.0, 0.0, u, u, u, 0.0, 0.0, 0.0, A, B, C);
        }
    });
}

// A removed instance's tiles and interfacial count.
__global__ __launch_bounds__(kBlock) void kb_release(uint32_t* __restrict__ tile_inst, uint32_t n, uint32_t* nfi) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) tile_inst[i] = kNoInst;
    if (i == 0) *nfi = 0;
}

// out[k] = l2ring[at[k]]
__global__ __launch_bounds__(kBlock) void kb_pick_l2(const double* __restrict__ l2ring, const uint64_t* __restrict__ at,
                                                     uint32_t n, double* __restrict__ out) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k < n) out[k] = l2ring[at[k]];
}

// The post-streaming state, density and flux at the end of the LB phase of
// the instances whose 256-node tiles are listed in v.act
template <typename E>
__global__ __launch_bounds__(kBlock) void kb_extract(BatchView<E, E> v, double* rho, double* j) {
    const uint32_t tile = v.act[blockIdx.x];
    const BInst& in = v.insts[v.tile_inst[tile]];
    const uint32_t i = tile * kTile + threadIdx.x;
    if (i >= in.node_end || in.end_t <= 0) return;
    Neighbours nb;
    nb.load(v.maps + in.map_off, v.nodes[i] & kIndexMask, in.dlx, in.dly, in.lz);
    const E* src = (in.end_t - 1) & 1 ? v.f1 : v.f0;
    E* dst = in.end_t & 1 ? v.f1 : v.f0;
    if constexpr (std::is_same<E, float>::value)
        extract_node_shift(src, dst, rho, j, nb, i, v.Np, in.rho0, in.end_fm[0], in.end_fm[1], in.end_fm[2]);
    else
        extract_node(src, dst, rho, nb, i, v.Np);
}

// control blocks of the instances ids, as their moment propagation starts
__global__ __launch_bounds__(64) void kb_reset_ctrl(Ctrl* ctrl, const uint32_t* __restrict__ ids, uint32_t n) {
    const uint32_t k = blockIdx.x * 64 + threadIdx.x;
    if (k < n) reset_ctrl(ctrl + ids[k], 2);
}

// mp_prep_tile on the MP tiles listed in v.act
template <typename W>
__global__ __launch_bounds__(kBlock) void kb_mp_prep(BatchMpView<W> v, const double* rho, const double* j, uint64_t Np,
                                                     double eps) {
    const uint32_t tile = v.act[xcd_tile()];
    const uint32_t id = v.tile_inst[tile];
    const BInst& in = v.insts[id];
    MpPrepArgs<W> a;
    a.t = v.t;
    a.f = v.f;
    a.rho = rho;
    a.j = j;
    a.nodes = v.nodes;
    a.map = v.maps + in.map_off;
    a.partials = v.part[0];
    a.ctrl = v.ctrl + id;
    a.dlx = in.dlx;
    a.dly = in.dly;
    a.lz = in.lz;
    a.Np = Np;
    a.fx = in.F[0];
    a.fy = in.F[1];
    a.fz = in.F[2];
    a.lambda = in.lambda;
    a.eps = eps;
    a.tp = in.tp;
    mp_prep_tile<1, W>(a, tile);
}

// VACF(0) of the instances ids (one block each)
template <typename W>
__global__ __launch_bounds__(kBlock) void kb_mp_vacf0(BatchMpView<W> v, const uint32_t* __restrict__ ids) {
    __shared__ double lds[kBlock / 64 * 3];
    const uint32_t id = ids[blockIdx.x];
    const BInst& in = v.insts[id];
    mp_reduce_block<3, kBlock>(v.part[0] + 3 * (uint64_t)in.mp_tile0, in.mp_ntiles, nullptr, v.ctrl + id, 0, 0, 0, 0.0,
                               0.0, lds);
}

// The steps of one phase of a round in one cooperative launch: every block
// loops over its share of the tiles with a grid-wide barrier between steps,
// then the closing reduction.  The per-tile work and its order of partial sums
// are those of the per-step launches, so the results are the same bits.  Every
// block runs every barrier: the loops have grid-uniform bounds and the
// per-tile functions only return from the tile, never from the kernel.
// f(l) for this block's share of the logical tiles: the tiles of XCD x
// (blocks b = x mod 8) are one contiguous range
template <typename F>
__device__ __forceinline__ void block_share(uint32_t ntiles, F&& f) {
    const uint32_t nb = gridDim.x, b = blockIdx.x, x = b & 7u, local = b >> 3;
    const uint32_t nblk = (nb >> 3) + (x < (nb & 7u) ? 1u : 0u);
    const uint32_t per = (ntiles + 7u) / 8u;
    const uint32_t t0 = x * per, t1 = min(ntiles, t0 + per);
    for (uint32_t l = t0 + local; l < t1; l += nblk) f(l);
}

template <int BLOCK, bool Wide, typename E, typename R>
__global__ __launch_bounds__(BLOCK) void kb_lb_round(BatchView<E, R> v, int64_t S, uint32_t ntiles, uint32_t ninst,
                                                     int32_t redo_only) {
    cooperative_groups::grid_group grid = cooperative_groups::this_grid();
    for (int64_t k = 0; k < S; ++k) {
        block_share(ntiles, [&](uint32_t l) { kb_lb_tile<BLOCK, Wide, E, R>(v, active_tile<BLOCK>(v.act, l), k); });
        grid.sync();
    }
    if (redo_only) return;
    for (uint32_t id = blockIdx.x; id < ninst; id += gridDim.x)
        if (threadIdx.x < 64) kb_lb_finalize_inst(v.insts, v.slots, v.l2ring, v.ctrl, id);
}

template <typename W, bool GEN>
__global__ __launch_bounds__(kBlock, (GEN ? 2 : 4)) void kb_mp_round(BatchMpView<W> v, int64_t S, uint32_t ntiles,
                                                                     uint32_t ninst) {
    cooperative_groups::grid_group grid = cooperative_groups::this_grid();
    for (int64_t k = 0; k < S; ++k) {
        block_share(ntiles, [&](uint32_t l) { kb_mp_tile<W, GEN>(v, v.act[l], k, 1); });
        grid.sync();
    }
    for (uint32_t id = blockIdx.x; id < ninst; id += gridDim.x)
        if ((v.insts[id].mp_general != 0) == GEN) kb_mp_reduce_inst(v, id);  // those that this launch stepped
}

// ------------------------------------------------------------------ host

// first-fit allocator of [0, cap) in units
struct RangeAlloc {
    std::map<uint64_t, uint64_t> free_;  // start -> length
    void init(uint64_t cap) {
        free_.clear();
        if (cap) free_[0] = cap;
    }
    bool take(uint64_t n, uint64_t* start) {
        for (auto it = free_.begin(); it != free_.end(); ++it)
            if (it->second >= n) {
                *start = it->first;
                const uint64_t rest = it->second - n, s = it->first + n;
                free_.erase(it);
                if (rest) free_[s] = rest;
                return true;
            }
        return false;
    }
    void give(uint64_t start, uint64_t n) {
        auto it = free_.emplace(start, n).first;
        auto nx = std::next(it);
        if (nx != free_.end() && it->first + it->second == nx->first) {
            it->second += nx->second;
            free_.erase(nx);
        }
        if (it != free_.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) {
                pv->second += it->second;
                free_.erase(it);
            }
        }
    }
    uint64_t largest() const {
        uint64_t m = 0;
        for (auto& kv : free_) m = std::max(m, kv.second);
        return m;
    }
};

enum Phase : int32_t { kFree = 0, kLb = 1, kRedo = 2, kLbDone = 3, kMp = 4, kDone = 5, kFailed = 6 };

struct HostInst {
    Phase phase = kFree;
    int32_t status = LBX_OK;
    int32_t lx = 0, ly = 0, lz = 0, stage = 1, exit_reason = 0;
    uint32_t N = 0, Nf = 0;
    uint64_t map_n = 0;
    double F[3] = {0, 0, 0};
    double Db = 0, ka = 0, kd = 0, lambda = 0;
    int64_t t = 0, max_lb = 0, switch_step = INT64_MAX, check_after = 2;
    int64_t mp_it = 0, mp_target = 0;
    std::vector<double> vacf;       // (mp_it+1) x 3
    double deff[3] = {0, 0, 0};
};

}  // namespace

struct lbxb {
    int32_t prec = LBX_PREC_FP64;
    bool wide = false;       // 64-bit addressing of the population buffers
    bool wide_auto = false;  // what the capacity alone selects
    uint64_t Np = 0, cap_box = 0;
    uint32_t cap_inst = 0, ntiles_cap = 0;
    int32_t lb_block = 256, mp_block = 256;
    bool graphs = true;
    bool persistent = false;  // a round's launches of each phase as one cooperative launch
    int32_t num_cu = 0;
    int32_t check_every = kCheckEvery;  // FP32 storage: stage-2 steps between l2err measurements
    int64_t floor_window = 1000;        // FP32 storage: l2err floor test of the instances added from now on
    hipStream_t stream = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    // device arrays
    double* f[2] = {nullptr, nullptr};
    float* g[2] = {nullptr, nullptr};
    float* j32 = nullptr;
    double* j = nullptr;
    double* rho = nullptr;
    uint32_t* nodes = nullptr;
    uint32_t* maps = nullptr;
    uint32_t* tile_inst = nullptr;
    int8_t* nature = nullptr;    // of the instance being admitted
    uint32_t* counts = nullptr;  // its fluid nodes by chunk (lbx_nodes.h)
    uint32_t* nfi = nullptr;     // interfacial nodes of each instance
    BInst* insts = nullptr;
    unsigned long long* slots = nullptr;
    double* l2ring = nullptr;
    Ctrl* ctrl = nullptr;
    MpTiles mpt;                 // MP tiles: 2 ntiles_cap
    uint32_t* mp_tile_inst = nullptr;
    MpFields<double> mpf;        // FP64 form
    MpFields<float> mpf32;       // FP32-storage forms
    uint32_t *walk_count = nullptr, *walk_base = nullptr;  // scratch of the layout builds, grown as needed
    Block block, walk_block;     // the allocations: all arrays above and below, the scratch
    uint32_t* ids = nullptr;     // [max instances]
    // admissions go through two pinned buffers in turn (kStage bytes each)
    char* stage[2] = {nullptr, nullptr};
    hipEvent_t stage_ev[2] = {nullptr, nullptr};
    int stage_at = 0;
    MpBuild* builds = nullptr;   // [max instances]
    MpBuilt* built = nullptr;
    uint8_t* split = nullptr;    // layout builds: parts of each tile (log2)
    double* part[2] = {nullptr, nullptr};
    double* vtrace = nullptr;
    // host state
    std::vector<BInst> tab;
    std::vector<Ctrl> ctrl_h;  // per instance slot: what reset_inst_ctrl uploads (kept until the stream syncs)
    std::vector<HostInst> hi;
    std::vector<uint32_t> mp_tile_inst_h;
    // the tiles of the instances with LB (0) or MP (1) work in the launches
    // about to run (built by upload_active; host copy kept until the stream syncs)
    uint32_t* act[2] = {nullptr, nullptr};
    std::vector<uint32_t> act_h[2];
    uint32_t n_act[2] = {0, 0};
    uint32_t n_gen = 0;       // general MP tiles, the last of act[1]
    RangeAlloc node_alloc, map_alloc;
    // graphs of a round's launches, keyed by (phase, launches)
    struct Graph {
        hipGraphExec_t exec = nullptr;
        int32_t block = 0;
        uint32_t grid_tiles = 0;  // active tiles of the phase
        uint32_t gen_tiles = 0;   // ... of the general kernel
    };
    std::map<std::pair<int, int64_t>, Graph> graph_cache;
    // statistics
    double lb_ms = 0, mp_ms = 0;
    int64_t lb_box_updates = 0, lb_fluid_updates = 0, mp_box_updates = 0, mp_fluid_updates = 0;
};

namespace {

void clear_graphs(lbxb* b) {
    for (auto& kv : b->graph_cache)
        if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
    b->graph_cache.clear();
}

void free_all(lbxb* b) {
    clear_graphs(b);
    give_block(&b->block);
    give_block(&b->walk_block);
    for (int k = 0; k < 2; ++k) {
        if (b->stage[k]) (void)hipHostFree(b->stage[k]);
        if (b->stage_ev[k]) (void)hipEventDestroy(b->stage_ev[k]);
        b->stage[k] = nullptr;
        b->stage_ev[k] = nullptr;
    }
    for (auto& e : b->ev)
        if (e) (void)hipEventDestroy(e), e = nullptr;
    if (b->stream) (void)hipStreamDestroy(b->stream), b->stream = nullptr;
}

// populations stored as FP32 deviations (FP32-shift and FP32-store forms);
// their moment propagation keeps its probabilities in FP32
bool shift(const lbxb* b) { return b->prec == LBX_PREC_FP32_SHIFT || b->prec == LBX_PREC_FP32_STORE; }

// The upload reads the batch's ctrl_h[id], which no other call changes before
// the stream has synchronised (an instance is reset at most once between two
// synchronisations).
int reset_inst_ctrl(lbxb* b, uint32_t id, int64_t check_after) {
    Ctrl& h = b->ctrl_h[id];
    h = Ctrl{};
    h.negpop = -1;
    for (int k = 0; k < 2; ++k) {
        h.l2min[k] = HUGE_VAL;
        h.l2min_step[k] = check_after;
    }
    return hip_status(hipMemcpyAsync(b->ctrl + id, &h, sizeof(Ctrl), hipMemcpyHostToDevice, b->stream));
}

// blocks of a launch: LB tiles are cut into blocks, MP tiles are one block each
uint32_t grid_of(const lbxb* b, int block, int phase /*0 LB, 1 MP*/) {
    return phase == 0 ? b->n_act[0] * (kTile / block) : b->n_act[1];
}

// The active tile lists of the work table as it stands (lb_on / mp_on), for
// the launches that follow; call after the table changes which instances take
// part and before those launches.
int upload_active(lbxb* b) {
    LBX_TRY(hipStreamSynchronize(b->stream));  // the previous lists' uploads have been read
    for (int ph = 0; ph < 2; ++ph) {
        // (first tile, tiles) of the phase's instances, those of the general MP kernel last
        std::vector<std::pair<uint32_t, uint32_t>> r, gen;
        for (uint32_t id = 0; id < b->cap_inst; ++id) {
            const BInst& in = b->tab[id];
            if (ph == 0 && in.lb_on) r.emplace_back(in.tile_first, in.ntiles);
            if (ph == 1 && in.mp_on) (in.mp_general ? gen : r).emplace_back(in.mp_tile0, in.mp_ntiles);
        }
        std::sort(r.begin(), r.end());
        std::sort(gen.begin(), gen.end());
        uint32_t n_gen = 0;
        for (const auto& x : gen) n_gen += x.second;
        if (ph == 1) b->n_gen = n_gen;
        r.insert(r.end(), gen.begin(), gen.end());
        std::vector<uint32_t>& a = b->act_h[ph];
        a.clear();
        for (const auto& x : r)
            for (uint32_t t = 0; t < x.second; ++t) a.push_back(x.first + t);
        b->n_act[ph] = (uint32_t)a.size();
        if (!a.empty())
            LBX_TRY(hipMemcpyAsync(b->act[ph], a.data(), a.size() * sizeof(uint32_t), hipMemcpyHostToDevice,
                                   b->stream));
    }
    return LBX_OK;
}

template <typename E, typename R = E>
BatchView<E, R> lb_view(lbxb* b) {
    BatchView<E, R> v;
    v.insts = b->insts;
    v.tile_inst = b->tile_inst;
    v.act = b->act[0];
    if constexpr (std::is_same<E, float>::value) {
        v.f0 = b->g[0];
        v.f1 = b->g[1];
        if constexpr (std::is_same<R, float>::value) v.j = b->j32; else v.j = b->j;
    } else {
        v.f0 = b->f[0];
        v.f1 = b->f[1];
        v.j = b->j;
    }
    v.nodes = b->nodes;
    v.maps = b->maps;
    v.slots = b->slots;
    v.l2ring = b->l2ring;
    v.ctrl = b->ctrl;
    v.Np = b->Np;
    return v;
}

template <typename W>
MpFields<W>& mp_fields(lbxb* b) {
    if constexpr (std::is_same<W, float>::value) return b->mpf32; else return b->mpf;
}

template <typename W>
BatchMpView<W> mp_view(lbxb* b) {
    BatchMpView<W> v;
    v.insts = b->insts;
    v.tile_inst = b->mp_tile_inst;
    v.act = b->act[1];
    v.t = b->mpt;
    v.f = mp_fields<W>(b);
    v.nodes = b->nodes;
    v.maps = b->maps;
    v.part[0] = b->part[0];
    v.part[1] = b->part[1];
    v.vtrace = b->vtrace;
    v.vt_stride = b->cap_inst;
    v.ctrl = b->ctrl;
    return v;
}

// f(std::integral_constant<int, B>{}) for the block size B of a launch (64, 128 or 256 nodes)
template <typename F>
void with_block(int block, F&& f) {
    if (block == 64)
        f(std::integral_constant<int, 64>{});
    else if (block == 128)
        f(std::integral_constant<int, 128>{});
    else
        f(std::integral_constant<int, 256>{});
}

// the LB kernel of one launch: addressing form, and streaming stores when the
// active tiles' two population sets outgrow the last-level cache (a function
// of the active tile count, which a cached graph's validity already checks)
template <int BL, typename E, typename R = E>
auto lb_kernel(const lbxb* b) {
    const bool nt = 2ull * kQ * b->n_act[0] * kTile * sizeof(E) > (uint64_t)LBX_NT_MIN_BYTES;
    if (b->wide) return nt ? kb_lb_step<BL, true, E, R, true> : kb_lb_step<BL, true, E, R>;
    return nt ? kb_lb_step<BL, false, E, R, true> : kb_lb_step<BL, false, E, R>;
}

// launch LB step k of a round over the tiles of the instances with LB work
void launch_lb(lbxb* b, int64_t k, int block) {
    const uint32_t grid = grid_of(b, block, 0);
    if (!grid) return;
    with_block(block, [&](auto BT) {
        constexpr int BL = decltype(BT)::value;
        if (b->prec == LBX_PREC_FP32_SHIFT) {
            auto v = lb_view<float>(b);
            hipLaunchKernelGGL((lb_kernel<BL, float>(b)), dim3(grid), dim3(BL), 0, b->stream, v, k);
        } else if (b->prec == LBX_PREC_FP32_STORE) {
            auto v = lb_view<float, double>(b);
            hipLaunchKernelGGL((lb_kernel<BL, float, double>(b)), dim3(grid), dim3(BL), 0, b->stream, v, k);
        } else {
            auto v = lb_view<double>(b);
            hipLaunchKernelGGL((lb_kernel<BL, double>(b)), dim3(grid), dim3(BL), 0, b->stream, v, k);
        }
    });
}

// MP step k of a round: one launch for the instances on brick tiles, and one
// for those that need the general kernel (236 VGPRs and 65 KB of LDS in FP64,
// two waves per SIMD: two 128x128x96 boxes 112 us a step, 213 when a small
// general instance beside them took them to it, 130 with a launch of its own)
void launch_mp(lbxb* b, int64_t k, int reduce_prev) {
    auto go = [&](auto wtag) {
        using W = decltype(wtag);
        BatchMpView<W> v = mp_view<W>(b);
        const uint32_t n = b->n_act[1] - b->n_gen;
        if (n) hipLaunchKernelGGL((kb_mp_step<W, false>), dim3(n), dim3(kBlock), 0, b->stream, v, k, reduce_prev);
        v.act += n;
        if (b->n_gen)
            hipLaunchKernelGGL((kb_mp_step<W, true>), dim3(b->n_gen), dim3(kBlock), 0, b->stream, v, k, reduce_prev);
    };
    if (shift(b))
        go(float{});
    else
        go(double{});
}

void launch_lb_finalize(lbxb* b) {
    hipLaunchKernelGGL(kb_lb_finalize, dim3(b->cap_inst), dim3(64), 0, b->stream, b->insts, b->slots, b->l2ring,
                       b->ctrl);
}

void launch_mp_reduce_last(lbxb* b) {
    if (shift(b))
        hipLaunchKernelGGL(kb_mp_reduce_last<float>, dim3(b->cap_inst), dim3(kBlock), 0, b->stream, mp_view<float>(b));
    else
        hipLaunchKernelGGL(kb_mp_reduce_last<double>, dim3(b->cap_inst), dim3(kBlock), 0, b->stream,
                           mp_view<double>(b));
}

// the S launches of one phase of a round (+ its closing reduction), replayed
// from a captured graph when graphs are on
int run_phase(lbxb* b, int phase /*0 LB, 1 MP*/, int64_t S) {
    if (S <= 0) return LBX_OK;
    const int block = phase == 0 ? b->lb_block : kBlock;
    auto emit = [&]() {
        for (int64_t k = 0; k < S; ++k) {
            if (phase == 0)
                launch_lb(b, k, block);
            else
                launch_mp(b, k, 1);
        }
        if (phase == 0)
            launch_lb_finalize(b);
        else
            launch_mp_reduce_last(b);
    };
    if (!b->graphs) {
        emit();
        return hip_status(hipGetLastError());
    }
    auto key = std::make_pair(phase, S);
    auto it = b->graph_cache.find(key);
    const uint32_t gen = phase == 1 ? b->n_gen : 0;
    if (it != b->graph_cache.end() &&
        (it->second.block != block || it->second.grid_tiles != b->n_act[phase] || it->second.gen_tiles != gen)) {
        (void)hipGraphExecDestroy(it->second.exec);
        b->graph_cache.erase(it);
        it = b->graph_cache.end();
    }
    if (it == b->graph_cache.end()) {
        // one graph per (phase, round length): bounded by the callers' round
        // sizes, but callers that vary them freely would grow the cache; start
        // over past a few dozen entries
        if (b->graph_cache.size() >= kGraphCacheMax) clear_graphs(b);
        hipGraph_t graph = nullptr;
        LBX_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        emit();
        const hipError_t ce = hipStreamEndCapture(b->stream, &graph);
        if (ce != hipSuccess) return hip_status(ce);
        lbxb::Graph gr;
        const hipError_t ie = hipGraphInstantiate(&gr.exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ie != hipSuccess) return hip_status(ie);
        gr.block = block;
        gr.grid_tiles = b->n_act[phase];
        gr.gen_tiles = gen;
        it = b->graph_cache.emplace(key, gr).first;
    }
    return hip_status(hipGraphLaunch(it->second.exec, b->stream));
}

// One phase of a round as a single cooperative launch (grid: blocks that are
// resident at once, at most one per tile)
int run_phase_persistent(lbxb* b, int phase, int64_t S, int32_t redo_only) {
    if (S <= 0) return LBX_OK;
    uint32_t nt = grid_of(b, b->lb_block, phase), ni = b->cap_inst;
    if (!nt) return LBX_OK;
    auto launch = [&](auto kern, uint32_t tiles, int block, void** args) -> int {
        int per_cu = 0;
        LBX_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, block, 0));
        if (per_cu <= 0) return LBX_ERR_DEVICE;
        // 8 waves a CU: the grid barrier's time grows with the blocks, faster than more of them
        // save.  LB + MP us per step of 256-thread blocks, all that fit / 2 / 1 a CU: six 96^3 media
        // FP64 538 + 298 / 421 + 267 / 454 + 358, FP32-shift 567 + 327 / 340 + 248 / 389 + 279;
        // 64 cells 1x100x100 FP64 185 + 143 / 117 + 86 / 94 + 77
        per_cu = std::min(per_cu, 512 / block);
        const uint32_t grid = std::min<uint32_t>(tiles, (uint32_t)per_cu * (uint32_t)b->num_cu);
        return hip_status(hipLaunchCooperativeKernel((const void*)kern, dim3(grid), dim3(block), args, 0, b->stream));
    };
    if (phase == 1) {
        auto go = [&](auto wtag) -> int {
            using W = decltype(wtag);
            BatchMpView<W> v = mp_view<W>(b);
            uint32_t ngen = b->n_gen;
            nt -= ngen;
            void* args[] = {&v, &S, &nt, &ni};
            if (nt) LBX_TRY(launch(kb_mp_round<W, false>, nt, kBlock, args));
            v.act += nt;
            void* gargs[] = {&v, &S, &ngen, &ni};
            return ngen ? launch(kb_mp_round<W, true>, ngen, kBlock, gargs) : LBX_OK;
        };
        return shift(b) ? go(float{}) : go(double{});
    }
    auto go = [&](auto etag, auto rtag, auto btag) -> int {
        using E = decltype(etag);  // population storage
        using R = decltype(rtag);  // LB arithmetic
        constexpr int BL = decltype(btag)::value;
        BatchView<E, R> v = lb_view<E, R>(b);
        void* args[] = {&v, &S, &nt, &ni, &redo_only};
        return launch(b->wide ? kb_lb_round<BL, true, E, R> : kb_lb_round<BL, false, E, R>, nt, BL, args);
    };
    int st = LBX_OK;
    with_block(b->lb_block, [&](auto BT) {
        if (b->prec == LBX_PREC_FP32_SHIFT)
            st = go(float{}, float{}, BT);
        else if (b->prec == LBX_PREC_FP32_STORE)
            st = go(float{}, double{}, BT);
        else
            st = go(double{}, double{}, BT);
    });
    return st;
}

template <typename T>
int download(lbxb* b, const T* src, uint64_t count, T* dst) {
    LBX_TRY(hipMemcpyAsync(dst, src, count * sizeof(T), hipMemcpyDeviceToHost, b->stream));
    return hip_status(hipStreamSynchronize(b->stream));
}

// MP layouts of the instances ids, built together (lbx_mp.h; as build_tiles of
// the single-lattice path, so an instance gets the same tiles there and here)
int build_tiles(lbxb* b, const std::vector<uint32_t>& ids) {
    std::vector<MpBuild> builds(ids.size());
    std::vector<MpBuilt> built(ids.size());
    std::vector<Bricks> halves(ids.size());
    uint64_t walk = 0;
    for (size_t k = 0; k < ids.size(); ++k) {
        const HostInst& h = b->hi[ids[k]];
        const BInst& in = b->tab[ids[k]];
        MpBuild& d = builds[k];
        d = MpBuild{};
        d.b = make_bricks((uint32_t)h.lx, (uint32_t)h.ly, (uint32_t)h.lz);
        halves[k] = make_bricks((uint32_t)h.lx, (uint32_t)h.ly, (uint32_t)h.lz, true);
        d.nodes = b->nodes;
        d.map = b->maps + in.map_off;
        d.dlx = in.dlx;
        d.dly = in.dly;
        d.order_off = (uint32_t)walk;
        d.tile0 = 2 * in.tile_first;
        d.bound = (uint32_t)mp_tile_bound(h.Nf);  // 2 in.ntiles
        d.serial = 1;
        walk += std::max(d.b.norder, halves[k].norder);
    }
    LBX_TRY(take_block(&b->walk_block, [&](auto&& take) {
        take(b->walk_count, walk);
        take(b->walk_base, walk);
    }, true));
    uint32_t *count = b->walk_count, *base = b->walk_base;
    constexpr uint32_t kGridY = 65535;        // lattices of one launch at most,
    constexpr uint64_t kEmptyBlocks = 65536;  // and its empty blocks
    std::vector<MpBuilt> counts_h;            // read until the stream has synchronised
    const auto counted = [&](const std::vector<size_t>& which) -> const std::vector<MpBuilt>& {
        counts_h.clear();
        for (size_t k : which) counts_h.push_back(built[k]);
        return counts_h;
    };
    const auto size_of = [&](size_t k) { return std::max((uint64_t)builds[k].b.norder, (uint64_t)builds[k].bound); };
    // one pass over the lattices `which`: their tiles, cut by split where `cut`;
    // marks (in split) those whose halo is too large where `mark`; general: keep
    // what has an LDS slot
    auto pass = [&](std::vector<size_t>& which, bool cut, bool mark, bool general) -> int {
        // largest first; a launch's grid is the largest lattice's for each, so it ends
        // before its empty blocks get to be many, and at a grid's rows
        std::stable_sort(which.begin(), which.end(), [&](size_t x, size_t y) { return size_of(x) > size_of(y); });
        std::vector<MpBuild> d;
        for (size_t k : which) d.push_back(builds[k]);
        const uint32_t nd = (uint32_t)d.size();
        // f(first, lattices, blocks for one wave a brick, blocks for one a tile) per launch
        const auto slices = [&](auto&& f) {
            for (uint32_t s0 = 0, s1; s0 < nd; s0 = s1) {
                uint32_t gw = 0, gt = 0;
                uint64_t empty = 0;
                for (s1 = s0; s1 < nd && s1 - s0 < kGridY; ++s1) {
                    empty += size_of(which[s0]) - size_of(which[s1]);
                    if (empty > kEmptyBlocks) break;
                    gw = std::max(gw, (d[s1].b.norder + kBlock / 64 - 1) / (kBlock / 64));
                    gt = std::max(gt, d[s1].bound);
                }
                f(s0, s1 - s0, gw, gt);
            }
        };
        LBX_TRY(hipMemcpyAsync(b->builds, d.data(), nd * sizeof(MpBuild), hipMemcpyHostToDevice, b->stream));
        if (cut)  // by the last pass's tiles, of lattices in another order there: their counts once more
            LBX_TRY(hipMemcpyAsync(b->built, counted(which).data(), nd * sizeof(MpBuilt), hipMemcpyHostToDevice,
                                   b->stream));
        slices([&](uint32_t s0, uint32_t n, uint32_t gw, uint32_t gt) {
            if (cut)
                hipLaunchKernelGGL(k_mpb_parts, dim3(gt, n), dim3(kBlock), 0, b->stream, b->builds + s0,
                                   b->built + s0, base, b->mpt, b->split);
            else if (!general)
                hipLaunchKernelGGL(k_mpb_count, dim3(gw, n), dim3(kBlock), 0, b->stream, b->builds + s0, count);
        });
        hipLaunchKernelGGL(k_mpb_group, dim3(nd), dim3(kBlock), 0, b->stream, b->builds, b->built, count, base,
                           b->mpt.info, cut ? b->split : nullptr);
        slices([&](uint32_t s0, uint32_t n, uint32_t gw, uint32_t gt) {
            hipLaunchKernelGGL(k_mpb_place, dim3(gw, n), dim3(kBlock), 0, b->stream, b->builds + s0, b->built + s0,
                               base, b->mpt.perm, b->mpt.inv);
            hipLaunchKernelGGL((general ? k_mpb_table<true> : k_mpb_table<false>), dim3(gt, n), dim3(kBlock), 0,
                               b->stream, b->builds + s0, b->built + s0, b->mpt, mark ? b->split : nullptr);
        });
        LBX_TRY(hipGetLastError());
        std::vector<MpBuilt> r(nd);
        LBX_TRY(hipMemcpyAsync(r.data(), b->built, nd * sizeof(MpBuilt), hipMemcpyDeviceToHost, b->stream));
        LBX_TRY(hipStreamSynchronize(b->stream));
        for (uint32_t k = 0; k < nd; ++k) built[which[k]] = r[k];
        return LBX_OK;
    };
    // the layouts of the lattices `which`; those that take more than their bound of tiles go to `beyond`
    std::vector<size_t> gen;
    auto settle = [&](std::vector<size_t> which, std::vector<size_t>* beyond) -> int {
        if (which.empty()) return LBX_OK;
        LBX_TRY(pass(which, false, true, false));
        std::vector<size_t> cut;
        for (size_t k : which)
            if (built[k].ntiles == 0)
                beyond->push_back(k);
            else if (built[k].halo_max > kHaloMax)
                cut.push_back(k);
        if (cut.empty()) return LBX_OK;
        LBX_TRY(pass(cut, true, false, false));
        for (size_t k : cut)
            if (built[k].ntiles == 0) beyond->push_back(k);
        return LBX_OK;
    };
    std::vector<size_t> some(ids.size()), whole;
    for (size_t k = 0; k < ids.size(); ++k) some[k] = k;
    LBX_TRY(settle(some, &gen));
    some.clear();
    for (size_t k = 0; k < ids.size(); ++k)
        if (halves[k].inner > 1 && built[k].ntiles > 0 && try_halves(built[k].ntiles, b->hi[ids[k]].Nf))
            some.push_back(k);
    std::vector<MpBuild> was = builds;
    for (size_t k : some) {
        builds[k].b = halves[k];
        builds[k].bound = halves_bound(built[k].ntiles);
        builds[k].serial = 0;
    }
    LBX_TRY(settle(some, &whole));
    for (size_t k : whole) builds[k] = was[k];
    LBX_TRY(settle(whole, &gen));
    if (!gen.empty()) LBX_TRY(pass(gen, false, false, true));
    for (size_t k = 0; k < ids.size(); ++k) {
        BInst& in = b->tab[ids[k]];
        in.mp_tile0 = 2 * in.tile_first;
        in.mp_ntiles = built[k].ntiles;
        for (uint32_t t = 0; t < 2 * in.ntiles; ++t)
            b->mp_tile_inst_h[in.mp_tile0 + t] = t < in.mp_ntiles ? ids[k] : kNoInst;
    }
    LBX_TRY(hipMemcpyAsync(b->mp_tile_inst, b->mp_tile_inst_h.data(), b->mp_tile_inst_h.size() * sizeof(uint32_t),
                           hipMemcpyHostToDevice, b->stream));
    for (size_t k : gen) b->tab[ids[k]].mp_general = 1;
    return LBX_OK;
}

// extract + MP layout + prep + VACF(0) of the instances ids, whose LB phases
// have ended: one launch of each for all of them (one per instance, a few
// blocks at a time, took 50 ms for 1024 2-D instances)
int mp_setup_insts(lbxb* b, const std::vector<uint32_t>& ids) {
    if (ids.empty()) return LBX_OK;
    LBX_TRY(build_tiles(b, ids));
    const double eps = DBL_EPSILON;
    std::vector<uint32_t> nfi(b->cap_inst);
    LBX_TRY(download(b, b->nfi, b->cap_inst, nfi.data()));
    for (BInst& in : b->tab) in.lb_on = in.mp_on = 0;
    for (uint32_t id : ids) {
        HostInst& h = b->hi[id];
        BInst& in = b->tab[id];
        TracerParams tp{};
        const double K = (std::fabs(h.kd) <= eps) ? 0.0 : h.ka / h.kd;  // module_moment_propagation.f90:46-50
        tp.ads[0] = std::fabs(K) > eps;                                 // :52-56
        tp.bw[0] = 1.0 / ((double)h.Nf + K * (double)nfi[id]);            // :97
        tp.ka[0] = h.ka;
        tp.kd[0] = h.kd;
        tp.one_minus_kd[0] = 1.0 - h.kd;
        in.tp = tp;
        in.any_ads = tp.ads[0];
        in.lambda = h.lambda;
        in.end_t = h.t;
        for (int a = 0; a < 3; ++a) {
            in.F[a] = h.F[a];
            in.end_fm[a] = h.t > h.switch_step ? h.F[a] / 2.0 : 0.0;
        }
        in.lb_on = in.mp_on = 1;  // the tiles of both lists
    }
    LBX_TRY(hipMemcpyAsync(b->insts, b->tab.data(), b->tab.size() * sizeof(BInst), hipMemcpyHostToDevice, b->stream));
    LBX_TRY(hipMemcpyAsync(b->ids, ids.data(), ids.size() * sizeof(uint32_t), hipMemcpyHostToDevice, b->stream));
    LBX_TRY(upload_active(b));
    const uint32_t n = (uint32_t)ids.size();
    auto go = [&](auto wtag) {
        using W = decltype(wtag);
        const BatchMpView<W> v = mp_view<W>(b);
        BatchView<W, W> lv = lb_view<W, W>(b);
        hipLaunchKernelGGL(kb_extract<W>, dim3(b->n_act[0]), dim3(kBlock), 0, b->stream, lv, b->rho, b->j);
        hipLaunchKernelGGL(kb_reset_ctrl, dim3((n + 63) / 64), dim3(64), 0, b->stream, b->ctrl, b->ids, n);
        hipLaunchKernelGGL(kb_mp_prep<W>, dim3(b->n_act[1]), dim3(kBlock), 0, b->stream, v, b->rho, b->j, b->Np, eps);
        hipLaunchKernelGGL(kb_mp_vacf0<W>, dim3(n), dim3(kBlock), 0, b->stream, v, b->ids);
    };
    if (shift(b))
        go(float{});
    else
        go(double{});
    for (BInst& in : b->tab) in.lb_on = in.mp_on = 0;
    LBX_TRY(hipGetLastError());
    std::vector<Ctrl> ctrl(b->cap_inst);
    LBX_TRY(download(b, b->ctrl, b->cap_inst, ctrl.data()));
    for (uint32_t id : ids) {
        HostInst& h = b->hi[id];
        const Ctrl& c = ctrl[id];
        if (c.restpart) {
            h.phase = kFailed;
            h.status = LBX_ERR_RESTPART;
            continue;
        }
        if (!shift(b) && c.mp_divide) b->tab[id].mp_general = 1;
        h.vacf.assign(c.vacf0, c.vacf0 + 3);
        h.mp_it = 0;
        h.phase = h.mp_target > 0 ? kMp : kDone;
        if (h.phase == kDone)
            for (int a_ = 0; a_ < 3; ++a_) h.deff[a_] = c.deff_s[a_] + c.deff_c[a_];
    }
    return LBX_OK;
}

void set_capacity(lbxb* b, int32_t precision, int64_t nodes, int64_t box, int32_t instances) {
    b->prec = precision;
    b->Np = ((uint64_t)nodes + kTile - 1) / kTile * kTile;
    b->cap_box = (uint64_t)box;
    b->cap_inst = (uint32_t)instances;
    b->ntiles_cap = (uint32_t)(b->Np / kTile);
    b->mpt.pitch = kHaloMaxGen;
}

// all device arrays of a batch
template <typename Take>
void batch_arrays(lbxb* b, Take&& take) {
    const uint64_t Np = b->Np, tiles = Np / kTile, ni = b->cap_inst;
    const uint64_t M = 2 * Np;  // entries of the MP tiles
    for (int k = 0; k < 2; ++k)
        if (shift(b)) take(b->g[k], kQ * Np); else take(b->f[k], kQ * Np);
    if (b->prec == LBX_PREC_FP32_SHIFT) take(b->j32, 3 * Np);
    take(b->j, 3 * Np);
    take(b->rho, Np);
    take(b->nodes, Np);
    take(b->maps, b->cap_box);
    take(b->tile_inst, tiles);
    take(b->nature, (b->cap_box + 15) / 16 * 16);
    take(b->counts, (b->cap_box + kNodeChunk - 1) / kNodeChunk);
    take(b->nfi, ni);
    take(b->act[0], tiles);
    take(b->act[1], 2 * tiles);
    take(b->insts, ni);
    take(b->slots, ni * 3 * kSlots);
    take(b->l2ring, ni * kRing);
    take(b->ctrl, ni);
    const auto fields = [&](auto& f) {
        take(f.rem, M);
        take(f.ustar, 3 * M);
        for (int k = 0; k < 2; ++k) {
            take(f.P[k], 3 * M);
            take(f.Pa[k], 3 * M);
        }
    };
    if (shift(b)) {
        fields(b->mpf32);
        take(b->mpf32.win, 9 * M);
    } else {
        fields(b->mpf);
        take(b->mpf.rv, 2 * M);
    }
    for (int k = 0; k < 2; ++k) take(b->part[k], 2 * tiles * 3);
    take(b->mpt.info, M / kTile);
    take(b->mpt.halo, M / kTile * b->mpt.pitch);
    take(b->mpt.tab4, M);
    take(b->mpt.tab2, M);
    take(b->mpt.perm, M);
    take(b->mpt.inv, Np);
    take(b->mp_tile_inst, M / kTile);
    take(b->split, M / kTile);
    take(b->builds, ni);
    take(b->built, ni);
    take(b->ids, ni);
    take(b->vtrace, (uint64_t)kRoundMax * ni * 3);
}

}  // namespace

// ------------------------------------------------------------------ C-ABI

extern "C" {

int64_t lbxb_footprint_bytes(int32_t precision, int64_t capacity_nodes, int64_t capacity_box, int32_t max_instances) {
    if (capacity_nodes <= 0 || capacity_box <= 0 || max_instances <= 0) return -1;
    lbxb b;
    set_capacity(&b, precision, capacity_nodes, capacity_box, max_instances);
    return (int64_t)block_bytes([&](auto&& take) { batch_arrays(&b, take); });
}

int lbxb_create(int32_t precision, int64_t capacity_nodes, int64_t capacity_box, int32_t max_instances,
                lbxb** out) {
    if (!out) return LBX_ERR_ARG;
    *out = nullptr;
    if (precision != LBX_PREC_FP64 && precision != LBX_PREC_FP32_SHIFT && precision != LBX_PREC_FP32_STORE)
        return LBX_ERR_ARG;
    if (capacity_nodes <= 0 || capacity_box <= 0 || max_instances <= 0) return LBX_ERR_ARG;
    const uint64_t Np = ((uint64_t)capacity_nodes + kTile - 1) / kTile * kTile;
    if (kQ * Np >= (1ull << 32) || (uint64_t)capacity_box >= (1ull << 32)) return LBX_ERR_ARG;
    lbxb* b = new (std::nothrow) lbxb();
    if (!b) return LBX_ERR_NOMEM;
    set_capacity(b, precision, capacity_nodes, capacity_box, max_instances);
    // 32-bit byte offsets reach every array while the populations (the
    // largest: 19 per node, FP64 or FP32 by form) stay below 4 GiB
    b->wide = b->wide_auto =
        (uint64_t)kQ * Np * (precision == LBX_PREC_FP64 ? sizeof(double) : sizeof(float)) >= (1ull << 32);
    {
        int dev = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&b->num_cu, hipDeviceAttributeMultiprocessorCount, dev);
    }
    int st = LBX_OK;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) st = LBX_ERR_DEVICE;
    if (!st) st = take_block(&b->block, [&](auto&& take) { batch_arrays(b, take); });
    for (int k = 0; k < 2; ++k) {
        if (!st) st = hip_status(hipHostMalloc((void**)&b->stage[k], kStage));
        if (!st) st = hip_status(hipEventCreateWithFlags(&b->stage_ev[k], hipEventDisableTiming));
    }
    if (!st && (hipEventCreate(&b->ev[0]) != hipSuccess || hipEventCreate(&b->ev[1]) != hipSuccess))
        st = LBX_ERR_DEVICE;
    if (!st) {
        b->tab.assign(max_instances, BInst{});
        b->ctrl_h.assign(max_instances, Ctrl{});
        b->hi.assign(max_instances, HostInst{});
        b->mp_tile_inst_h.assign(2 * (size_t)b->ntiles_cap, kNoInst);
        b->node_alloc.init(b->ntiles_cap);
        b->map_alloc.init(b->cap_box);
        st = hip_status(hipMemsetAsync(b->tile_inst, 0xFF, b->ntiles_cap * sizeof(uint32_t), b->stream));  // kNoInst
        if (!st) st = hip_status(hipMemsetAsync(b->nfi, 0, b->cap_inst * sizeof(uint32_t), b->stream));
    }
    if (!st) st = hip_status(hipMemcpyAsync(b->insts, b->tab.data(), b->tab.size() * sizeof(BInst),
                                            hipMemcpyHostToDevice, b->stream));
    if (!st) st = hip_status(hipStreamSynchronize(b->stream));
    if (st) {
        free_all(b);
        delete b;
        return st;
    }
    *out = b;
    return LBX_OK;
}

int lbxb_destroy(lbxb* b) {
    if (!b) return LBX_ERR_ARG;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    free_all(b);
    delete b;
    return LBX_OK;
}

int lbxb_add(lbxb* b, int32_t lx, int32_t ly, int32_t lz, const int8_t* nature, double tau, double rho0,
             const double fext[3], double target_error, int64_t max_lb_steps, double Db, double ka, double kd,
             int64_t mp_steps, int32_t* id_out) {
    if (!b || !nature || !fext || !id_out || lx <= 0 || ly <= 0 || lz <= 0 || mp_steps < 0 || max_lb_steps < 0)
        return LBX_ERR_ARG;
    *id_out = -1;
    if (!(tau >= 0.5)) return LBX_ERR_TAU;
    const double eps = DBL_EPSILON;
    if (ka < -eps || kd < -eps || !(Db > eps)) return LBX_ERR_ARG;
    const uint64_t N = (uint64_t)lx * ly * lz;
    if (N >= (1ull << 29)) return LBX_ERR_ARG;
    uint32_t id = 0;
    while (id < b->cap_inst && b->hi[id].phase != kFree) ++id;
    if (id == b->cap_inst) return LBX_ERR_NOMEM;
    HostInst h;
    h.Nf = count_fluid(nature, N);
    if (h.Nf == 0) return LBX_ERR_ARG;
    const uint64_t ntiles = (h.Nf + kTile - 1) / kTile;
    uint64_t tile0 = 0, map0 = 0;
    if (!b->node_alloc.take(ntiles, &tile0)) return LBX_ERR_NOMEM;  // HBM admission
    if (!b->map_alloc.take(N, &map0)) {
        b->node_alloc.give(tile0, ntiles);
        return LBX_ERR_NOMEM;
    }
    h.lx = lx;
    h.ly = ly;
    h.lz = lz;
    h.N = (uint32_t)N;
    h.map_n = N;
    for (int a = 0; a < 3; ++a) h.F[a] = fext[a];
    h.Db = Db;
    h.ka = ka;
    h.kd = kd;
    h.lambda = 4.0 * Db / kKbt;  // calc_lambda, module_moment_propagation.f90:331-337
    h.max_lb = max_lb_steps;
    h.mp_target = mp_steps;
    h.phase = kLb;
    BInst in{};
    in.node_off = (uint32_t)(tile0 * kTile);
    in.node_end = in.node_off + h.Nf;
    in.tile_first = (uint32_t)tile0;
    in.ntiles = (uint32_t)ntiles;
    in.map_off = (uint32_t)map0;
    in.lz = (uint32_t)lz;
    in.dlx.set((uint32_t)lx);
    in.dly.set((uint32_t)ly);
    in.A = 1.0 - 1.0 / tau;  // module_collision.f90:99-101
    in.B = 1.0 / tau;
    in.C = 1.0 - 1.0 / (2.0 * tau);
    if (b->prec == LBX_PREC_FP32_SHIFT) {  // FP32 collision: A + B = 1 exactly
        float a32, b32;
        fp32_relaxation(tau, &a32, &b32);
        in.A = a32;
        in.B = b32;
    }
    in.check_every = 1;
    in.check_base = 0;
    in.check_inv = 1.0;
    in.rho0 = rho0;
    in.target = target_error;
    in.floor_window = shift(b) ? b->floor_window : 0;
    // the nature, through a pinned buffer where it fits, so that the call needs no wait
    const bool staged = N <= kStage;
    const int at = b->stage_at;
    int st = staged ? hip_status(hipEventSynchronize(b->stage_ev[at])) : LBX_OK;
    if (staged) std::memcpy(b->stage[at], nature, N);
    if (!st) st = hip_status(hipMemcpyAsync(b->nature, staged ? (const void*)b->stage[at] : (const void*)nature, N,
                                            hipMemcpyHostToDevice, b->stream));
    const uint32_t chunks = node_chunks(N);
    if (!st && chunks > kNodeCountChunks)
        hipLaunchKernelGGL(k_node_count, dim3(chunks), dim3(kNodeThreads), 0, b->stream, b->nature, (uint32_t)N,
                           b->counts);
    // node list, map (global packed indices), rest state and the opening collision of step 1 (no force)
    if (!st) {
        auto admit = [&](auto* f, auto* jold) {
            using E = std::remove_pointer_t<decltype(f)>;
            using R = std::remove_pointer_t<decltype(jold)>;
            hipLaunchKernelGGL((kb_admit<E, R>), dim3(std::max<uint32_t>((uint32_t)ntiles, chunks)), dim3(kBlock), 0,
                               b->stream, f, jold, b->rho, b->j, in, id, b->tile_inst, b->slots, b->l2ring, b->ctrl,
                               b->Np, b->nature, (uint32_t)N, chunks > kNodeCountChunks ? b->counts : nullptr,
                               b->nodes, b->maps, b->nfi);
        };
        if (b->prec == LBX_PREC_FP32_SHIFT)
            admit(b->g[0], b->j32);
        else if (b->prec == LBX_PREC_FP32_STORE)
            admit(b->g[0], b->j);  // j_old is j itself
        else
            admit(b->f[0], b->j);
        st = hip_status(hipGetLastError());
    }
    if (!st && staged) st = hip_status(hipEventRecord(b->stage_ev[at], b->stream));
    if (staged) b->stage_at ^= 1;
    if (!st && !staged) st = hip_status(hipStreamSynchronize(b->stream));  // the nature is the caller's
    if (st) {
        b->node_alloc.give(tile0, ntiles);
        b->map_alloc.give(map0, N);
        return st;
    }
    b->tab[id] = in;
    b->hi[id] = std::move(h);
    *id_out = (int32_t)id;
    return LBX_OK;
}

int lbxb_remove(lbxb* b, int32_t id) {
    if (!b || id < 0 || (uint32_t)id >= b->cap_inst || b->hi[id].phase == kFree) return LBX_ERR_ARG;
    // no wait: what follows on the stream finds the tiles free
    BInst& in = b->tab[id];
    hipLaunchKernelGGL(kb_release, dim3((in.ntiles + kBlock - 1) / kBlock), dim3(kBlock), 0, b->stream, b->tile_inst + in.tile_first,
                       in.ntiles, b->nfi + id);
    b->node_alloc.give(in.tile_first, in.ntiles);
    b->map_alloc.give(in.map_off, b->hi[id].map_n);
    b->hi[id] = HostInst{};
    in = BInst{};
    return hip_status(hipGetLastError());
}

// One round: redo launches of instances whose stage 1 ended, lb_steps LB
// launches, mp_steps MP launches, then the host bookkeeping (stage switches,
// ends of the LB phase -> MP set-up, ends of the MP phase).
int lbxb_round(lbxb* b, int32_t lb_steps, int32_t mp_steps, int32_t* active) {
    if (!b || lb_steps < 0 || mp_steps < 0 || lb_steps > kRoundMax || mp_steps > kRoundMax) return LBX_ERR_ARG;
    const uint32_t ni = b->cap_inst;
    const double zero[3] = {0.0, 0.0, 0.0};
    // 1. redo of the switch step (equilibration.f90:377-386), with the force on
    bool any_redo = false;
    for (uint32_t id = 0; id < ni; ++id) {
        BInst& in = b->tab[id];
        in.lb_on = in.mp_on = 0;
        HostInst& h = b->hi[id];
        if (h.phase != kRedo) continue;
        any_redo = true;
        LBX_TRY(reset_inst_ctrl(b, id, h.t));
        in.lb_on = 1;
        in.lb_redo = 1;
        in.lb_t0 = h.t;
        in.lb_n = 1;
        in.check_after = INT64_MAX;
        for (int a = 0; a < 3; ++a) {
            in.fm[a] = zero[a] / 2.0;
            in.fc[a] = h.F[a];
        }
        h.stage = 2;
        h.switch_step = h.t;
        h.check_after = h.t;
        h.phase = kLb;
    }
    if (any_redo) {
        LBX_TRY(hipMemcpyAsync(b->insts, b->tab.data(), ni * sizeof(BInst), hipMemcpyHostToDevice, b->stream));
        LBX_TRY(upload_active(b));
        launch_lb(b, 0, b->lb_block);
        LBX_TRY(hipGetLastError());
        LBX_TRY(hipStreamSynchronize(b->stream));  // the table upload has been read
        for (uint32_t id = 0; id < ni; ++id) b->tab[id].lb_on = 0, b->tab[id].lb_redo = 0;
    }
    // 2. this round's work table
    int64_t lb_box = 0, lb_fluid = 0, mp_box = 0, mp_fluid = 0;
    int64_t S_lb = 0, S_mp = 0;
    for (uint32_t id = 0; id < ni; ++id) {
        BInst& in = b->tab[id];
        HostInst& h = b->hi[id];
        if (h.phase == kLb && lb_steps > 0) {
            int64_t n = lb_steps;
            if (h.max_lb > 0) n = std::min<int64_t>(n, h.max_lb - h.t);
            if (n <= 0) continue;
            in.lb_on = 1;
            in.lb_redo = 0;
            in.lb_t0 = h.t + 1;
            in.lb_n = n;
            in.check_after = h.check_after;
            // l2err of every step in stage 1; in stage 2 of the FP32 storage
            // forms every kCheckEvery steps from the force switch
            in.check_every = (h.stage == 2 && shift(b)) ? b->check_every : 1;
            in.check_base = h.stage == 2 ? h.switch_step : 0;
            in.check_inv = 1.0 / in.check_every;
            for (int a = 0; a < 3; ++a) {
                const double F = h.stage == 1 ? 0.0 : h.F[a];
                in.fm[a] = F / 2.0;
                in.fc[a] = F;
            }
            S_lb = std::max(S_lb, n);
        } else if (h.phase == kMp && mp_steps > 0) {
            const int64_t n = std::min<int64_t>(mp_steps, h.mp_target - h.mp_it);
            if (n <= 0) continue;
            in.mp_on = 1;
            in.mp_it0 = h.mp_it;
            in.mp_n = n;
            S_mp = std::max(S_mp, n);
        }
    }
    LBX_TRY(hipMemcpyAsync(b->insts, b->tab.data(), ni * sizeof(BInst), hipMemcpyHostToDevice, b->stream));
    LBX_TRY(upload_active(b));
    if (S_lb > 0) {
        LBX_TRY(hipEventRecord(b->ev[0], b->stream));
        LBX_TRY(b->persistent ? run_phase_persistent(b, 0, S_lb, 0) : run_phase(b, 0, S_lb));
        LBX_TRY(hipEventRecord(b->ev[1], b->stream));
        LBX_TRY(hipEventSynchronize(b->ev[1]));
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, b->ev[0], b->ev[1]);
        b->lb_ms += ms;
    }
    if (S_mp > 0) {
        LBX_TRY(hipEventRecord(b->ev[0], b->stream));
        LBX_TRY(b->persistent ? run_phase_persistent(b, 1, S_mp, 0) : run_phase(b, 1, S_mp));
        LBX_TRY(hipEventRecord(b->ev[1], b->stream));
        LBX_TRY(hipEventSynchronize(b->ev[1]));
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, b->ev[0], b->ev[1]);
        b->mp_ms += ms;
    }
    // 3. bookkeeping
    std::vector<Ctrl> ctrl(ni);
    LBX_TRY(download(b, b->ctrl, ni, ctrl.data()));
    std::vector<double> vt;
    if (S_mp > 0) {
        vt.resize((size_t)S_mp * ni * 3);
        LBX_TRY(download(b, b->vtrace, vt.size(), vt.data()));
    }
    std::vector<uint32_t> to_mp, capped;
    for (uint32_t id = 0; id < ni; ++id) {
        BInst& in = b->tab[id];
        HostInst& h = b->hi[id];
        const Ctrl& c = ctrl[id];
        if (in.lb_on) {
            int64_t last = in.lb_t0 + in.lb_n - 1;
            if (c.negpop >= 0) last = std::min<int64_t>(last, c.negpop);
            if (c.stop) last = std::min<int64_t>(last, c.exit_step);
            lb_box += (last - h.t) * (int64_t)h.N;
            lb_fluid += (last - h.t) * (int64_t)h.Nf;
            if (c.negpop >= 0) {
                h.phase = kFailed;
                h.status = LBX_ERR_NEG_POP;
                h.t = c.negpop;
            } else if (c.stop) {
                h.t = c.exit_step;
                if (h.stage == 1) {
                    h.phase = kRedo;
                } else {
                    h.exit_reason = c.floor_hit ? LBX_EXIT_FLOOR : LBX_EXIT_CONVERGED;
                    h.phase = kLbDone;
                }
            } else {
                h.t = last;
                if (h.max_lb > 0 && h.t >= h.max_lb) {
                    capped.push_back(id);
                    h.phase = kLbDone;
                }
            }
            if (h.phase == kLbDone) to_mp.push_back(id);
        } else if (in.mp_on) {
            mp_box += in.mp_n * (int64_t)h.N;
            mp_fluid += in.mp_n * (int64_t)h.Nf;
            for (int64_t k = 0; k < in.mp_n; ++k)
                for (int a = 0; a < 3; ++a) h.vacf.push_back(vt[((size_t)k * ni + id) * 3 + a]);
            h.mp_it += in.mp_n;
            if (h.mp_it >= h.mp_target) {
                h.phase = kDone;
                for (int a = 0; a < 3; ++a) h.deff[a] = c.deff_s[a] + c.deff_c[a];
            }
        }
        in.lb_on = in.mp_on = 0;
    }
    if (!capped.empty()) {  // l2err of their last step, all in one copy (one per instance took 15 ms for 1024)
        const uint32_t n = (uint32_t)capped.size();
        std::vector<uint64_t> at;
        for (uint32_t id : capped) at.push_back((uint64_t)id * kRing + (uint64_t)(b->hi[id].t % kRing));
        uint64_t* at_d = (uint64_t*)b->vtrace + n;  // of kRoundMax x 3 per instance, read above
        std::vector<double> l2(n);
        LBX_TRY(hipMemcpyAsync(at_d, at.data(), n * sizeof(uint64_t), hipMemcpyHostToDevice, b->stream));
        hipLaunchKernelGGL(kb_pick_l2, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, b->stream, b->l2ring, at_d, n, b->vtrace);
        LBX_TRY(hipGetLastError());
        LBX_TRY(download(b, b->vtrace, n, l2.data()));
        for (uint32_t k = 0; k < n; ++k) {
            HostInst& h = b->hi[capped[k]];
            h.exit_reason = (h.stage == 2 && h.t > h.check_after && l2[k] <= b->tab[capped[k]].target)
                                ? LBX_EXIT_CONVERGED
                                : LBX_EXIT_CAP;
        }
    }
    b->lb_box_updates += lb_box;
    b->lb_fluid_updates += lb_fluid;
    b->mp_box_updates += mp_box;
    b->mp_fluid_updates += mp_fluid;
    LBX_TRY(mp_setup_insts(b, to_mp));
    int32_t n = 0;
    for (uint32_t id = 0; id < ni; ++id) n += b->hi[id].phase >= kLb && b->hi[id].phase <= kMp;
    if (active) *active = n;
    return hip_status(hipStreamSynchronize(b->stream));
}

int lbxb_info(lbxb* b, int32_t id, int32_t* phase, int32_t* status, int64_t* lb_steps, int32_t* exit_reason,
              int64_t* mp_steps_done) {
    if (!b || id < 0 || (uint32_t)id >= b->cap_inst) return LBX_ERR_ARG;
    const HostInst& h = b->hi[id];
    if (phase) *phase = h.phase;
    if (status) *status = h.status;
    if (lb_steps) *lb_steps = h.t;
    if (exit_reason) *exit_reason = h.exit_reason;
    if (mp_steps_done) *mp_steps_done = h.mp_it;
    return LBX_OK;
}

int lbxb_result(lbxb* b, int32_t id, double deff[3], double* vacf, int64_t vacf_rows, double* rho, double* jx,
                double* jy, double* jz) {
    if (!b || id < 0 || (uint32_t)id >= b->cap_inst || b->hi[id].phase == kFree) return LBX_ERR_ARG;
    const HostInst& h = b->hi[id];
    const BInst& in = b->tab[id];
    if (deff)
        for (int a = 0; a < 3; ++a) deff[a] = h.deff[a];
    if (vacf) {
        const int64_t rows = std::min<int64_t>(vacf_rows, (int64_t)h.vacf.size() / 3);
        std::memcpy(vacf, h.vacf.data(), (size_t)rows * 3 * sizeof(double));
    }
    // flow fields of the instance (valid once its LB phase has ended)
    double* dst[4] = {rho, jx, jy, jz};
    std::vector<uint32_t> nodes;
    if (rho || jx || jy || jz) {
        nodes.resize(h.Nf);
        LBX_TRY(download(b, b->nodes + in.node_off, h.Nf, nodes.data()));
    }
    for (int k = 0; k < 4; ++k) {
        if (!dst[k]) continue;
        std::vector<double> tmp(h.Nf);
        const double* src = k == 0 ? b->rho + in.node_off : b->j + (uint64_t)(k - 1) * b->Np + in.node_off;
        LBX_TRY(download(b, src, h.Nf, tmp.data()));
        std::memset(dst[k], 0, (size_t)h.N * sizeof(double));
        for (uint32_t i = 0; i < h.Nf; ++i) dst[k][nodes[i] & kIndexMask] = tmp[i];
    }
    return LBX_OK;
}

int lbxb_set_block(lbxb* b, int32_t lb_block, int32_t mp_block) {
    auto ok = [](int32_t x) { return x == 64 || x == 128 || x == 256; };
    if (!b || !ok(lb_block) || !ok(mp_block)) return LBX_ERR_ARG;
    b->lb_block = lb_block;
    b->mp_block = mp_block;
    return LBX_OK;
}

int lbxb_set_check_interval(lbxb* b, int32_t steps) {
    if (!b || steps < 1 || steps > 4096 || (steps & (steps - 1)) != 0) return LBX_ERR_ARG;
    if (steps != 1 && !shift(b)) return LBX_ERR_ARG;
    b->check_every = steps;
    return LBX_OK;
}

int lbxb_set_floor_window(lbxb* b, int64_t steps) {
    if (!b || steps < 0) return LBX_ERR_ARG;
    if (steps > 0 && !shift(b)) return LBX_ERR_ARG;
    b->floor_window = steps;
    return LBX_OK;
}

int lbxb_set_launch_mode(lbxb* b, int32_t mode) {
    if (!b || mode < LBXB_LAUNCH_STREAM || mode > LBXB_LAUNCH_PERSISTENT) return LBX_ERR_ARG;
    b->graphs = mode == LBXB_LAUNCH_GRAPH;
    b->persistent = mode == LBXB_LAUNCH_PERSISTENT;
    if (!b->graphs) clear_graphs(b);
    return LBX_OK;
}

int lbxb_set_addressing(lbxb* b, int32_t wide) {
    if (!b || wide < 0 || wide > 1) return LBX_ERR_ARG;
    b->wide = b->wide_auto || wide == 1;
    clear_graphs(b);  // captured launches name the kernels of the previous form
    return LBX_OK;
}

int lbxb_addressing(lbxb* b) { return b ? (b->wide ? 1 : 0) : -1; }

int lbxb_launch_mode(lbxb* b) {
    if (!b) return -1;
    return b->persistent ? LBXB_LAUNCH_PERSISTENT : (b->graphs ? LBXB_LAUNCH_GRAPH : LBXB_LAUNCH_STREAM);
}

// The autotuner's search space: the block size of the LB launches (64, 128 or
// 256 nodes, i.e. 1, 2 or 4 waves per block and 4, 2 or 1 blocks per
// 256-node tile; an MP launch has one block a tile) and the launch mode of the
// rounds (one launch per step, the same launches replayed from a captured
// graph, or one cooperative persistent launch per phase).  Every point is timed
// on the current state without changing it: LB launches redo each LB instance's
// last completed step (same inputs, same outputs), MP launches recompute its
// last MP step without the VACF reduction.  The fastest LB block size is kept,
// then the mode with the least LB + MP time at that size; mp_block stays as it
// is.  times[LBXB_AUTOTUNE_TIMES] (may be NULL): mean ms per step of LB-64,
// LB-128, LB-256, MP three times (per-step launches), LB-graph, MP-graph,
// LB-persistent, MP-persistent (0 when a phase had no instance to time).
int lbxb_autotune(lbxb* b, int32_t launches, int32_t* lb_block, int32_t* mp_block, double* times) {
    if (!b || launches <= 0) return LBX_ERR_ARG;
    const uint32_t ni = b->cap_inst;
    constexpr int kSizes = 3;
    const int sizes[kSizes] = {64, 128, 256};
    double tm[kSizes] = {0, 0, 0}, tmp = 0;  // LB by block size, MP
    bool any[2] = {false, false};
    for (uint32_t id = 0; id < ni; ++id) {
        BInst& in = b->tab[id];
        const HostInst& h = b->hi[id];
        in.lb_on = in.mp_on = 0;
        if (h.phase == kLb && h.t >= 1) {
            in.lb_on = 1;
            in.lb_redo = 1;  // write_l2 = 0: recompute step t, slots and control untouched
            in.lb_t0 = h.t;
            in.lb_n = 1;
            in.check_after = INT64_MAX;
            const bool on = h.stage == 2 && h.t > h.switch_step;
            for (int a = 0; a < 3; ++a) {
                in.fm[a] = (on ? h.F[a] : 0.0) / 2.0;
                in.fc[a] = h.stage == 2 ? h.F[a] : 0.0;
            }
            any[0] = true;
        } else if (h.phase == kMp && h.mp_it >= 1) {
            in.mp_on = 1;
            in.mp_it0 = h.mp_it - 1;  // recompute step mp_it
            in.mp_n = 1;
            any[1] = true;
        }
    }
    LBX_TRY(hipMemcpyAsync(b->insts, b->tab.data(), ni * sizeof(BInst), hipMemcpyHostToDevice, b->stream));
    LBX_TRY(upload_active(b));
    auto launch = [&](int phase, int block) {
        if (phase == 0) launch_lb(b, 0, block); else launch_mp(b, 0, 0);
    };
    auto elapsed = [&](double* out) -> int {
        LBX_TRY(hipEventRecord(b->ev[1], b->stream));
        LBX_TRY(hipEventSynchronize(b->ev[1]));
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, b->ev[0], b->ev[1]);
        *out = ms / launches;
        return LBX_OK;
    };
    // per-step launches: LB with every block size, MP
    auto timed = [&](int phase, int block, double* out) -> int {
        launch(phase, block);  // warm
        LBX_TRY(hipEventRecord(b->ev[0], b->stream));
        for (int32_t k = 0; k < launches; ++k) launch(phase, block);
        return elapsed(out);
    };
    int best = 0;
    for (int k = 0; any[0] && k < kSizes; ++k) {
        LBX_TRY(timed(0, sizes[k], &tm[k]));
        if (tm[k] < tm[best]) best = k;
    }
    if (any[0]) b->lb_block = sizes[best];
    if (any[1]) LBX_TRY(timed(1, kBlock, &tmp));
    // the same launches replayed from a captured graph
    double tg[2] = {0, 0};
    for (int phase = 0; phase < 2; ++phase) {
        if (!any[phase]) continue;
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        LBX_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        for (int32_t k = 0; k < launches; ++k) launch(phase, b->lb_block);
        const hipError_t ce = hipStreamEndCapture(b->stream, &graph);
        if (ce != hipSuccess) return hip_status(ce);
        const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ie != hipSuccess) return hip_status(ie);
        int st = hip_status(hipGraphLaunch(exec, b->stream));  // warm
        if (!st) st = hip_status(hipEventRecord(b->ev[0], b->stream));
        if (!st) st = hip_status(hipGraphLaunch(exec, b->stream));
        if (!st) st = elapsed(&tg[phase]);
        (void)hipStreamSynchronize(b->stream);
        (void)hipGraphExecDestroy(exec);
        LBX_TRY(st);
    }
    // one cooperative launch of `launches` repeated steps per phase
    double tp[2] = {0, 0};
    for (uint32_t id = 0; id < ni; ++id) {
        BInst& in = b->tab[id];
        if (in.lb_on) in.lb_n = launches;  // lb_redo: every launch recomputes step t
        if (in.mp_on) in.mp_n = launches, in.mp_repeat = 1;
    }
    LBX_TRY(hipStreamSynchronize(b->stream));
    LBX_TRY(hipMemcpyAsync(b->insts, b->tab.data(), ni * sizeof(BInst), hipMemcpyHostToDevice, b->stream));
    for (int phase = 0; phase < 2; ++phase) {
        if (!any[phase]) continue;
        LBX_TRY(run_phase_persistent(b, phase, 1, 1));  // warm
        LBX_TRY(hipEventRecord(b->ev[0], b->stream));
        LBX_TRY(run_phase_persistent(b, phase, launches, 1));
        LBX_TRY(elapsed(&tp[phase]));
    }
    for (uint32_t id = 0; id < ni; ++id) {
        BInst& in = b->tab[id];
        in.lb_on = in.mp_on = in.lb_redo = in.mp_repeat = 0;
    }
    LBX_TRY(hipMemcpyAsync(b->insts, b->tab.data(), ni * sizeof(BInst), hipMemcpyHostToDevice, b->stream));
    // the launch mode with the least time over the timed phases
    if (any[0] || any[1]) {
        const double t_stream = tm[best] + tmp, t_graph = tg[0] + tg[1], t_pers = tp[0] + tp[1];
        b->persistent = t_pers < t_graph && t_pers < t_stream;
        b->graphs = !b->persistent && t_graph <= t_stream;
    }
    clear_graphs(b);
    if (lb_block) *lb_block = b->lb_block;
    if (mp_block) *mp_block = b->mp_block;
    if (times) {
        for (int k = 0; k < kSizes; ++k) {
            times[k] = tm[k];
            times[kSizes + k] = tmp;
        }
        times[6] = tg[0];
        times[7] = tg[1];
        times[8] = tp[0];
        times[9] = tp[1];
    }
    return hip_status(hipStreamSynchronize(b->stream));
}

int lbxb_stats(lbxb* b, double* lb_ms, int64_t* lb_box_updates, int64_t* lb_fluid_updates, double* mp_ms,
               int64_t* mp_box_updates, int64_t* mp_fluid_updates) {
    if (!b) return LBX_ERR_ARG;
    if (lb_ms) *lb_ms = b->lb_ms;
    if (lb_box_updates) *lb_box_updates = b->lb_box_updates;
    if (lb_fluid_updates) *lb_fluid_updates = b->lb_fluid_updates;
    if (mp_ms) *mp_ms = b->mp_ms;
    if (mp_box_updates) *mp_box_updates = b->mp_box_updates;
    if (mp_fluid_updates) *mp_fluid_updates = b->mp_fluid_updates;
    return LBX_OK;
}

int64_t lbxb_free_tiles(lbxb* b) {
    if (!b) return -1;
    return (int64_t)b->node_alloc.largest();
}

}  // extern "C"
