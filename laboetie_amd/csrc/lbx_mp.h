// Moment propagation of liblbx on tiles of spatially compact nodes, shared by
// the single-lattice path (lbx.hip) and the batch engine (lbx_batch.hip).
//
// The box is cut into bricks of at most 256 box nodes (8 x 4 x 8 where the
// box allows it).  A tile is one 256-thread block's share: the fluid nodes of
// one brick, or of consecutive bricks together while they hold at most 256.
// A node's 18 neighbours then lie in its own tile or in the shell around its
// bricks (the tile's halo, listed once per tile), so a step reads every value
// a tile needs once (2.3 node values per node on porous media), stages it in
// LDS, and takes all 18 neighbours from there through 10-bit LDS slots laid
// out once per geometry.
//
// Per-node arrays of the propagation are stored tile by tile: node `lane` of
// tile k is entry 256 k + lane, whatever its place in the packed node list of
// the LB kernels (perm and inv translate).  Tiles that are not full leave
// their last entries unused.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "lbx_kernels.h"

#pragma clang fp contract(off)

namespace {

using namespace lbx;

constexpr uint32_t kMpTile = 256;                // nodes (and threads) of a tile
constexpr uint32_t kZeroSlot = 256;              // LDS slot of the solid neighbour: P = 0
constexpr uint32_t kHalo0 = 257;                 // LDS slot of the first halo node
constexpr uint32_t kFarSlot = 1023;              // neighbour without an LDS slot (general tiles only)
constexpr uint32_t kHaloMax = 344;               // halo nodes of one brick at most (shell of 8 x 4 x 8)
constexpr uint32_t kHaloMaxGen = kFarSlot - kHalo0;  // halo nodes of a general tile at most
constexpr uint32_t kSlots1 = 608;                // LDS slots of a tile with at most kHaloMax halo nodes
constexpr uint32_t kSlotsGen = 1024;
constexpr uint32_t kTabInterfacial = 1u << 31;   // table bits: the node is interfacial,
constexpr uint32_t kTabNode = 1u << 30;          // the entry holds a node
static_assert(kHalo0 + kHaloMax <= kSlots1, "slots of a brick tile");
constexpr int kPace = 3;                         // neighbours whose LDS reads are in flight together
constexpr uint32_t kColumn = 8;                  // bricks are walked in columns of 8 by 8 bricks along z

// A lattice's cut into bricks.
struct Bricks {
    uint32_t lx, ly, lz;
    uint32_t bx, by, bz;      // box nodes of a brick
    uint32_t nbx, nby, nbz;   // bricks per axis
    uint32_t cx, cy;          // bricks of a column along x, y
    uint32_t ncx;             // columns along x
    uint32_t inner;           // bricks along z that are walked together
    uint32_t norder;          // entries of the walk (places outside the box hold no nodes)
};

// halves: the bricks are cut in two along z, the two walked one after the other.
inline Bricks make_bricks(uint32_t lx, uint32_t ly, uint32_t lz, bool halves = false) {
    Bricks b{};
    b.lx = lx;
    b.ly = ly;
    b.lz = lz;
    // 8 nodes along x are one 128-byte line of value pairs; y and z as the
    // least shell per node allows
    b.bx = lx < 8 ? lx : 8;
    const uint32_t ex = b.bx + 2 < lx ? b.bx + 2 : lx;
    double best = 0.0;
    for (uint32_t y = 1; y <= ly && y * b.bx <= kMpTile; ++y) {
        uint32_t z = kMpTile / (b.bx * y);
        if (z > lz) z = lz;
        const uint32_t ey = y + 2 < ly ? y + 2 : ly, ez = z + 2 < lz ? z + 2 : lz;
        const uint32_t vol = b.bx * y * z, shell = ex * ey * ez - vol;
        if (shell > kHaloMax) continue;
        const double cost = ((double)(ex * ey * ez) + 40.0) / vol;
        if (b.by == 0 || cost < best) {
            best = cost;
            b.by = y;
            b.bz = z;
        }
    }
    b.inner = halves && b.bz > 1 ? 2 : 1;
    b.bz = (b.bz + b.inner - 1) / b.inner;
    b.nbx = (lx + b.bx - 1) / b.bx;
    b.nby = (ly + b.by - 1) / b.by;
    b.nbz = (lz + b.bz - 1) / b.bz;
    // a plane of a column is what an XCD's share of blocks in flight and its L2
    // hold: the plane below it is still there when the next one is stepped
    b.cx = b.nbx < kColumn ? b.nbx : kColumn;
    b.cy = b.nby < kColumn ? b.nby : kColumn;
    b.ncx = (b.nbx + b.cx - 1) / b.cx;
    b.norder = b.ncx * ((b.nby + b.cy - 1) / b.cy) * b.cx * b.cy * ((b.nbz + b.inner - 1) / b.inner * b.inner);
    return b;
}

// Tiles a lattice of nf fluid nodes is laid out in at most: two consecutive
// tiles hold more than 256 nodes together (so k tiles need floor(k/2) 257 <= nf,
// less than twice nf/256 rounded up), and tiles are only cut while the count
// stays within this.
inline uint64_t mp_tile_bound(uint64_t nf) { return 2 * ((nf + kMpTile - 1) / kMpTile); }

// Whether a layout of nt tiles is tried again with halves of the bricks: bricks
// that hold a little over half a tile each (fine-grained media of porosity 0.5
// to 0.67) merge with none of their neighbours, halves of them by three.  Taken
// where that saves a tenth of the tiles, cuts included.  us per step at 128^3,
// whole / halves: white noise of porosity 0.6 FP64 61.6 / 46.6, FP32-shift
// 53.7 / 47.9; a medium of correlation length 8 and porosity 0.6, whose merged
// halves' halos are cut, 40.5 / 46.4: its tiles are 0.89 full and not tried.
// Fewer tiles than CUs: a step is a launch's time either way.
inline bool try_halves(uint32_t nt, uint32_t nf) { return nt >= 256 && (uint64_t)nt * (kMpTile * 7 / 10) > nf; }
inline uint32_t halves_bound(uint32_t nt) { return nt - nt / 10; }

// One lattice's layout to build (a batch builds several at once).
struct MpBuild {
    Bricks b;
    const uint32_t* nodes;   // the lattice's packed nodes and full-box map
    const uint32_t* map;
    FastDiv dlx, dly;
    uint32_t order_off;      // its entries in the walk's scratch arrays
    uint32_t tile0;          // its first tile
    uint32_t bound;          // tiles it may use
    uint32_t serial;         // one thread may group all bricks where the runs' ends take too many
};
// What the build finds, per lattice.
struct MpBuilt {
    uint32_t ntiles;
    uint32_t halo_max;       // largest halo of its tiles (kHaloMaxGen + 1: beyond a general tile's slots)
};

// The layout's arrays, over all tiles of the lattice or batch.
struct MpTiles {
    uint32_t* info = nullptr;   // nodes of the tile
    uint32_t* halo = nullptr;   // [tile][pitch] entries of the halo nodes, then kSolidSlot
    uint4* tab4 = nullptr;      // LDS slots of the 18 neighbours, three 10-bit fields a word;
    uint2* tab2 = nullptr;      // kTab* bits in the first word
    uint32_t* perm = nullptr;   // packed node of each entry
    uint32_t* inv = nullptr;    // entry of each packed node
    uint32_t pitch = 0;
};

// brick (x, y, z) of place o of the walk; false outside the box
__device__ __forceinline__ bool walk_brick(const Bricks& b, uint32_t o, uint32_t& x, uint32_t& y, uint32_t& z) {
    const uint32_t plane = b.cx * b.cy, column = plane * ((b.nbz + b.inner - 1) / b.inner * b.inner);
    const uint32_t c = o / column, k = o % column, m = k / b.inner;
    x = (c % b.ncx) * b.cx + m % b.cx;
    y = (c / b.ncx) * b.cy + m / b.cx % b.cy;
    z = m / plane * b.inner + k % b.inner;
    return x < b.nbx && y < b.nby && z < b.nbz;
}

// f(box node is fluid, its packed node, fluid nodes of the brick before it)
// for the box nodes of a brick, one wave per brick; returns its fluid nodes
template <typename F>
__device__ __forceinline__ uint32_t walk_nodes(const MpBuild& d, uint32_t bx, uint32_t by, uint32_t bz, F&& f) {
    const Bricks& b = d.b;
    const uint32_t lane = threadIdx.x & 63u, vol = b.bx * b.by * b.bz;
    uint32_t n = 0;
    for (uint32_t k0 = 0; k0 < vol; k0 += 64) {
        const uint32_t k = k0 + lane;
        const uint32_t x = bx * b.bx + k % b.bx, y = by * b.by + (k / b.bx) % b.by, z = bz * b.bz + k / (b.bx * b.by);
        uint32_t q = kSolidSlot;
        if (k < vol && x < b.lx && y < b.ly && z < b.lz) q = d.map[x + b.lx * (y + b.ly * z)];
        const unsigned long long m = __ballot(q != kSolidSlot);
        f(q != kSolidSlot, q, n + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)));
        n += (uint32_t)__popcll(m);
    }
    return n;
}

// fluid nodes of every brick, in walk order (grid: waves over the walk, y: lattices)
__global__ __launch_bounds__(kBlock) void k_mpb_count(const MpBuild* __restrict__ builds, uint32_t* count) {
    const MpBuild& d = builds[blockIdx.y];
    const uint32_t o = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    if (o >= d.b.norder) return;
    uint32_t x, y, z, n = 0;
    if (walk_brick(d.b, o, x, y, z)) n = walk_nodes(d, x, y, z, [](bool, uint32_t, uint32_t) {});
    if ((threadIdx.x & 63u) == 0) count[d.order_off + o] = n;
}

// Bricks into tiles, in walk order: a brick joins the current tile while the
// tile holds at most 256 nodes.  base[o] = entry of the brick's first node.
// split != NULL: tile k of the call without it is cut into 2^split[k] parts, by
// the place of each brick's first node in it (256 parts: every brick alone).
// One block per lattice; a thread
// groups whole runs of kRun bricks, so tiles end at the runs' ends (under 1%
// of a tile's fill where a run fills a hundred, up to a quarter where a sparse
// medium's fills two), unless that takes more tiles than the lattice may use:
// then one thread groups all bricks (one thread's walk of a 256^3 medium's
// 65 536 bricks took 15 ms).
constexpr uint32_t kRun = 128;

// f(o, nodes, tile of the run, nodes of the tile before it) per brick with nodes; returns the run's tiles, and those of the unsplit run, which begin at
// old0.  A thread's loads go out eight at a time: one by one, each a round trip
// to memory, the second grouping of a 96^3 lattice took 113 us, now 69.
struct RunTiles {
    uint32_t tiles, unsplit;
};

template <typename F>
__device__ __forceinline__ RunTiles group_run(const uint32_t* __restrict__ count, uint32_t o0, uint32_t o1,
                                              const uint8_t* __restrict__ split, uint32_t old0, F&& f) {
    constexpr uint32_t kAhead = 8;
    uint32_t tile = 0, acc = 0, old = 0, old_acc = 0, part = 0, exponent = 0;
    bool any = false;
    for (uint32_t o8 = o0; o8 < o1; o8 += kAhead) {
        uint32_t c[kAhead];
#pragma unroll
        for (uint32_t k = 0; k < kAhead; ++k) c[k] = o8 + k < o1 ? count[o8 + k] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kAhead; ++k) {
            if (c[k] == 0) continue;
            bool cut = old_acc + c[k] > kMpTile;
            if (cut) {
                ++old;
                old_acc = 0;
            }
            // read with a brick of the tile only: past the last tile there is no entry
            if (split && (cut || !any)) exponent = split[old0 + old];
            const uint32_t p = (old_acc << exponent) >> 8;
            cut = cut || (any && p != part);
            part = p;
            old_acc += c[k];
            if (cut) {
                ++tile;
                acc = 0;
            }
            f(o8 + k, c[k], tile, acc);
            acc += c[k];
            any = true;
        }
    }
    return any ? RunTiles{tile + 1, old + 1} : RunTiles{0, 0};
}

__global__ __launch_bounds__(kBlock) void k_mpb_group(const MpBuild* __restrict__ builds, MpBuilt* built,
                                                      const uint32_t* __restrict__ counts, uint32_t* base,
                                                      uint32_t* info, const uint8_t* __restrict__ split) {
    __shared__ uint32_t sums[kBlock + 1];
    const MpBuild& d = builds[blockIdx.x];
    const uint32_t* count = counts + d.order_off;
    const uint32_t n = d.b.norder;
    uint32_t run = kRun * d.b.inner, per = 0, r0 = 0, r1 = 0;
    // thread t's runs are [r0, r1); their first tile, and that of the unsplit grouping
    const auto scan = [&](uint32_t mine) {
        __syncthreads();
        sums[threadIdx.x] = mine;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t s = 0;
            for (uint32_t t = 0; t < kBlock; ++t) {
                const uint32_t v = sums[t];
                sums[t] = s;
                s += v;
            }
            sums[kBlock] = s;
        }
        __syncthreads();
        return sums[threadIdx.x];
    };
    const auto none = [](uint32_t, uint32_t, uint32_t, uint32_t) {};
    uint32_t old0 = 0;
    for (int pass = 0; pass < 2; ++pass) {
        const uint32_t nruns = (n + run - 1) / run;
        per = (nruns + kBlock - 1) / kBlock;
        r0 = min(nruns, threadIdx.x * per);
        r1 = min(nruns, r0 + per);
        uint32_t mine = 0;
        for (uint32_t r = r0; r < r1; ++r)
            mine += group_run(count, r * run, min(n, (r + 1) * run), nullptr, 0, none).tiles;
        old0 = scan(mine);
        if (sums[kBlock] <= d.bound || !d.serial) break;
        run = n;
    }
    uint32_t tile0 = old0, total = sums[kBlock];
    if (split) {
        uint32_t mine = 0, old = old0;
        for (uint32_t r = r0; r < r1; ++r) {
            const uint32_t o0 = r * run, o1 = min(n, (r + 1) * run);
            const RunTiles k = group_run(count, o0, o1, split, d.tile0 + old, none);
            mine += k.tiles;
            old += k.unsplit;
        }
        tile0 = scan(mine);
        total = sums[kBlock];
    }
    if (threadIdx.x == 0) {
        built[blockIdx.x].ntiles = total <= d.bound ? total : 0u;  // 0: more tiles than the lattice may use
        built[blockIdx.x].halo_max = 0;
    }
    if (total > d.bound) return;
    uint32_t old = old0;
    for (uint32_t r = r0; r < r1; ++r) {
        const uint32_t o0 = r * run, o1 = min(n, (r + 1) * run), t0 = d.tile0 + tile0;
        const RunTiles k = group_run(count, o0, o1, split, d.tile0 + old,
                                     [&](uint32_t o, uint32_t c, uint32_t tile, uint32_t acc) {
                                         base[d.order_off + o] = (t0 + tile) * kMpTile + acc;
                                         info[t0 + tile] = acc + c;
                                     });
        tile0 += k.tiles;
        old += k.unsplit;
    }
}

// perm and inv (grid as k_mpb_count)
__global__ __launch_bounds__(kBlock) void k_mpb_place(const MpBuild* __restrict__ builds,
                                                      const MpBuilt* __restrict__ built,
                                                      const uint32_t* __restrict__ base, uint32_t* perm,
                                                      uint32_t* inv) {
    const MpBuild& d = builds[blockIdx.y];
    const uint32_t o = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    uint32_t x, y, z;
    if (o >= d.b.norder || built[blockIdx.y].ntiles == 0 || !walk_brick(d.b, o, x, y, z)) return;
    const uint32_t e0 = base[d.order_off + o];
    walk_nodes(d, x, y, z, [&](bool fluid, uint32_t q, uint32_t n) {
        if (fluid) {
            perm[e0 + n] = q;
            inv[q] = e0 + n;
        }
    });
}

// Halo list and slot table of every tile (grid x: a lattice's tiles, y:
// lattices).  The distinct outside neighbours are collected in an LDS hash
// table and sorted, so that consecutive slots read consecutive entries.
// split (may be NULL) receives 1 for a tile with more than kHaloMax.
// A table of 1024 places is enough to tell a tile that must be cut; the general
// tiles keep up to kHaloMaxGen of theirs.
template <bool GEN>
__global__ __launch_bounds__(kBlock) void k_mpb_table(const MpBuild* __restrict__ builds, MpBuilt* built, MpTiles t,
                                                      uint8_t* split) {
    constexpr uint32_t kHashSize = GEN ? 4096 : 1024, kHashMax = GEN ? 2048 : 512;
    static_assert(kHashMax + 2 * kMpTile <= kHashSize && kHashMax > kHaloMax, "room to stop inserting");
    __shared__ uint32_t key[kHashSize];
    __shared__ uint32_t count;
    const MpBuild& d = builds[blockIdx.y];
    if (blockIdx.x >= built[blockIdx.y].ntiles) return;
    const uint32_t tile = d.tile0 + blockIdx.x, e = tile * kMpTile + threadIdx.x;
    const bool valid = threadIdx.x < t.info[tile];
    for (uint32_t k = threadIdx.x; k < kHashSize; k += kBlock) key[k] = kSolidSlot;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    uint32_t q[kQ], word = 0;
    if (valid) {
        word = d.nodes[t.perm[e]];
        Neighbours nb;
        nb.load(d.map, word & kIndexMask, d.dlx, d.dly, d.b.lz);
        static_for<1, kQ>([&](auto I) {
            constexpr int L = I;
            q[L] = nb.q[L] != kSolidSlot ? t.inv[nb.q[L]] : kSolidSlot;
            if (q[L] == kSolidSlot || q[L] / kMpTile == tile) return;
            // bounded: at most one more per thread once the count is past kHashMax
            if (*(volatile uint32_t*)&count > kHashMax) return;
            uint32_t h = (q[L] * 2654435761u) >> (GEN ? 20 : 22);
            for (uint32_t n = 0; n < kHashSize; ++n) {
                const uint32_t was = atomicCAS(&key[h], kSolidSlot, q[L]);
                if (was == kSolidSlot) atomicAdd(&count, 1u);
                if (was == kSolidSlot || was == q[L]) break;
                h = (h + 1) & (kHashSize - 1);
            }
        });
    }
    __syncthreads();
    // bitonic sort, empty places (the largest value) last
    for (uint32_t size = 2; size <= kHashSize; size <<= 1)
        for (uint32_t step = size >> 1; step > 0; step >>= 1) {
            for (uint32_t k = threadIdx.x; k < kHashSize / 2; k += kBlock) {
                const uint32_t i = 2 * k - (k & (step - 1)), j = i + step;
                const uint32_t a = key[i], b = key[j];
                if ((a > b) == ((i & size) == 0)) {
                    key[i] = b;
                    key[j] = a;
                }
            }
            __syncthreads();
        }
    const uint32_t n = count, kept = min(n, min(kHaloMaxGen, t.pitch));
    for (uint32_t k = threadIdx.x; k < t.pitch; k += kBlock)
        t.halo[(uint64_t)tile * t.pitch + k] = k < kept ? key[k] : kSolidSlot;
    uint32_t w[6] = {0, 0, 0, 0, 0, 0};  // an entry without a node
    if (valid) {
        w[0] = kTabNode;
        static_for<1, kQ>([&](auto I) {
            constexpr int L = I;
            uint32_t s = kZeroSlot;
            if (q[L] != kSolidSlot) {
                if (q[L] / kMpTile == tile) {
                    s = q[L] % kMpTile;
                } else {
                    uint32_t lo = 0, hi = kept;  // first place whose key is >= q
                    while (lo < hi) {
                        const uint32_t mid = (lo + hi) / 2;
                        if (key[mid] < q[L]) lo = mid + 1; else hi = mid;
                    }
                    s = lo < kept && key[lo] == q[L] ? kHalo0 + lo : kFarSlot;
                }
            }
            w[(L - 1) / 3] |= s << (10 * ((L - 1) % 3));
        });
        if (word & kNodeInterfacial) w[0] |= kTabInterfacial;
    }
    t.tab4[e] = make_uint4(w[0], w[1], w[2], w[3]);
    t.tab2[e] = make_uint2(w[4], w[5]);
    if (threadIdx.x == 0) {
        if (split) split[tile] = n > kHaloMax ? 1 : 0;
        atomicMax(&built[blockIdx.y].halo_max, n);
    }
}

// place of brick (x, y, z) in the walk (walk_brick's inverse)
__device__ __forceinline__ uint32_t brick_place(const Bricks& b, uint32_t x, uint32_t y, uint32_t z) {
    const uint32_t plane = b.cx * b.cy, column = plane * ((b.nbz + b.inner - 1) / b.inner * b.inner);
    const uint32_t m = x % b.cx + b.cx * (y % b.cy) + plane * (z / b.inner);
    return (x / b.cx + b.ncx * (y / b.cy)) * column + m * b.inner + z % b.inner;
}

// For every tile that split marks (grid as k_mpb_table), the least k for which
// none of its 2^k parts has more than kHaloMax halo nodes, into split: the parts'
// distinct outside neighbours, those in the tile's other parts included, are
// counted in an LDS hash table.  Every brick alone (k = 8) always fits.  (The
// parts laid out and tabled at each k in turn: two more passes over a lattice's
// tiles, 0.85 ms more for a batch of eight 3-D lattices.)
__global__ __launch_bounds__(kBlock) void k_mpb_parts(const MpBuild* __restrict__ builds,
                                                      const MpBuilt* __restrict__ built,
                                                      const uint32_t* __restrict__ base, MpTiles t, uint8_t* split) {
    constexpr uint32_t kPlaces = 8192;  // for at most 18 pairs a node
    static_assert(18 * kMpTile < kPlaces, "room for every pair");
    __shared__ unsigned long long key[kPlaces];
    __shared__ uint32_t count[kMpTile];
    __shared__ uint8_t start[kMpTile];  // of its brick in the tile, by node
    const MpBuild& d = builds[blockIdx.y];
    if (blockIdx.x >= built[blockIdx.y].ntiles) return;
    const uint32_t tile = d.tile0 + blockIdx.x;
    if (split[tile] == 0) return;
    const bool valid = threadIdx.x < t.info[tile];
    uint32_t q[kQ];
    if (valid) {
        const uint32_t r = d.nodes[t.perm[tile * kMpTile + threadIdx.x]] & kIndexMask;
        const uint32_t x = r % d.b.lx, y = r / d.b.lx % d.b.ly, z = r / d.b.lx / d.b.ly;
        start[threadIdx.x] =
            (uint8_t)(base[d.order_off + brick_place(d.b, x / d.b.bx, y / d.b.by, z / d.b.bz)] - tile * kMpTile);
        Neighbours nb;
        nb.load(d.map, r, d.dlx, d.dly, d.b.lz);
        static_for<1, kQ>([&](auto I) { q[I] = nb.q[I] != kSolidSlot ? t.inv[nb.q[I]] : kSolidSlot; });
    }
    uint32_t k = 0;
    for (bool over = true; over && k < 8;) {
        ++k;
        __syncthreads();  // the last round's counts have been read
        for (uint32_t i = threadIdx.x; i < kPlaces; i += kBlock) key[i] = ~0ull;
        count[threadIdx.x] = 0;
        __syncthreads();
        if (valid) {
            const uint32_t part = ((uint32_t)start[threadIdx.x] << k) >> 8;
            static_for<1, kQ>([&](auto I) {
                constexpr int L = I;
                if (q[L] == kSolidSlot) return;
                if (q[L] / kMpTile == tile && ((uint32_t)start[q[L] % kMpTile] << k) >> 8 == part) return;
                const unsigned long long want = (unsigned long long)part << 32 | q[L];
                uint32_t h = ((q[L] ^ part * 0x9E3779B9u) * 2654435761u) >> 19;
                for (uint32_t n = 0; n < kPlaces; ++n) {
                    const unsigned long long was = atomicCAS(&key[h], ~0ull, want);
                    if (was == ~0ull) atomicAdd(&count[part], 1u);
                    if (was == ~0ull || was == want) break;
                    h = (h + 1) & (kPlaces - 1);
                }
            });
        }
        __syncthreads();
        over = __syncthreads_or(count[threadIdx.x] > kHaloMax) != 0;
    }
    if (threadIdx.x == 0) split[tile] = (uint8_t)k;
}

// ------------------------------------------------------- per-node values
// Three values per node of type E (a tracer's moments, u*) side by side, tile
// by tile: a halo node taken from another tile costs one or two cache lines
// whatever its place there.
template <typename E>
struct Trio {
    typedef E Pair __attribute__((ext_vector_type(2), aligned(sizeof(E))));
    // group g of G groups (tracers) of entry e
    static __device__ __forceinline__ uint64_t index(uint32_t e, int G, int g) {
        return (((uint64_t)(e / kMpTile) * G + g) * kMpTile + e % kMpTile) * 3;
    }
    static __device__ __forceinline__ void load(const E* p, uint32_t e, int G, int g, E (&v)[3]) {
        const E* b = p + index(e, G, g);
        const Pair x = *(const Pair*)b;
        v[0] = x[0];
        v[1] = x[1];
        v[2] = b[2];
    }
    static __device__ __forceinline__ void store(E* p, uint32_t e, int G, int g, const E (&v)[3]) {
        E* b = p + index(e, G, g);
        Pair x;
        x[0] = v[0];
        x[1] = v[1];
        *(Pair*)b = x;
        b[2] = v[2];
    }
};

// (rho, vx), (vy, vz) of entry e, v = j + f the tracer flow
__device__ __forceinline__ uint64_t rv_index(uint32_t e) { return 2 * (uint64_t)e; }

// the probabilities coming in from directions 2p+1, 2p+2 of entry e
__device__ __forceinline__ uint64_t win_index(uint32_t e, int p) {
    return ((uint64_t)(e / kMpTile) * 9 + p) * kMpTile + e % kMpTile;
}

// The static fields of a propagation and its moments.
template <typename W>
struct MpFields {
    Vec2<double>* rv = nullptr;   // recomputed form: (rho, v); else NULL
    Vec2<W>* win = nullptr;       // stored form: the 18 incoming probabilities in 9 pairs; else NULL
    double* rem = nullptr;
    W* ustar = nullptr;
    double* P[2] = {nullptr, nullptr};
    double* Pa[2] = {nullptr, nullptr};
};

template <typename W>
struct MpPrepArgs {
    MpTiles t;
    MpFields<W> f;
    const double* rho;      // packed density and flux of the flow
    const double* j;
    const uint32_t* nodes;
    const uint32_t* map;
    double* partials;       // VACF(0) partials, 3T per tile
    Ctrl* ctrl;
    FastDiv dlx, dly;
    uint32_t lz;
    uint64_t Np;            // packed plane stride
    double fx, fy, fz;      // lb.in f_ext (drop_tracers.f90:92)
    double lambda, eps;
    TracerParams tp;
};

// update_tracer_population (drop_tracers.f90:97-100) fused with
// moment_propagation::init (module_moment_propagation.f90:105-137) and the
// static part of propagate (:218-249): per fluid node, the scattering
// probabilities s(r,l) = n_l/rho - w_l + lambda w_l / 2 towards fluid
// neighbours, the rest probability rem, u* = sum s c, and per tracer P(r,1)
// and the VACF(0) contribution; Pa = 0.
template <int T, typename W>
__device__ __forceinline__ void mp_prep_tile(const MpPrepArgs<W>& a, uint32_t tile) {
    __shared__ double lds[kBlock / 64 * 3 * T];
    const uint32_t e = tile * kMpTile + threadIdx.x;
    double vp[3 * T];
#pragma unroll
    for (int k = 0; k < 3 * T; ++k) vp[k] = 0.0;
    if (threadIdx.x < a.t.info[tile]) {
        const uint32_t i = a.t.perm[e], word = a.nodes[i];
        Neighbours nb;
        nb.load(a.map, word & kIndexMask, a.dlx, a.dly, a.lz);
        const double rr = a.rho[i];
        const double vx = a.j[i] + a.fx, vy = a.j[a.Np + i] + a.fy, vz = a.j[2 * a.Np + i] + a.fz;
        if (a.f.rv) {
            a.f.rv[rv_index(e)] = Vec2<double>{rr, vx};
            a.f.rv[rv_index(e) + 1] = Vec2<double>{vy, vz};
        }
        Vec2<W> wp;
        double us[3] = {0.0, 0.0, 0.0};
        double p1[3 * T];
#pragma unroll
        for (int k = 0; k < 3 * T; ++k) p1[k] = 0.0;
        double remv = 1.0;
        static_for<1, kQ>([&](auto I) {
            constexpr int L = I;
            constexpr int Li = kInv[L];
            constexpr int cx = kCX[L], cy = kCY[L], cz = kCZ[L];
            const uint32_t q = nb.q[L];
            wp[(L - 1) & 1] = W(0);
            if (q != kSolidSlot) {
                const double s = scatter_prob<L, W>(rr, vx, vy, vz, a.lambda);
                remv = remv - s;
                if constexpr (cx != 0) us[0] = us[0] + sgn<cx>(s);
                if constexpr (cy != 0) us[1] = us[1] + sgn<cy>(s);
                if constexpr (cz != 0) us[2] = us[2] + sgn<cz>(s);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    if constexpr (cx != 0) vp[3 * t + 0] = vp[3 * t + 0] + a.tp.bw[t] * s;
                    if constexpr (cy != 0) vp[3 * t + 1] = vp[3 * t + 1] + a.tp.bw[t] * s;
                    if constexpr (cz != 0) vp[3 * t + 2] = vp[3 * t + 2] + a.tp.bw[t] * s;
                }
                const double rn = a.rho[q];
                const double wx = a.j[q] + a.fx, wy = a.j[a.Np + q] + a.fy, wz = a.j[2 * a.Np + q] + a.fz;
                const double sp = scatter_prob<Li, W>(rn, wx, wy, wz, a.lambda);
                wp[(L - 1) & 1] = (W)sp;
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    if constexpr (cx != 0) p1[3 * t + 0] = p1[3 * t + 0] + sgn<-cx>(sp) * a.tp.bw[t];
                    if constexpr (cy != 0) p1[3 * t + 1] = p1[3 * t + 1] + sgn<-cy>(sp) * a.tp.bw[t];
                    if constexpr (cz != 0) p1[3 * t + 2] = p1[3 * t + 2] + sgn<-cz>(sp) * a.tp.bw[t];
                }
            }
            if constexpr ((L & 1) == 0)
                if (a.f.win) a.f.win[win_index(e, (L - 2) / 2)] = wp;
        });
        a.f.rem[e] = remv;
        bool low = false;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const double rt = (a.tp.ads[t] && (word & kNodeInterfacial)) ? remv - a.tp.ka[t] : remv;
            low = low || rt < a.eps;
        }
        if (low) a.ctrl->restpart = 1;
        // outside the range that quotient() is exact for: the general step divides
        const double big = fmax(fmax(fabs(vx), fabs(vy)), fabs(vz));
        if (!(rr >= 0x1p-400 && rr <= 0x1p400 && big <= 0x1p400)) a.ctrl->mp_divide = 1;
        W usw[3];
        for (int c = 0; c < 3; ++c) usw[c] = (W)us[c];
        Trio<W>::store(a.f.ustar, e, 1, 0, usw);
        const double zero[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const double p[3] = {p1[3 * t], p1[3 * t + 1], p1[3 * t + 2]};
            Trio<double>::store(a.f.P[0], e, T, t, p);
            if (a.f.Pa[0]) {
                Trio<double>::store(a.f.Pa[0], e, T, t, zero);
                Trio<double>::store(a.f.Pa[1], e, T, t, zero);
            }
        }
    }
    block_partial<3 * T, kBlock>(vp, a.partials + 3 * T * (uint64_t)tile, lds);
}

template <typename W>
struct MpStepArgs {
    MpTiles t;
    const Vec2<double>* rv;          // as in MpFields
    const Vec2<W>* win;
    const double* rem;
    const W* ustar;
    const double* Pn;                // P, Pa before the step, and after it
    double* Px;
    const double* Pan;
    double* Pax;
    int32_t any_ads;                 // some tracer of the batch adsorbs (Pa allocated)
    double* partials;                // this step's VACF partials, 3T per tile
    const double* prev_partials;     // the previous step's, reduced by one block (NULL: none)
    double* prev_vtrace;             // where VACF(it-1) goes
    int64_t it;
    int32_t check_conv = 0;          // that block also applies the convergence test to VACF(it-1)
    double lim1 = 0.0, lim2 = 0.0;   // its limits (module_moment_propagation.f90:284)
    double lambda;
    Ctrl* ctrl;
    TracerParams tp;
    // general tiles: the neighbours without an LDS slot
    const uint32_t* nodes;
    const uint32_t* map;
    FastDiv dlx, dly;
    uint32_t lz;

    // the fields f before the step whose input is buffer `now`
    __host__ __device__ __forceinline__ void fields(const MpFields<W>& f, bool now) {
        rv = f.rv;
        win = f.win;
        rem = f.rem;
        ustar = f.ustar;
        Pn = now ? f.P[1] : f.P[0];
        Px = now ? f.P[0] : f.P[1];
        Pan = now ? f.Pa[1] : f.Pa[0];
        Pax = now ? f.Pa[0] : f.Pa[1];
    }
};

// VACF(it-1) from the previous step's nparts partials and, with check_conv,
// the convergence test: a stop set here ends the run at step it-1 (this
// launch's tiles may have started step it already; they write only the other
// buffer of P, and every later launch returns at once).
template <int T, typename W>
__device__ __forceinline__ void mp_reduce_prev(const MpStepArgs<W>& a, uint32_t nparts) {
    __shared__ double red[kBlock / 64 * 3 * T];
    if (!a.prev_partials || block_flag(vload(&a.ctrl->mp_stop) != 0)) return;
    mp_reduce_block<3 * T, kBlock>(a.prev_partials, nparts, a.prev_vtrace, a.ctrl, 1, a.it - 1, a.check_conv, a.lim1,
                                   a.lim2, red);
}

// Sums of a tile's NV values per thread, in a fixed order: over the four waves
// lane by lane, then over the lanes, value a by wave a mod 4 (a quarter of the
// lane sums that each wave summing all its values would take).  lds: NV * 256
// doubles that no wave still reads.
template <int NV>
__device__ __forceinline__ void tile_partial(const double (&v)[NV], double* out, double* lds) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < NV; ++a) lds[a * kMpTile + threadIdx.x] = v[a];
    __syncthreads();
#pragma unroll
    for (int a0 = 0; a0 < NV; a0 += 4) {
        const uint32_t a = a0 + wave;
        if (a < NV) {
            double s = lds[a * kMpTile + lane];
            for (int w = 1; w < 4; ++w) s = s + lds[a * kMpTile + 64 * w + lane];
            s = wave_sum(s);
            if (lane == 0) out[a] = s;
        }
    }
}

// One moment-propagation step of T tracers on one tile,
// module_moment_propagation.f90:207-253:
// P(r,t+1) = sum_l P(r+c_l,t) s(r+c_l, inv l) + rem(r) P(r,t) [+ kd Pa],
// Pa(r,t+1) = (1-kd) Pa(r,t) + ka P(r,t) at adsorbing interfacial nodes,
// VACF(t) = sum_r P(r,t) . u*(r).
// The incoming probabilities are recomputed from the neighbours' (rho, v)
// with the set-up's arithmetic (the same bits), once for all tracers; the
// tracers' P pass through LDS one after the other, the next one's values in
// flight meanwhile.  A solid neighbour is the zero slot: it adds w * 0.
// GEN: some tile has neighbours without an LDS slot, or some density or flow
// is outside the range of quotient().
template <int T, typename W, bool RV, bool GEN>
__device__ __forceinline__ void mp_step_tile(const MpStepArgs<W>& a, uint32_t tile) {
    constexpr uint32_t S = GEN ? kSlotsGen : kSlots1;
    constexpr int NH = GEN ? 3 : 2;  // halo nodes per thread
    // LDS by slot: tracer values in (pA, pB)[0] and [1] in turn, (rho, v) and 1/rho
    // in (rv0, rv1, ri), whose place the second tracer's values take
    constexpr uint32_t kBuf = S * 24;
    __shared__ __align__(16) char smem[RV ? S * 40 + kBuf : (T > 1 ? 2 * kBuf : kBuf)];
    __shared__ int32_t stop;
    Vec2<double>* const pA[2] = {(Vec2<double>*)smem, (Vec2<double>*)(smem + kBuf)};
    double* const pB[2] = {(double*)(smem + S * 16), (double*)(smem + kBuf + S * 16)};
    Vec2<double>* const rv0 = (Vec2<double>*)(smem + kBuf);
    Vec2<double>* const rv1 = rv0 + S;
    double* const ri = (double*)(rv1 + S);
    const auto put_p = [&](int buf, uint32_t s, const double (&v)[3]) {
        pA[buf][s] = Vec2<double>{v[0], v[1]};
        pB[buf][s] = v[2];
    };
    const uint32_t lane = threadIdx.x;
    __syncthreads();  // a previous tile of this block (persistent launches) has read the LDS arrays
    // Everything is issued as early as its address is known: the halo list,
    // the tile's own values and the stop flag in one round trip to memory,
    // the halo's values in the next; the flag is looked at after the barrier.
    const uint32_t e = tile * kMpTile + lane;
    const double* const Pn = a.Pn;
    uint32_t h[NH];
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        const uint32_t s = lane + k * kMpTile;
        h[k] = s < a.t.pitch ? a.t.halo[(uint64_t)tile * a.t.pitch + s] : kSolidSlot;
    }
    const uint4 t4 = a.t.tab4[e];
    const uint2 t2 = a.t.tab2[e];
    const uint32_t tab[6] = {t4.x, t4.y, t4.z, t4.w, t2.x, t2.y};
    const int32_t stopped = vload(&a.ctrl->mp_stop);
    const bool valid = (tab[0] & kTabNode) != 0;
    double rm = 0.0, p[3] = {0.0, 0.0, 0.0}, hp[NH][3];
    W us[3] = {W(0), W(0), W(0)};
    Vec2<W> wp[9];  // stored form
    {
        Vec2<double> r0, r1, h0[NH], h1[NH];
#pragma unroll
        for (int k = 0; k < NH; ++k)
            if (h[k] != kSolidSlot) {
                if constexpr (RV) {
                    h0[k] = a.rv[rv_index(h[k])];
                    h1[k] = a.rv[rv_index(h[k]) + 1];
                }
                Trio<double>::load(Pn, h[k], T, 0, hp[k]);
            }
        if (valid) {
            if constexpr (RV) {
                r0 = a.rv[rv_index(e)];
                r1 = a.rv[rv_index(e) + 1];
            }
            Trio<double>::load(Pn, e, T, 0, p);
            rm = a.rem[e];
            Trio<W>::load(a.ustar, e, 1, 0, us);
            if constexpr (!RV)
                for (int k = 0; k < 9; ++k) wp[k] = a.win[win_index(e, k)];
        }
        const auto put = [&](uint32_t s, const Vec2<double>& x0, const Vec2<double>& x1,
                             const double (&v)[3]) {
            if constexpr (RV) {
                rv0[s] = x0;
                rv1[s] = x1;
                ri[s] = 1.0 / x0[0];
            }
            put_p(0, s, v);
        };
        if (valid) put(lane, r0, r1, p);
        if (lane == 0) {
            stop = stopped;
            const double zero[3] = {0.0, 0.0, 0.0};
            put(kZeroSlot, Vec2<double>{1.0, 0.0}, Vec2<double>{0.0, 0.0}, zero);
        }
#pragma unroll
        for (int k = 0; k < NH; ++k)
            if (h[k] != kSolidSlot) put(kHalo0 + lane + k * kMpTile, h0[k], h1[k], hp[k]);
    }
    __syncthreads();
    if (stop) return;
    const auto slot = [&](auto I) {
        constexpr int L = I;
        return (tab[(L - 1) / 3] >> (10 * ((L - 1) % 3))) & 1023u;
    };
    // general tiles: the entry of neighbour L
    const auto far_entry = [&](auto I) {
        constexpr int L = I;
        Nbr nb;
        nb.init(a.nodes[a.t.perm[e]] & kIndexMask, a.dlx, a.dly, a.lz);
        return a.t.inv[a.map[nb.at<kCX[L], kCY[L], kCZ[L]>()]];
    };
    // keeps the LDS reads of a few directions in flight, not of all 18 (registers)
    const auto pace = [](auto I) {
        if constexpr (I % kPace == 0) __builtin_amdgcn_sched_barrier(0);
    };
    double w[kQ], vp[3 * T];
#pragma unroll
    for (int k = 0; k < 3 * T; ++k) vp[k] = 0.0;
    // the probability coming in from neighbour L
    const auto incoming = [&](auto I) {
        constexpr int L = I;
        if constexpr (!RV) return (double)wp[(L - 1) / 2][(L - 1) & 1];
        const uint32_t s = slot(I);
        Vec2<double> r0, r1;
        double x = 0.0;
        if (GEN && s == kFarSlot) {
            const uint32_t q = far_entry(I);
            r0 = a.rv[rv_index(q)];
            r1 = a.rv[rv_index(q) + 1];
            x = 1.0 / r0[0];
        } else {
            r0 = rv0[s];
            r1 = rv1[s];
            x = ri[s];
        }
        if constexpr (GEN) return scatter_prob<kInv[L], W>(r0[0], r0[1], r1[0], r1[1], a.lambda);
        return scatter_prob<kInv[L], W>(r0[0], x, r0[1], r1[0], r1[1], a.lambda);
    };
    const bool ads_node = a.any_ads && (tab[0] & kTabInterfacial) != 0;
    static_for<0, T>([&](auto TT) {
        constexpr int t = TT;
        constexpr int buf = t & 1;
        if constexpr (t > 0) {
            // every wave is past its reads of this buffer's last contents:
            // (rho, v) for t = 1, tracer t-2 (whose readers passed the barrier of t-1) after
            if constexpr (t == 1 && RV) __syncthreads();
            if (valid) put_p(buf, lane, p);
            if (t == 1 && lane == 0) {
                const double zero[3] = {0.0, 0.0, 0.0};
                put_p(buf, kZeroSlot, zero);
            }
#pragma unroll
            for (int k = 0; k < NH; ++k)
                if (h[k] != kSolidSlot) put_p(buf, kHalo0 + lane + k * kMpTile, hp[k]);
            __syncthreads();
        }
        double pn[3];  // the next tracer's values, in flight during this one's sum
        if constexpr (t + 1 < T) {
            if (valid) Trio<double>::load(Pn, e, T, t + 1, pn);
#pragma unroll
            for (int k = 0; k < NH; ++k)
                if (h[k] != kSolidSlot) Trio<double>::load(Pn, h[k], T, t + 1, hp[k]);
        }
        if (valid) {
            double pa[3] = {0.0, 0.0, 0.0};
            if (ads_node) Trio<double>::load(a.Pan, e, T, t, pa);
            double acc[3] = {0.0, 0.0, 0.0};
            static_for<1, kQ>([&](auto I) {
                constexpr int L = I;
                pace(I);
                if constexpr (t == 0 || !RV) w[L] = incoming(I);  // kept for the other tracers
                const uint32_t s = slot(I);
                double q[3];
                if (GEN && s == kFarSlot) {
                    Trio<double>::load(Pn, far_entry(I), T, t, q);
                } else {
                    const Vec2<double> x = pA[buf][s];
                    q[0] = x[0];
                    q[1] = x[1];
                    q[2] = pB[buf][s];
                }
                for (int c = 0; c < 3; ++c) acc[c] = acc[c] + q[c] * w[L];
            });
            double px[3];
            for (int c = 0; c < 3; ++c) vp[3 * t + c] = p[c] * (double)us[c];
            if (!ads_node) {
                for (int c = 0; c < 3; ++c) px[c] = acc[c] + rm * p[c];
            } else {
                double pax[3];
                const double rt = rm - a.tp.ka[t];
                for (int c = 0; c < 3; ++c) {
                    if (a.tp.ads[t]) {
                        px[c] = (acc[c] + rt * p[c]) + pa[c] * a.tp.kd[t];
                        pax[c] = pa[c] * a.tp.one_minus_kd[t] + p[c] * a.tp.ka[t];
                    } else {  // a tracer without adsorption keeps Pa = 0
                        px[c] = acc[c] + rm * p[c];
                        pax[c] = pa[c];
                    }
                }
                Trio<double>::store(a.Pax, e, T, t, pax);
            }
            Trio<double>::store(a.Px, e, T, t, px);
        }
        if constexpr (t + 1 < T)
            for (int c = 0; c < 3; ++c) p[c] = pn[c];
    });
    __syncthreads();
    static_assert(sizeof(smem) >= 3 * T * kMpTile * sizeof(double), "tile_partial's space");
    tile_partial<3 * T>(vp, a.partials + (uint64_t)(3 * T) * tile, (double*)smem);
}

// A whole chunk of steps of one tracer in one launch of one block, for a
// lattice of at most kRunTiles tiles: P stays in LDS, the probabilities, Pa and
// everything else of a node in its thread's registers, and a step costs two
// barriers in place of a launch.  The sums are those of mp_step_tile,
// tile_partial and mp_reduce_block in their order, so the bits are the same.
// us per step launched / here: 60 nodes 3.6 / 1.5, 512 (a 4x4x34 slit) 3.8 / 1.7,
// 768 (three tiles) 3.7 / 1.75, 1024 (four, all a block's threads) 3.8 / 2.0.
constexpr uint32_t kRunTiles = 4;

// lane k of wave 0 holds component k of the running sums
template <typename W>
__global__ __launch_bounds__(1024) void k_mp_run(MpStepArgs<W> a, int64_t S, uint32_t ntiles, double* P0, double* P1,
                                                 double* Pa0, double* Pa1, double* vtrace) {
    constexpr uint32_t E = kRunTiles * kMpTile, kNone = E;  // kNone: a solid neighbour's slot
    __shared__ Vec2<double> pA[E + 1];
    __shared__ double pB[E + 1];
    __shared__ double vs[3 * E];              // P . u* by component and entry
    __shared__ double part[3 * kRunTiles];    // tile sums
    __shared__ int32_t stop;
    if (block_flag(vload(&a.ctrl->mp_stop) != 0)) return;
    const uint32_t e = threadIdx.x, lane = e & 63u, wave = e >> 6, nwaves = blockDim.x >> 6;
    const bool valid = e % kMpTile < a.t.info[e / kMpTile];
    uint16_t slot[kQ];
    double w[kQ], p[3] = {0.0, 0.0, 0.0}, pa[3] = {0.0, 0.0, 0.0}, rm = 0.0;
    W us[3] = {W(0), W(0), W(0)};
    bool ads = false;
    if (valid) {
        const uint32_t word = a.nodes[a.t.perm[e]];
        Neighbours nb;
        nb.load(a.map, word & kIndexMask, a.dlx, a.dly, a.lz);
        static_for<1, kQ>([&](auto I) {
            constexpr int L = I;
            slot[L] = (uint16_t)kNone;
            w[L] = 0.0;
            if (nb.q[L] != kSolidSlot) {
                const uint32_t q = a.t.inv[nb.q[L]];
                slot[L] = (uint16_t)q;
                if (a.rv) {
                    const Vec2<double> r0 = a.rv[rv_index(q)], r1 = a.rv[rv_index(q) + 1];
                    w[L] = scatter_prob<kInv[L], W>(r0[0], r0[1], r1[0], r1[1], a.lambda);
                } else {
                    w[L] = (double)a.win[win_index(e, (L - 1) / 2)][(L - 1) & 1];
                }
            }
        });
        Trio<double>::load(a.Pn, e, 1, 0, p);
        rm = a.rem[e];
        Trio<W>::load(a.ustar, e, 1, 0, us);
        ads = a.any_ads && (word & kNodeInterfacial) != 0;
        if (ads) Trio<double>::load(a.Pan, e, 1, 0, pa);
        pA[e] = Vec2<double>{p[0], p[1]};
        pB[e] = p[2];
    }
    const double ka = a.tp.ka[0], kd = a.tp.kd[0], keep = a.tp.one_minus_kd[0];
    double run_s = 0.0, run_c = 0.0;
    if (e < 3) {
        run_s = a.ctrl->deff_s[e];
        run_c = a.ctrl->deff_c[e];
    }
    if (e == 0) {
        pA[kNone] = Vec2<double>{0.0, 0.0};
        pB[kNone] = 0.0;
        stop = 0;
    }
    // VACF of the chunk's step k from the tile sums (wave 0), and the convergence test
    const auto reduce = [&](int64_t k) {
        double s[3];
        for (int c = 0; c < 3; ++c) s[c] = lane < ntiles ? part[3 * lane + c] : 0.0;
        wave_sums<3>(s);
        bool below = true;
        if (lane < 3) {
            const double t = lane == 0 ? s[0] : lane == 1 ? s[1] : s[2];
            vtrace[3 * k + lane] = t;
            const double u = run_s + t;
            run_c = run_c + ((fabs(run_s) >= fabs(t)) ? (run_s - u) + t : (t - u) + run_s);
            run_s = u;
            below = fabs(t) < a.lim1 && fabs(t) < a.lim2;
        }
        return a.check_conv && a.it + k > 2 && __all(below);
    };
    __syncthreads();
    int64_t ran = 0;
    bool conv = false;
    for (int64_t k = 0; k < S; ++k) {
        if (k > 0 && wave == 0) {
            const bool c = reduce(k - 1);
            if (lane == 0 && c) stop = 1;
        }
        double px[3] = {0.0, 0.0, 0.0}, vp[3] = {0.0, 0.0, 0.0};
        if (valid) {
            double acc[3] = {0.0, 0.0, 0.0};
            static_for<1, kQ>([&](auto I) {
                constexpr int L = I;
                if constexpr (L % kPace == 0) __builtin_amdgcn_sched_barrier(0);
                const Vec2<double> x = pA[slot[L]];
                const double y = pB[slot[L]];
                acc[0] = acc[0] + x[0] * w[L];
                acc[1] = acc[1] + x[1] * w[L];
                acc[2] = acc[2] + y * w[L];
            });
            for (int c = 0; c < 3; ++c) {
                vp[c] = p[c] * (double)us[c];
                px[c] = acc[c] + rm * p[c];
                if (ads) px[c] = (acc[c] + (rm - ka) * p[c]) + pa[c] * kd;
            }
        }
        for (int c = 0; c < 3; ++c) vs[c * E + e] = vp[c];
        __syncthreads();  // every read of P and of the tile sums is over
        conv = stop != 0;
        if (conv) break;
        if (valid) {
            pA[e] = Vec2<double>{px[0], px[1]};
            pB[e] = px[2];
            for (int c = 0; c < 3; ++c) {
                if (ads) pa[c] = pa[c] * keep + p[c] * ka;
                p[c] = px[c];
            }
        }
        // tile_partial's sums, one (tile, component) a wave
        for (uint32_t q = wave; q < 3 * ntiles; q += nwaves) {
            const double* v = vs + (q % 3) * E + (q / 3) * kMpTile + lane;
            double s = v[0];
            for (int x = 1; x < 4; ++x) s = s + v[64 * x];
            s = wave_sum(s);
            if (lane == 0) part[q] = s;
        }
        ran = k + 1;
        __syncthreads();
    }
    if (!conv && wave == 0) {
        const bool c = reduce(S - 1);
        if (lane == 0 && c) stop = 1;
    }
    if (e < 3) {
        a.ctrl->deff_s[e] = run_s;
        a.ctrl->deff_c[e] = run_c;
    }
    if (e == 0 && stop) {
        a.ctrl->mp_conv_step = a.it + ran - 1;
        a.ctrl->mp_stop = 1;
    }
    if (valid) {  // the buffer that `ran` launched steps would have left
        const bool other = (ran & 1) != 0;
        Trio<double>::store(other ? P1 : P0, e, 1, 0, p);
        if (ads) Trio<double>::store(other ? Pa1 : Pa0, e, 1, 0, pa);
    }
}

// P or Pa (p0 or p1 by blockIdx.y) of tracer t of T in the full box, three
// values per box node of [r0, r0 + n), 0 at solids
__global__ __launch_bounds__(kBlock) void k_mp_box(const double* __restrict__ p0, const double* __restrict__ p1,
                                                   const uint32_t* __restrict__ inv, const uint32_t* __restrict__ map,
                                                   int32_t T, int32_t tracer, double* __restrict__ out, uint32_t r0,
                                                   uint32_t n) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    const uint32_t q = map[r0 + k];
    double v[3] = {0.0, 0.0, 0.0};
    if (q != kSolidSlot) Trio<double>::load(blockIdx.y ? p1 : p0, inv[q], T, tracer, v);
    for (int c = 0; c < 3; ++c) out[3 * ((uint64_t)blockIdx.y * n + k) + c] = v[c];
}

}  // namespace
