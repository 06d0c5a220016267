// The packed node list, map and interfacial flags of a lattice, built on the
// GPU from its nature (0 = fluid), for the single-lattice path and the batch
// engine: one byte per box node crosses the bus instead of four per box node
// and four per fluid node, and the host only counts the fluid nodes.  Host lists
// and uploads before / this: a context of 64^3 1.9 / 0.7 ms, of 256^3 137 / 3 ms;
// 1024 2-D cells (10 000 box nodes at most) admitted to a batch 50 / 20 ms, eight
// 3-D requests (96^3 at most) 6.6 / 0.4 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

#include "lbx_device.h"

namespace {

using namespace lbx;

constexpr uint32_t kNodeThreads = 256;
constexpr uint32_t kNodeRows = 16;                          // box nodes per thread
constexpr uint32_t kNodeChunk = kNodeThreads * kNodeRows;   // box nodes of a block
// Up to this many chunks a block counts the fluid nodes before its own chunk
// itself (at most 8 16-byte loads a thread); above it a first launch counts
// them chunk by chunk.
constexpr uint32_t kNodeCountChunks = 8;

inline uint32_t node_chunks(uint64_t N) { return (uint32_t)((N + kNodeChunk - 1) / kNodeChunk); }
inline uint32_t count_fluid(const int8_t* nature, uint64_t N) {
    uint32_t n = 0;
    for (uint64_t r = 0; r < N; ++r) n += nature[r] == 0;
    return n;
}

__device__ __forceinline__ uint32_t zero_bytes(uint32_t v) {
    return __popc(~(((v & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v | 0x7f7f7f7fu));
}

// the block's sum of v, in every thread (lds: 4 words that no wave still reads)
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* lds) {
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    if ((threadIdx.x & 63u) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    return lds[0] + lds[1] + lds[2] + lds[3];
}

// fluid nodes of each chunk
__global__ __launch_bounds__(kNodeThreads) void k_node_count(const int8_t* __restrict__ nature, uint32_t N,
                                                             uint32_t* __restrict__ counts) {
    __shared__ uint32_t lds[4];
    const uint32_t r0 = blockIdx.x * kNodeChunk + threadIdx.x;
    uint32_t n = 0;
    for (uint32_t k = 0; k < kNodeRows; ++k) {
        const uint32_t r = r0 + k * kNodeThreads;
        if (r < N) n += nature[r] == 0;
    }
    n = block_sum(n, lds);
    if (threadIdx.x == 0) counts[blockIdx.x] = n;
}

// One chunk (one block of kNodeThreads): the packed index of its fluid nodes
// is `first` and the number of fluid nodes before them in the box; *nfi
// collects the interfacial ones (a neighbour along any of the 18 directions is
// solid, lbx_detect_interfacial).  nature is 16-byte aligned.
__device__ __forceinline__ void node_chunk(const int8_t* __restrict__ nature, uint32_t N,
                                           const uint32_t* __restrict__ counts, uint32_t chunk, uint32_t first,
                                           uint32_t* __restrict__ nodes, uint32_t* __restrict__ map, uint32_t* nfi,
                                           const FastDiv& dlx, const FastDiv& dly, uint32_t lz) {
    __shared__ uint32_t lds[4], ilds[4], off[64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t before = 0;
    if (counts) {
        for (uint32_t k = tid; k < chunk; k += kNodeThreads) before += counts[k];
    } else {
        const uint4* v = (const uint4*)nature;
        for (uint32_t k = tid; k < chunk * (kNodeChunk / 16); k += kNodeThreads) {
            const uint4 x = v[k];
            before += zero_bytes(x.x) + zero_bytes(x.y) + zero_bytes(x.z) + zero_bytes(x.w);
        }
    }
    const uint32_t r0 = chunk * kNodeChunk + tid;
    uint32_t fluid = 0;  // bit k: row k's node
    for (uint32_t k = 0; k < kNodeRows; ++k) {
        const uint32_t r = r0 + k * kNodeThreads;
        if (r < N && nature[r] == 0) fluid |= 1u << k;
    }
    for (uint32_t k = 0; k < kNodeRows; ++k) {
        const unsigned long long m = __ballot((fluid >> k) & 1u);
        if (lane == 0) off[k * 4 + wave] = (uint32_t)__popcll(m);
    }
    before = block_sum(before, lds);
    if (wave == 0) {  // row by row, wave by wave: exclusive sums
        const uint32_t own = off[lane];
        uint32_t s = own;
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t t = __shfl_up(s, d);
            if ((int)lane >= d) s += t;
        }
        off[lane] = s - own;
    }
    __syncthreads();
    uint32_t ni = 0;
    for (uint32_t k = 0; k < kNodeRows; ++k) {
        const uint32_t r = r0 + k * kNodeThreads;
        const bool f = (fluid >> k) & 1u;
        const unsigned long long m = __ballot(f);
        if (r >= N) continue;
        if (!f) {
            map[r] = 0xFFFFFFFFu;
            continue;
        }
        const uint32_t i = first + before + off[k * 4 + wave] + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        Nbr nb;
        nb.init(r, dlx, dly, lz);
        int solid = 0;
        static_for<1, kQ>([&](auto I) {
            constexpr int L = I;
            solid |= nature[nb.at<kCX[L], kCY[L], kCZ[L]>()];
        });
        map[r] = i;
        nodes[i] = r | (solid ? 0x80000000u : 0u);
        ni += solid != 0;
    }
    ni = block_sum(ni, ilds);
    if (tid == 0 && ni) atomicAdd(nfi, ni);  // cleared by the caller
}

}  // namespace
