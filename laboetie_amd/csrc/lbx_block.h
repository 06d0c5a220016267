// Status codes of HIP calls and the device allocations of liblbx: single
// arrays, and blocks that hold all arrays of one purpose.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/lbx.h"

namespace {

int hip_status(hipError_t e) {
    if (e == hipSuccess) return LBX_OK;
    (void)hipGetLastError();
    return e == hipErrorOutOfMemory ? LBX_ERR_NOMEM : LBX_ERR_DEVICE;
}
int hip_status(int st) { return st; }  // an lbx status passes through

#define LBX_TRY(expr)                            \
    do {                                         \
        int _st = hip_status(expr);              \
        if (_st != LBX_OK) return _st;           \
    } while (0)

template <typename T>
int dalloc(T** p, uint64_t count) {
    *p = nullptr;
    if (count == 0) return LBX_OK;
    hipError_t e = hipMalloc((void**)p, count * sizeof(T));
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
        return e == hipErrorOutOfMemory ? LBX_ERR_NOMEM : LBX_ERR_DEVICE;
    }
    return LBX_OK;
}

template <typename T>
void dfree(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

// One device allocation that several arrays share.  The driver takes and
// gives back every large allocation by itself, some 0.1-0.2 ms each, and a
// context made right after another went waits for the other's.  ms with an
// allocation per array / with blocks: contexts made and destroyed in turn, 32^3
// nodes 0.6-0.9 / 0.25, 128^3 3.4 / 0.6; lbx_mp_init again, 64^3 1.4 / 0.045;
// batches of 1 M nodes made and destroyed 4.7 / 0.66.
struct Block {
    char* at = nullptr;
    uint64_t bytes = 0;
};

// lay(take) names a block's arrays by take(pointer, count); each begins where
// an allocation of its own would, as far as its addresses matter: at a page, or
// a 2 MiB page once it fills one.
uint64_t block_align(uint64_t at, uint64_t bytes) {
    const uint64_t a = bytes >= (2u << 20) ? 2u << 20 : 4096u;
    return (at + a - 1) / a * a;
}
template <typename Lay>
uint64_t block_bytes(Lay&& lay) {
    uint64_t n = 0;
    lay([&](auto*& p, uint64_t count) { n = block_align(n, count * sizeof(*p)) + count * sizeof(*p); });
    return n;
}
template <typename Lay>
void block_place(const Block& b, Lay&& lay) {
    uint64_t n = 0;
    lay([&](auto*& p, uint64_t count) {
        n = block_align(n, count * sizeof(*p));
        p = (std::remove_reference_t<decltype(p)>)(b.at + n);
        n += count * sizeof(*p);
    });
}
void give_block(Block* b) {
    dfree(b->at);
    b->bytes = 0;
}
// A block that lay's arrays fit, and them in it.  The one there is kept while
// they fill three quarters of it (grow: while they fit).
template <typename Lay>
int take_block(Block* b, Lay&& lay, bool grow = false) {
    const uint64_t n = block_bytes(lay);
    if (n > b->bytes || (!grow && n < b->bytes / 4 * 3)) {
        give_block(b);
        LBX_TRY(dalloc(&b->at, n));
        b->bytes = n;
    }
    block_place(*b, lay);
    return LBX_OK;
}

}  // namespace
