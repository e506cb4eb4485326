// k44_pack_index.hpp — index arithmetic of packed row reads (host and device; no HIP types, so that
// it can be checked on the host at sizes no test allocates).
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define K44_PACK_HD __host__ __device__ __forceinline__
#else
#define K44_PACK_HD inline
#endif

namespace k44dev {

// Element i of [rows][cols] is column c of row r.
template <typename I>
struct RowCol {
    I r, c;
};

template <typename I>
K44_PACK_HD RowCol<I> row_col(I i, I cols) {
    const I r = i / cols;
    return {r, (I)(i - r * cols)};
}

// Calls f(first, n, cols) with the index type the read needs: 32-bit division while every index of
// this part and `cols` itself, which belongs to the whole read (one row of 2^32 and more elements is
// read in parts of 2^19), fit.  Parts end below 2^31: a grid-stride loop's last step then stays below
// 2^32.
template <typename F>
inline void with_pack_index(uint64_t first, uint64_t n, uint64_t cols, F &&f) {
    if (first + n < (1ull << 31) && cols < (1ull << 32))
        f((uint32_t)first, (uint32_t)n, (uint32_t)cols);
    else
        f(first, n, cols);
}

}  // namespace k44dev
