// tile_extent.h - sizes of the buffer resources that a 128-key tile's copies read through. Plain arithmetic, so that it is also
// checked on the CPU.
#ifndef FMHA_TILE_EXTENT_H
#define FMHA_TILE_EXTENT_H

#include <stdint.h>

#ifdef __HIP__
#define FMHA_TILE_FN __host__ __device__ __forceinline__
#else
#define FMHA_TILE_FN inline
#endif

// Bytes from a tile's first row that its copies may read: `left` rows lie before the end of the range (none when it is negative),
// a tile has 128. The rows are clamped before they are multiplied, so the size is below 2^31 for every stride below 16 MiB
// (65536 KV heads are 8 MiB): a whole K of 2 GiB or more, or many heads past a short range, would wrap. No copy addresses the
// other heads' bytes behind the last row's own.
FMHA_TILE_FN uint32_t tile_extent(int32_t left, uint32_t stride) {
    int32_t rows = left < 0 ? 0 : left;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+s"(rows));   // two scalar instructions: as one clamp the compiler takes a vector one, and every size back from it
#endif
    return (uint32_t)(rows > 128 ? 128 : rows) * stride;
}

// The sizes of consecutive tiles as running state: those of the current K tile and of the V tile `LAG` tiles (0 or 1) behind it.
// advance() steps to the next ones, after the current copies are out, so that none of its instructions stands before them.
template <int LAG>
struct TileSizes {
    int32_t left;    // rows from the current K tile's first one to the end of the range
    uint32_t k, v;   // the current K and V tiles' sizes
    FMHA_TILE_FN void init(uint32_t end, uint32_t kkey, uint32_t stride) {
        left = (int32_t)(end - kkey);
        k = tile_extent(left, stride);
        v = LAG ? tile_extent(left + 128, stride) : k;
    }
    FMHA_TILE_FN void advance(uint32_t stride) {
        left -= 128;
        if (LAG) v = k;
        k = tile_extent(left, stride);
        if (!LAG) v = k;
    }
};

#endif
