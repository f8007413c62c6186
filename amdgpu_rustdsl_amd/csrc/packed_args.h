// packed_args.h - kernel arguments of the packed-rows kernel and of the 256-row kernel with split last blocks, shared by
// host and device code. Include fmha_mxfp8.h first.
#ifndef FMHA_PACKED_ARGS_H
#define FMHA_PACKED_ARGS_H

#include <stdint.h>

// `flags`: FMHA_FLAG_CAUSAL and FMHA_FLAG_V_SEQ32 as in fmha_mxfp8_args, and
enum { kPackedF32 = 0x100u,      // partial rows in f32 (512 B) instead of fp16 (256 B)
       kPackedWhole = 0x200u };  // the softmax reference is taken over whole 128-key tiles (else over each 64-key half)

typedef struct fmha_packed_args {
    const void *q, *k, *v, *qs, *ks, *vd;
    void *ohat, *lse;        // partial rows and their base-2 LSE, row (b S + s) H + h of each of parts x sub splits
    uint32_t S, SK, H, HK;
    float softmax_scale;     // at 0x50, where the `_scaled` kernels read it
    uint32_t gshift;         // log2(H / HK)
    uint32_t parts, sub;     // the reference's key ranges, and how many blocks share each
    uint32_t groups;         // B parts sub (the grid is HK x row tiles x groups)
    uint32_t rows_total;     // B S H
    uint32_t flags;
} fmha_packed_args;

typedef struct fmha_tail_args {
    fmha_mxfp8_args base;
    void *ohat, *lse;        // f32 partial rows and base-2 LSE, row (range x ntail + block) x 256 + row of the block
    uint32_t nfull, ntail;   // blocks that run whole, blocks cut into `sub` ranges
    uint32_t sub, pad;
} fmha_tail_args;

#endif
