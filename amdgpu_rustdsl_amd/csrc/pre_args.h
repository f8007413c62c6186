// pre_args.h - kernel arguments of the kernels that the one-call entry launches itself, shared by host and device code.
#ifndef FMHA_PRE_ARGS_H
#define FMHA_PRE_ARGS_H

#include <stdint.h>

// Bits of `extra` above a kernel's counts: the KV split (split count in bits 0..15) and the packed rows (parts in bits 0..7,
// shares in bits 8..12)
enum { kPreF32 = 0x10000u,      // partial rows in f32 (512 B) instead of fp16 (256 B)
       kPreWhole = 0x20000u,    // packed rows: the softmax reference over whole 128-key tiles (else over each 64-key half)
       kPreByXcd = 0x40000u };  // the placement by XCD applies: B x splits is a multiple of 8 (KV split: and one query tile)

// The first fourteen dwords are preloaded into SGPRs. Addresses are 48 bits: the low words, then the high halves in pairs.
// heads: H in bits 0..15, log2(H / HK) in 16..19, FMHA_FLAG_* in 24..27. rows_total (B S H) and o / lse as partial rows and
// their base-2 LSE where the kernel writes partials. extra of the split last blocks: whole blocks << 12 | split ones << 4 |
// ranges of each.
typedef struct fmha_pre_args {
    uint32_t q_lo, k_lo, v_lo, qs_lo, ks_lo, vd_lo, hi_qk, hi_vqs, hi_ksvd;
    uint32_t S, SK, heads;
    float scale;
    uint32_t extra;
    void *o, *lse;
    uint32_t rows_total, pad;
    void *out, *lse_out;   // the split last blocks' whole ones: output rows and natural-log LSE
} fmha_pre_args;

#endif
