// quant_host.cpp - host side of the MXFP8 quantisers: the C ABI of include/mxfp8_quant.h.
//
// Argument checks, then launches of the kernels of quant_kernels.hip (embedded at build time, loaded once per
// device). No call allocates device memory; the V tensor scale keeps its partial maxima in the caller's descale buffer.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "../../include/mxfp8_quant.h"
#include "module_cache.h"

#ifndef MXQ_HSACO_PATH
#error "MXQ_HSACO_PATH must name the gfx950 code object built from quant_kernels.hip"
#endif
asm(".section .rodata.mxq_hsaco,\"a\",@progbits\n"
    ".balign 4096\n"
    ".global mxfp8_quant_hsaco_begin\n"
    "mxfp8_quant_hsaco_begin:\n"
    ".incbin \"" MXQ_HSACO_PATH "\"\n"
    ".global mxfp8_quant_hsaco_end\n"
    "mxfp8_quant_hsaco_end:\n"
    ".previous\n");
extern "C" const unsigned char mxfp8_quant_hsaco_begin[];
extern "C" const unsigned char mxfp8_quant_hsaco_end[];

namespace {

using fmha_internal::fail;

// The kernels' by-value argument structs (quant_kernels.hip).
struct QuantRowsArgs {
    const void* x;
    void* q;
    void* scale;
    uint64_t rows;
    float mul;
    uint32_t pad;
};
struct QuantTensorArgs {
    const void* x;
    void* q;
    void* descale;
    uint64_t n;
    uint32_t clear, pad;
};
struct QuantSeq32Args {
    const void* x;
    void* q;
    void* scale;
    uint32_t B, SK, HK, nblk;
    uint64_t tile0;
};
struct QuantQkvArgs {
    QuantRowsArgs q, k;
    QuantTensorArgs vt;
    QuantSeq32Args vs;
    void *q_slack, *k_slack;
    uint32_t q_slack_words, k_slack_words;
    uint32_t gq, gk, gv, seq32;
};
static_assert(sizeof(QuantQkvArgs) == 208, "qkv kernarg");
static_assert(sizeof(QuantRowsArgs) == 40, "rows kernarg");
static_assert(sizeof(QuantTensorArgs) == 40, "tensor kernarg");
static_assert(sizeof(QuantSeq32Args) == 48, "seq32 kernarg");

const char* const kQuantNames[5] = {
    "fmha_mxfp8_quant_rows", "fmha_mxfp8_quant_amax", "fmha_mxfp8_quant_tensor", "fmha_mxfp8_quant_seq32", "fmha_mxfp8_quant_qkv",
};
enum { Q_ROWS = 0, Q_AMAX = 1, Q_TENSOR = 2, Q_SEQ32 = 3, Q_QKV = 4 };
// quant_kernels.hip: the amax pass runs exactly 512 workgroups and leaves one partial maximum each in descale words
// [512, 1024); the descale buffer therefore spans 4096 bytes, the size the FMHA requires of it anyway.
constexpr uint32_t kAmaxGroups = 512;
constexpr uint64_t kDescaleBytes = 4096;

fmha_internal::ModuleCache<5> g_quant(mxfp8_quant_hsaco_begin, mxfp8_quant_hsaco_end, kQuantNames);

bool aligned(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

// Workgroups of the quantising pass over `chunks` 8-element chunks: enough to cover the chunks once, at most 4 per CU
// of a 256-CU part (each workgroup first reduces the 512 partial maxima, so fewer, longer workgroups read less).
uint32_t stride_grid(uint64_t chunks) {
    const uint64_t g = (chunks + 255) / 256;
    return (uint32_t)(g < 1 ? 1 : g > 1024 ? 1024 : g);
}

uint32_t rows_groups(int64_t rows) { return (uint32_t)((rows + 63) / 64); }   // 64 rows per workgroup

int check_rows(const void* x, const void* q, const void* scale, int64_t rows, uint64_t bytes_x, uint64_t bytes_q, uint64_t bytes_scale,
               char* err, size_t errlen) {
    if (rows < 1 || rows > (int64_t)0xFFFFFFFF * 64) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "rows outside [1, 2^38)");
    if (!x || !q || !scale) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "null pointer");
    if (!aligned(x, 16) || !aligned(q, 8) || !aligned(scale, 4))
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "x needs 16-byte, q 8-byte and scale 4-byte alignment");
    const uint64_t r = (uint64_t)rows;
    if (bytes_x < r * 256) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "x: buffer smaller than rows * 256 bytes");
    if (bytes_q < r * 128) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "q: buffer smaller than rows * 128 bytes");
    if (bytes_scale < r * 4) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "scale: buffer smaller than rows * 4 bytes");
    return FMHA_OK;
}

int check_tensor(const void* x, const void* q, const void* descale, int64_t n, uint64_t bytes_x, uint64_t bytes_q, uint64_t bytes_descale,
                 char* err, size_t errlen) {
    if (n < 8 || n % 8 != 0) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "n must be a positive multiple of 8");
    if (!x || !q || !descale) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "null pointer");
    if (!aligned(x, 16) || !aligned(q, 8) || !aligned(descale, 4))
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "x needs 16-byte, q 8-byte and descale 4-byte alignment");
    const uint64_t un = (uint64_t)n;
    if (bytes_x < un * 2) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "x: buffer smaller than n * 2 bytes");
    if (bytes_q < un) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "q: buffer smaller than n bytes");
    if (bytes_descale < kDescaleBytes) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "descale: buffer smaller than 4096 bytes");
    return FMHA_OK;
}

size_t seq32_bytes(int64_t B, int64_t SK, int64_t HK) {
    if (B < 1 || SK < 1 || HK < 1) return 0;
    return (size_t)((uint64_t)B * (uint64_t)((SK + 31) / 32) * (uint64_t)HK * 128u);
}

// one wave per 32-key tile, four to a workgroup
uint64_t seq32_tiles(int64_t B, int64_t SK, int64_t HK) { return (uint64_t)B * (uint64_t)((SK + 31) / 32) * (uint64_t)HK; }
uint64_t seq32_groups(int64_t B, int64_t SK, int64_t HK) { return (seq32_tiles(B, SK, HK) + 3) / 4; }
// Workgroups of 256 threads that one launch can have (its threads are counted in 32 bits).
constexpr uint64_t kMaxGroups = 0xFFFFFFFFull / 256;

int check_seq32(const void* x, const void* q, const void* scale, int32_t B, int32_t SK, int32_t HK, uint64_t bytes_x, uint64_t bytes_q,
                uint64_t bytes_scale, char* err, size_t errlen) {
    if (B < 1 || SK < 1 || HK < 1) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "B, SK, HK must be >= 1");
    if (!x || !q || !scale) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "null pointer");
    if (!aligned(x, 16) || !aligned(q, 8) || !aligned(scale, 8))
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "x needs 16-byte, q and scale 8-byte alignment");
    const uint64_t elems = (uint64_t)B * (uint64_t)SK * (uint64_t)HK * 128u;
    if (bytes_x < elems * 2) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "x: buffer smaller than B*SK*HK*256 bytes");
    if (bytes_q < elems) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "q: buffer smaller than B*SK*HK*128 bytes");
    if (bytes_scale < seq32_bytes(B, SK, HK))
        return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "scale: buffer smaller than B*ceil(SK/32)*HK*128 bytes");
    if ((seq32_tiles(B, SK, HK) + 15) / 16 > 0xFFFFFFFFull) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "tensor too large");
    return FMHA_OK;
}

int launch_seq32(QuantSeq32Args a, void* stream, char* err, size_t errlen) {
    const uint64_t groups = seq32_groups(a.B, a.SK, a.HK);
    for (uint64_t g = 0; g < groups; g += kMaxGroups) {
        a.tile0 = 4 * g;
        const int rc = g_quant.launch(Q_SEQ32, &a, sizeof(a), (uint32_t)std::min(kMaxGroups, groups - g), 1, 1, 256, stream, err, errlen);
        if (rc != FMHA_OK) return rc;
    }
    return FMHA_OK;
}

int quantize_tensor(const void* x, void* q, void* descale, int64_t n, bool clear, uint64_t bytes_x, uint64_t bytes_q, uint64_t bytes_descale,
                    void* stream, char* err, size_t errlen) {
    int rc = check_tensor(x, q, descale, n, bytes_x, bytes_q, bytes_descale, err, errlen);
    if (rc != FMHA_OK) return rc;
    QuantTensorArgs a = {x, q, descale, (uint64_t)n, clear ? 1u : 0u, 0u};
    rc = g_quant.launch(Q_AMAX, &a, sizeof(a), kAmaxGroups, 1, 1, 256, stream, err, errlen);
    if (rc == FMHA_OK) rc = g_quant.launch(Q_TENSOR, &a, sizeof(a), stride_grid((uint64_t)n / 8), 1, 1, 256, stream, err, errlen);
    return rc;
}

}  // namespace

extern "C" {

int fmha_mxfp8_quantize_rows(const void* x, void* q, void* scale, int64_t rows, float mul, uint64_t bytes_x, uint64_t bytes_q,
                             uint64_t bytes_scale, void* stream, char* err, size_t errlen) {
    const int rc = check_rows(x, q, scale, rows, bytes_x, bytes_q, bytes_scale, err, errlen);
    if (rc != FMHA_OK) return rc;
    QuantRowsArgs a = {x, q, scale, (uint64_t)rows, mul, 0u};
    return g_quant.launch(Q_ROWS, &a, sizeof(a), rows_groups(rows), 1, 1, 256, stream, err, errlen);
}

int fmha_mxfp8_quantize_tensor(const void* x, void* q, void* descale, int64_t n, uint64_t bytes_x, uint64_t bytes_q,
                               uint64_t bytes_descale, void* stream, char* err, size_t errlen) {
    return quantize_tensor(x, q, descale, n, false, bytes_x, bytes_q, bytes_descale, stream, err, errlen);
}

int fmha_mxfp8_quantize_v(const void* x, void* q, void* descale, int64_t n, uint64_t bytes_x, uint64_t bytes_q, uint64_t bytes_descale,
                          void* stream, char* err, size_t errlen) {
    return quantize_tensor(x, q, descale, n, true, bytes_x, bytes_q, bytes_descale, stream, err, errlen);
}

size_t fmha_mxfp8_seq32_scale_bytes(int64_t B, int64_t SK, int64_t HK) { return seq32_bytes(B, SK, HK); }

int fmha_mxfp8_quantize_seq32(const void* x, void* q, void* scale, int32_t B, int32_t SK, int32_t HK, uint64_t bytes_x,
                              uint64_t bytes_q, uint64_t bytes_scale, void* stream, char* err, size_t errlen) {
    const int rc = check_seq32(x, q, scale, B, SK, HK, bytes_x, bytes_q, bytes_scale, err, errlen);
    if (rc != FMHA_OK) return rc;
    return launch_seq32({x, q, scale, (uint32_t)B, (uint32_t)SK, (uint32_t)HK, (uint32_t)((SK + 31) / 32), 0u}, stream, err, errlen);
}

int fmha_mxfp8_quantize_qkv(const fmha_mxfp8_qkv_params* p, void* stream, char* err, size_t errlen) {
    if (!p) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "null params");
    if (p->B < 1 || p->S < 1 || p->H < 1 || p->SK < 1 || p->HK < 1)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "B, S, H, SK, HK must be >= 1");
    const int64_t rq = (int64_t)p->B * p->S * p->H, rk = (int64_t)p->B * p->SK * p->HK;
    int rc = check_rows(p->q, p->q8, p->q_scale, rq, p->bytes_q, p->bytes_q8, p->bytes_q_scale, err, errlen);
    if (rc == FMHA_OK) rc = check_rows(p->k, p->k8, p->k_scale, rk, p->bytes_k, p->bytes_k8, p->bytes_k_scale, err, errlen);
    if (rc == FMHA_OK)
        rc = p->v_seq32 ? check_seq32(p->v, p->v8, p->v_scale, p->B, p->SK, p->HK, p->bytes_v, p->bytes_v8, p->bytes_v_scale, err, errlen)
                        : check_tensor(p->v, p->v8, p->v_scale, rk * 128, p->bytes_v, p->bytes_v8, p->bytes_v_scale, err, errlen);
    if (rc != FMHA_OK) return rc;
    const uint64_t qsl = (p->bytes_q_scale - (uint64_t)rq * 4) / 4, ksl = (p->bytes_k_scale - (uint64_t)rk * 4) / 4;
    if (qsl > 0xFFFFFFFFull || ksl > 0xFFFFFFFFull) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "scale slack too large");
    QuantQkvArgs a;
    std::memset(&a, 0, sizeof(a));
    a.q = {p->q, p->q8, p->q_scale, (uint64_t)rq, p->q_mul, 0u};
    a.k = {p->k, p->k8, p->k_scale, (uint64_t)rk, 1.0f, 0u};
    a.vt = {p->v, p->v8, p->v_scale, (uint64_t)rk * 128, 1u, 0u};
    a.vs = {p->v, p->v8, p->v_scale, (uint32_t)p->B, (uint32_t)p->SK, (uint32_t)p->HK, (uint32_t)((p->SK + 31) / 32), 0u};
    a.q_slack = (char*)p->q_scale + rq * 4;
    a.k_slack = (char*)p->k_scale + rk * 4;
    a.q_slack_words = (uint32_t)qsl;
    a.k_slack_words = (uint32_t)ksl;
    const uint64_t gq = rows_groups(rq), gk = rows_groups(rk), gv = p->v_seq32 ? seq32_groups(p->B, p->SK, p->HK) : kAmaxGroups;
    const uint64_t gs = (qsl + 1023) / 1024 + (ksl + 1023) / 1024;
    a.seq32 = p->v_seq32 ? 1u : 0u;
    uint64_t grid = gs;
    if (gq + gk + gv + gs <= kMaxGroups) {
        a.gq = (uint32_t)gq;
        a.gk = (uint32_t)gk;
        a.gv = (uint32_t)gv;
        grid += gq + gk + gv;
    } else {   // more than one launch can have: one after the other, the slack by the launch below
        rc = g_quant.launch(Q_ROWS, &a.q, sizeof(a.q), (uint32_t)gq, 1, 1, 256, stream, err, errlen);
        if (rc == FMHA_OK) rc = g_quant.launch(Q_ROWS, &a.k, sizeof(a.k), (uint32_t)gk, 1, 1, 256, stream, err, errlen);
        if (rc == FMHA_OK)
            rc = p->v_seq32 ? launch_seq32(a.vs, stream, err, errlen)
                            : g_quant.launch(Q_AMAX, &a.vt, sizeof(a.vt), kAmaxGroups, 1, 1, 256, stream, err, errlen);
    }
    if (rc == FMHA_OK && grid) rc = g_quant.launch(Q_QKV, &a, sizeof(a), (uint32_t)grid, 1, 1, 256, stream, err, errlen);
    if (rc == FMHA_OK && !p->v_seq32)
        rc = g_quant.launch(Q_TENSOR, &a.vt, sizeof(a.vt), stride_grid((uint64_t)rk * 16), 1, 1, 256, stream, err, errlen);
    return rc;
}

}  // extern "C"
