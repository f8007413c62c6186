// fmha_host.cpp - host side of the MXFP8 FMHA forward: the C ABI of include/fmha_mxfp8.h.
//
// The host contract (validate), the dispatch rule, the kernarg filling and the launches through
// hipModuleLaunchKernel with HIP_LAUNCH_PARAM_BUFFER_POINTER, exactly the way the reference's generated
// headers launch its kernels (tests/gpu/generated/fmha_fwd_hd128_mxfp8_v3_vs128_abi.h:204-209). The gfx950
// code object (fmha_kernels.hip) is embedded in this library at build time and loaded once per device with
// hipModuleLoadData. No function allocates device memory; the KV-split workspace is the caller's.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <atomic>
#include <cstdlib>

#include "../../include/fmha_mxfp8.h"
#include "module_cache.h"
#include "pre_args.h"

static_assert(sizeof(fmha_mxfp8_args) == 656, "kernarg size (vs128_abi.h:126)");
static_assert(sizeof(fmha_mxfp8_params) == 192, "params layout (lib.py mirrors it)");
static_assert(offsetof(fmha_mxfp8_args, ptr_o) == 0x000, "ptr_o");
static_assert(offsetof(fmha_mxfp8_args, ptr_q) == 0x010, "ptr_q");
static_assert(offsetof(fmha_mxfp8_args, ptr_k) == 0x020, "ptr_k");
static_assert(offsetof(fmha_mxfp8_args, ptr_v) == 0x030, "ptr_v");
static_assert(offsetof(fmha_mxfp8_args, ptr_lse) == 0x040, "ptr_lse");
static_assert(offsetof(fmha_mxfp8_args, softmax_scale) == 0x050, "scale");
static_assert(offsetof(fmha_mxfp8_args, s_seq_len) == 0x060, "s_seq_len");
static_assert(offsetof(fmha_mxfp8_args, s_Seqs) == 0x070, "s_Seqs");
static_assert(offsetof(fmha_mxfp8_args, s_Hs) == 0x090, "s_Hs");
static_assert(offsetof(fmha_mxfp8_args, s_Bs) == 0x0A0, "s_Bs");
static_assert(offsetof(fmha_mxfp8_args, s_gqa) == 0x0B0, "s_gqa");
static_assert(offsetof(fmha_mxfp8_args, s_k_Seqs) == 0x0C0, "s_k_Seqs");
static_assert(offsetof(fmha_mxfp8_args, s_k_Hs) == 0x0D0, "s_k_Hs");
static_assert(offsetof(fmha_mxfp8_args, s_k_Bs) == 0x0E0, "s_k_Bs");
static_assert(offsetof(fmha_mxfp8_args, opt) == 0x0F0, "opt");
static_assert(offsetof(fmha_mxfp8_args, s_kv_seq_len) == 0x110, "s_kv_seq_len");
static_assert(offsetof(fmha_mxfp8_args, s_q_head_num) == 0x140, "s_q_head_num");
static_assert(offsetof(fmha_mxfp8_args, s_v_Seqs) == 0x150, "s_v_Seqs");
static_assert(offsetof(fmha_mxfp8_args, s_v_Hs) == 0x160, "s_v_Hs");
static_assert(offsetof(fmha_mxfp8_args, s_v_Bs) == 0x170, "s_v_Bs");
static_assert(offsetof(fmha_mxfp8_args, s_o_Seqs) == 0x180, "s_o_Seqs");
static_assert(offsetof(fmha_mxfp8_args, s_o_Hs) == 0x190, "s_o_Hs");
static_assert(offsetof(fmha_mxfp8_args, s_o_Bs) == 0x1A0, "s_o_Bs");
static_assert(offsetof(fmha_mxfp8_args, ptr_q_descale) == 0x200, "ptr_q_descale");
static_assert(offsetof(fmha_mxfp8_args, ptr_k_descale) == 0x210, "ptr_k_descale");
static_assert(offsetof(fmha_mxfp8_args, ptr_v_descale) == 0x220, "ptr_v_descale");
static_assert(offsetof(fmha_mxfp8_args, s_descale_q_Bs) == 0x230, "s_descale_q_Bs");
static_assert(offsetof(fmha_mxfp8_args, s_descale_q_Hs) == 0x240, "s_descale_q_Hs");
static_assert(offsetof(fmha_mxfp8_args, s_descale_k_Bs) == 0x250, "s_descale_k_Bs");
static_assert(offsetof(fmha_mxfp8_args, s_descale_k_Hs) == 0x260, "s_descale_k_Hs");
static_assert(offsetof(fmha_mxfp8_args, flags) == 0x280, "flags / abi_tail");
static_assert(sizeof(fmha_mxfp8_kvsplit_args) == 648, "kvsplit kernarg size (kvsplit_abi.h:136)");
static_assert(offsetof(fmha_mxfp8_kvsplit_args, ptr_ohat) == 0x270, "ptr_ohat");
static_assert(offsetof(fmha_mxfp8_kvsplit_args, ptr_lse) == 0x278, "ptr_lse");
static_assert(offsetof(fmha_mxfp8_kvsplit_args, kvs_splits) == 0x280, "kvs_splits");
static_assert(offsetof(fmha_mxfp8_kvsplit_args, kvs_rows_total) == 0x284, "kvs_rows_total");
static_assert(sizeof(fmha_mxfp8_combine_args) == 36, "combine kernarg size (combine8h_abi.h:34)");
static_assert(offsetof(fmha_mxfp8_combine_args, rows_total) == 0x18, "rows_total");
static_assert(offsetof(fmha_mxfp8_combine_args, splits) == 0x20, "splits");

// The code object, embedded by the build (FMHA_HSACO_PATH names the file built from fmha_kernels.hip).
#ifndef FMHA_HSACO_PATH
#error "FMHA_HSACO_PATH must name the gfx950 code object built from fmha_kernels.hip"
#endif
asm(".section .rodata.fmha_hsaco,\"a\",@progbits\n"
    ".balign 4096\n"
    ".global fmha_mxfp8_hsaco_begin\n"
    "fmha_mxfp8_hsaco_begin:\n"
    ".incbin \"" FMHA_HSACO_PATH "\"\n"
    ".global fmha_mxfp8_hsaco_end\n"
    "fmha_mxfp8_hsaco_end:\n"
    ".previous\n");
extern "C" const unsigned char fmha_mxfp8_hsaco_begin[];
extern "C" const unsigned char fmha_mxfp8_hsaco_end[];

namespace {

using fmha_internal::fail;
using fmha_internal::set_err;

const char* const kKernelNames[27] = {
    "fmha_fwd_hd128_mxfp8_v3_vs128",
    "fmha_fwd_hd128_mxfp8_v3_t128",
    "fmha_fwd_hd128_mxfp8_v3_kvsplit",
    "fmha_fwd_hd128_mxfp8_v3_kvsplit_combine8h",
    // extension kernels: the softmax scale at 0x050 applied in the kernel (FMHA_FLAG_SCALE / FMHA_KVS_SCALE)
    "fmha_fwd_hd128_mxfp8_v3_vs128_scaled",
    "fmha_fwd_hd128_mxfp8_v3_t128_scaled",
    "fmha_fwd_hd128_mxfp8_v3_kvsplit_scaled",
    // extension kernels: t128's grid with 512 threads, the two wave groups splitting each tile's keys
    "fmha_fwd_hd128_mxfp8_v3_t128_split_tiles",
    "fmha_fwd_hd128_mxfp8_v3_t128_split_tiles_scaled",
    // extension kernel: the combine with the splits spread over 4 waves (more than 8 partials per row)
    "fmha_fwd_hd128_mxfp8_v3_kvsplit_combine_wide",
    // extension kernels: short query ranges, the rows of a KV head's query heads packed; the merge with the LSE output
    "fmha_fwd_hd128_mxfp8_pre_packed",
    "fmha_fwd_hd128_mxfp8_pre_packed_scaled",
    "fmha_fwd_hd128_mxfp8_v3_combine_lse",
    // extension kernels: the 256-row kernel with split last blocks, and their merge
    "fmha_fwd_hd128_mxfp8_pre_vs128_tail",
    "fmha_fwd_hd128_mxfp8_pre_vs128_tail_scaled",
    "fmha_fwd_hd128_mxfp8_v3_tail_combine",
    // extension kernels: the bodies of the kernels above on preloaded parameters (fmha_pre_args)
    "fmha_fwd_hd128_mxfp8_pre_vs128",
    "fmha_fwd_hd128_mxfp8_pre_vs128_scaled",
    "fmha_fwd_hd128_mxfp8_pre_split_tiles",
    "fmha_fwd_hd128_mxfp8_pre_split_tiles_scaled",
    "fmha_fwd_hd128_mxfp8_pre_t128",
    "fmha_fwd_hd128_mxfp8_pre_t128_lut",
    "fmha_fwd_hd128_mxfp8_pre_kvsplit",
    "fmha_fwd_hd128_mxfp8_pre_packed_seq32",
    "fmha_fwd_hd128_mxfp8_pre_packed_scaled_seq32",
    "fmha_fwd_hd128_mxfp8_pre_vs128_tail_seq32",
    "fmha_fwd_hd128_mxfp8_pre_vs128_tail_scaled_seq32",
};
enum { K_VS128 = 0, K_T128 = 1, K_KVSPLIT = 2, K_COMBINE = 3, K_VS128_SC = 4, K_T128_SC = 5, K_KVSPLIT_SC = 6, K_T128ST = 7,
       K_T128ST_SC = 8, K_COMBINE_WIDE = 9, K_PACKED = 10, K_PACKED_SC = 11, K_COMBINE_LSE = 12,
       K_TAIL = 13, K_TAIL_SC = 14, K_TAIL_COMBINE = 15, K_PRE_VS128 = 16, K_PRE_VS128_SC = 17, K_PRE_T128ST = 18, K_PRE_T128ST_SC = 19,
       K_PRE_T128 = 20, K_PRE_T128_LUT = 21, K_PRE_KVSPLIT = 22, K_PACKED_VS = 23, K_PACKED_SC_VS = 24,
       K_TAIL_VS = 25, K_TAIL_SC_VS = 26 };

// The 128-row grids (t128's shapes, and vs128's half-chip and causal ones below) run on the split-tile kernel (512
// threads) from 7 key tiles on, and on the one-wave-per-SIMD kernel (256 threads, the reference's order) below that:
// with 4 to 6 key tiles the single-wave kernel is faster (measured on MI355X, us: B1H8S512 9.11 against 9.92,
// B1H8S1024 SK768 11.52 against 11.73, B4H8S512 9.45 against 10.28, B8H8S512 9.78 against 10.75; at SK1024 13.78
// against 13.16), and with fewer than 4 (the LUT recipe, state.rs:75-77) it keeps the reference's order. Causal
// shapes take the split-tile kernel from 4 key tiles on (unpaired it is ahead: B1H8S1024 causal 13.56 against 14.45)
// except on grids the causal q-tile pairing halves (more 128-row blocks than CUs) with at most 8 key tiles, where the
// single-wave kernel runs each pair faster (B16H8S512 15.13 against 17.07, B8H8S768 16.94 against 18.34, B8H8S1024
// 19.45 against 20.13; at 16 tiles, B4H8S2048, 28.37 against 26.63). The choice does not depend on the causal_pair
// field, so a forced pairing gives the same kernel, and so the same bits, as the automatic one.
int cu_count();
bool use_split_tiles(int64_t B, int64_t H, int64_t S, int64_t SK, bool causal) {
    const int64_t tiles = (SK + 127) / 128;
    if (!causal) return tiles >= 7;
    if (tiles < 4) return false;
    return !(tiles <= 8 && (S + 127) / 128 * H * B > (int64_t)cu_count());
}

// The one-call entry also runs the vs128 path on the 128-row grid when its 256-row grid holds at most 128 blocks (half
// of the 256 CUs or fewer): there the same shape fills twice the CUs. The kernel is chosen as for t128 (above). Below the
// split-tile threshold the 256-thread t128 kernel gives the vs128 kernel's order and bits
// (both take every tile whole) on twice the blocks; measured with the LUT recipe at B4H8S1024 SK256, B2H8S2048 SK384
// and B1H8S4096 SK128: 10.4 / 12.6 / 7.7 us against 11.9 / 14.3 / 9.5 (above 128 blocks of 256 rows the vs128 kernel
// stays ahead: B8H8S2048 SK256 25.4 against 36.4 us). The direct vs128 launcher keeps the 256-row kernel its grid names.
// Causal (extension): always from 4 key tiles on, so that the 128-row grid's causal q-tile pairing is available past one
// wave of blocks, except where the 256-row kernel gives the same bits sooner: grids of more 256-row blocks than CUs with
// 4 to 8 key tiles, whose 128-row form is the 256-thread kernel. With its heaviest query tiles first the 256-row kernel
// balances as well as the pairs do (us, 128-row / 256-row: B8 H16 S600 30.7 / 26.9, B9 H8 S1000 36.6 / 34.7, B16 H8 S1024
// 39.3 / 37.7; S < SK: B33 H8 S400 SK512 51.2 / 36.6, B16 H8 S768 SK1024 42.5 / 34.9, B40 H8 S140 SK1000 58.0 / 36.3; with V
// scales per 32 keys and the in-kernel scale the same way round). With at most 128 query rows half of
// its block is padding (B64 H8 S128 SK1024 38.4 / 40.9). A caller that asks for the pairing has it. From 9 key tiles on the 128-row
// form is the split-tile kernel, whose error against float64 is the smaller one (relative, split-tile / 256-row, three
// seeds each: B8 H8 S1152 0.0241 / 0.0245, S2048 0.0249 / 0.0252, B1 H32 HK8 S6144 0.0261 / 0.0264): it stays, though the
// 256-row kernel takes 147 us for the last of them and it 175.
bool vs128_on_128row_grid(int64_t B, int64_t H, int64_t S, int64_t SK, bool causal, bool pair_asked = false) {
    const int64_t blocks = (S + 255) / 256 * H * B;
    const int64_t tiles = (SK + 127) / 128;
    if (blocks <= 128) return true;
    if (!causal || tiles < 4) return false;
    return tiles > 8 || S <= 128 || blocks <= (int64_t)cu_count() || pair_asked;
}

fmha_internal::ModuleCache<27> g_fmha(fmha_mxfp8_hsaco_begin, fmha_mxfp8_hsaco_end, kKernelNames);

int get_functions(hipFunction_t** out, char* err, size_t errlen) { return g_fmha.get(out, err, errlen); }

int launch_raw(int which, const void* args, size_t nbytes, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t block,
               void* stream, char* err, size_t errlen) {
    return g_fmha.launch(which, args, nbytes, gx, gy, gz, block, stream, err, errlen);
}

typedef long long i64;

// The 0x000-0x26F rules shared by vs128 / t128 / kvsplit (vs128_abi.h:170-203), in the reference's four groups
// and order: buffer extents, kernarg ranges, kernarg relations, grid. `B` is grid.z for the single-kernel launches
// and the host symbol B for the KV split (kvsplit_abi.h).
// v_seq32: the per-32-key V-scale extension, whose ptr_v_descale holds E8M0 [B, ceil(SK/32), HK, 128]
int rules_extent(const fmha_mxfp8_args& a, const fmha_mxfp8_buffer_sizes& sz, i64 B, bool v_seq32, char* err, size_t errlen) {
    const i64 H = a.s_q_head_num;
    if (sz.ptr_q < (uint64_t)(B * (i64)a.s_Bs)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_q: buffer ptr_q smaller than declared allocation");
    if (sz.ptr_k < (uint64_t)(B * (i64)a.s_k_Bs)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_k: buffer ptr_k smaller than declared allocation");
    if (sz.ptr_v < (uint64_t)(B * (i64)a.s_v_Bs)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_v: buffer ptr_v smaller than declared allocation");
    if (sz.ptr_o < (uint64_t)(B * (i64)a.s_o_Bs)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_o: buffer ptr_o smaller than declared allocation");
    if (sz.ptr_q_descale < (uint64_t)(B * (i64)a.s_descale_q_Bs + 2048LL * H))
        return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_q_descale: buffer ptr_q_descale smaller than declared allocation");
    if (sz.ptr_k_descale < (uint64_t)(B * (i64)a.s_descale_k_Bs + 2560LL * H))
        return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_k_descale: buffer ptr_k_descale smaller than declared allocation");
    const uint64_t vd_need = v_seq32 ? (uint64_t)(B * (((i64)a.s_kv_seq_len + 31) / 32) * (i64)a.s_k_Seqs) : 4096ull;
    if (sz.ptr_v_descale < vd_need) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_v_descale: buffer ptr_v_descale smaller than declared allocation");
    return FMHA_OK;
}

int rules_range(const fmha_mxfp8_args& a, char* err, size_t errlen) {
    const i64 gqa = a.s_gqa;
    if (gqa < 1 || gqa > 16) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0xB0) outside contract");
    if (a.s_seq_len < 1) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x60) outside contract");
    if (a.s_kv_seq_len < 1) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x110) outside contract");
    if (a.s_Hs != 128) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x90) outside contract");
    if (a.s_k_Hs != 128) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0xD0) outside contract");
    if (a.s_v_Hs != 128) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x160) outside contract");
    if (a.s_o_Hs != 256) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x190) outside contract");
    if (a.s_descale_q_Hs != 4) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x240) outside contract");
    if (a.s_descale_k_Hs != 4) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x260) outside contract");
    return FMHA_OK;
}

int rules_is(const fmha_mxfp8_args& a, i64 HK, char* err, size_t errlen) {
    const i64 S = a.s_seq_len, SK = a.s_kv_seq_len, H = a.s_q_head_num;
    if (H != HK * (i64)a.s_gqa) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x140) relation failed");
    if ((i64)a.s_Seqs != H * 128) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x70) relation failed");
    if ((i64)a.s_Bs != S * (i64)a.s_Seqs) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0xA0) relation failed");
    if ((i64)a.s_k_Seqs != HK * 128) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0xC0) relation failed");
    if ((i64)a.s_k_Bs != SK * (i64)a.s_k_Seqs) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0xE0) relation failed");
    if (a.s_v_Seqs != a.s_k_Seqs) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x150) relation failed");
    if (a.s_v_Bs != a.s_k_Bs) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x170) relation failed");
    if ((i64)a.s_o_Seqs != H * 256) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x180) relation failed");
    if ((i64)a.s_o_Bs != S * (i64)a.s_o_Seqs) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x1A0) relation failed");
    if ((i64)a.s_descale_q_Bs != S * H * 4) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x230) relation failed");
    if ((i64)a.s_descale_k_Bs != SK * HK * 4) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x250) relation failed");
    return FMHA_OK;
}

int rules_grid(const fmha_mxfp8_args& a, uint32_t gx, uint32_t gy, int rows_per_block, char* err, size_t errlen) {
    if ((i64)gy != (i64)a.s_q_head_num) return fail(err, errlen, FMHA_ERR_GRID, "GV-HOST-GRID", "grid axis 1 relation failed");
    i64 want = ((i64)a.s_seq_len + rows_per_block - 1) / rows_per_block;
    if (a.flags & FMHA_FLAG_CAUSAL_PAIR) want = (want + 1) / 2;   // the causal q-tile pairing: two tiles per block
    if ((i64)gx != want) return fail(err, errlen, FMHA_ERR_GRID, "GV-HOST-GRID", "grid axis 0 relation failed");
    return FMHA_OK;
}

// Compute units of the current device (the causal pairing pays off only when the unpaired grid exceeds them), cached
// FMHA_MXFP8_CU_COUNT (a positive integer) replaces the device's count: the CU-dependent rules (the KV fill, the
// causal pairing, the causal split-tile choice) and so the output bits can then be checked for another part's count,
// also on a machine without a GPU.
int cu_count() {
    static const int env = [] {
        const char* e = std::getenv("FMHA_MXFP8_CU_COUNT");
        return e ? std::atoi(e) : 0;
    }();
    if (env > 0) return env;
    static std::atomic<int> cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cache[dev].load(std::memory_order_relaxed);
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cache[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// The in-kernel softmax scale (FMHA_FLAG_SCALE / FMHA_KVS_SCALE): c = f32(scale log2 e) must be a positive normal f32
// (its exponent then splits off exactly, and the Q scale exponents shift by it)
bool scale_ok(float scale) {
    const float c = scale * 1.44269504088896340736f;
    return std::isfinite(c) && std::isnormal(c) && c > 0.0f;
}
int rules_scale(const fmha_mxfp8_args& a, bool on, char* err, size_t errlen) {
    float scale;
    std::memcpy(&scale, &a.softmax_scale, 4);
    if (on && !scale_ok(scale))
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x50) outside contract (softmax scale)");
    return FMHA_OK;
}

int validate_base(const fmha_mxfp8_args& a, const fmha_mxfp8_buffer_sizes& sz, uint32_t gx, uint32_t gy, i64 B, i64 HK,
                  int rows_per_block, char* err, size_t errlen) {
    int rc;
    if ((rc = rules_extent(a, sz, B, (a.flags & FMHA_FLAG_V_SEQ32) != 0, err, errlen)) != FMHA_OK) return rc;
    if ((rc = rules_range(a, err, errlen)) != FMHA_OK) return rc;
    if ((a.flags & ~(FMHA_FLAG_CAUSAL | FMHA_FLAG_V_SEQ32 | FMHA_FLAG_SCALE | FMHA_FLAG_CAUSAL_PAIR)) != 0 ||
        ((a.flags & FMHA_FLAG_CAUSAL_PAIR) && !(a.flags & FMHA_FLAG_CAUSAL)))
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x280) outside contract");
    if ((rc = rules_scale(a, (a.flags & FMHA_FLAG_SCALE) != 0, err, errlen)) != FMHA_OK) return rc;
    if ((rc = rules_is(a, HK, err, errlen)) != FMHA_OK) return rc;
    return rules_grid(a, gx, gy, rows_per_block, err, errlen);
}

bool empty_split(i64 SK, i64 splits) {
    const i64 ntiles = (SK + 127) / 128;
    const i64 tps = (ntiles + splits - 1) / splits;
    return !((splits - 1) * tps < ntiles);
}

// KV-split fill (extension): the reference's `splits` chunks, each divided into `sub` consecutive key ranges, so that
// a grid of few blocks fills the CUs. sub doubles (up to 8) while the grid stays within the CU count and every range
// keeps at least 4 key tiles (the recipe of the reference's splits, which have at least 4). The combine merges the
// splits x sub partials.
i64 kv_fill(i64 B, i64 H, i64 S, i64 SK, i64 splits) {
    const i64 blocks = (S + 255) / 256 * H * B * splits, tiles = (SK + 127) / 128;
    i64 sub = 1;
    while (sub < 8 && blocks * sub * 2 <= (i64)cu_count() && tiles >= 4 * splits * sub * 2 && !empty_split(SK, splits * sub * 2))
        sub *= 2;
    return sub;
}

// The packed-rows kernel (extension) for short query ranges: the shares `sub` that each of the `parts` key ranges is cut
// into, or 0 to keep the path's own kernel. The rule compares estimated times (us, measured on MI355X):
// - a block costs kBlock besides its tiles: arguments, first loads, epilogue;
// - a 128-key tile costs a split-tile block kTile (less with idle waves: up to 96 rows), the 256-row kernel kTileWhole, and at
//   least what its 32 KiB take at the 5 TB/s that the chip reads when `readers` blocks stream distinct keys;
// - a merge that the path would not run anyway costs kMerge, and the partials their bytes, written and read back.
// Measured against the path's own kernels (kernel times without / with it): B8 H32 HK8 S1 SK8192 96 / 32.1 + merge 3.9,
// SK1024 19.0 / 10.0 + 3.4; B8 H32 HK8 S16 SK2048 28.3 / 14.0 + 3.8; KV split B1 H32 HK8 S1 SK16384 23.1 / 12.0,
// B4 H16 HK4 S16 SK5000 17.9 / 11.3, B4 H8 HK1 S64 SK8192 16.5 / 12.4, B1 H8 S128 SK16000 15.3 / 13.7.
// No gain, so the rule keeps the own kernel: full grids of 128-row blocks (B8 H8 S128 SK4096: 18.0 either way).
i64 packed_sub(i64 B, i64 H, i64 HK, i64 S, i64 SK, i64 parts, bool whole, bool split_path, bool f32, i64 own_blocks, i64 max_parts) {
    constexpr double kBlock = 6.0, kTile = 1.05, kTileIdle = 0.9, kTileWhole = 1.5, kMerge = 5.0, kReadTile = 0.0065, kBytes = 1.0e7;
    const i64 tiles = (SK + 127) / 128, cus = cu_count(), rows = S * (H / HK), qtiles = (rows + 127) / 128;
    if (S > 128 || tiles < 8) return 0;
    const i64 t = (tiles + parts - 1) / parts, n = qtiles * HK * B * parts;
    auto cost = [&](i64 blocks, i64 sharers, i64 per, double tile, i64 partials, double merge) {
        const double readers = (double)std::min(blocks, cus) / (double)sharers;
        const double bytes = partials ? 2.0 * (double)(partials * B * S * H) * (f32 ? 512.0 : 256.0) : 0.0;
        return (double)((blocks + cus - 1) / cus) * ((double)per * std::max(tile, readers * kReadTile) + kBlock) + merge + bytes / kBytes;
    };
    double best = cost(own_blocks, H / HK, t, whole ? kTileWhole : kTile, split_path ? parts : 0, 0.0) - 0.5;
    i64 sub = 0;
    for (i64 s = 1; s <= 16 && s <= t && s * parts <= max_parts; ++s) {
        const double c = cost(n * s, qtiles, (t + s - 1) / s, rows <= 96 ? kTileIdle : kTile, parts * s, split_path ? 0.0 : kMerge);
        if (c < best) {
            best = c;
            sub = s;
        }
    }
    return sub;
}

// The 256-row grid with split last blocks (extension): the ranges `sub` that each block past the last whole round of CUs is
// cut into, or 0. n blocks of t tiles on c CUs take ceil(n / c) rounds; with at most half the CUs busy in the last one,
// cutting its blocks into up to c / (n mod c) ranges shortens that round, for a merge and the partials' bytes; the rule
// takes the count with the least estimated time. Measured on MI355X, us per call whole / cut: B3 H8 S3001 (288 blocks
// of 24 tiles) 81.0 / 67.3 with 4 ranges (2: 73.3, 8: 69.9), B1 H32 HK8 S2049 56.9 / 53.3, B1 H12 S6000 158.0 / 117.3,
// B1 H9 S8192 183.8 / 139.3; where the rule keeps them whole a cut loses: 384 blocks of 24 tiles 79.8 / 83.3, 288 of 9
// tiles 40.0 / 40.5, 320 of 16 57.0 / 57.3.
i64 tail_sub(i64 blocks, i64 tiles) {
    constexpr double kBlock = 6.0, kTile = 1.5, kMerge = 5.0, kBytes = 4.0e6;
    const i64 cus = cu_count(), rem = blocks % cus;
    if (blocks < cus || rem == 0 || tiles < 8) return 0;
    double best = (double)tiles * kTile + kBlock - 1.0;
    i64 sub = 0;
    for (i64 s = 2; s <= 8 && s * rem <= cus; ++s) {
        // the seed tile counts for one; each partial row is written and read back
        const double c = (double)((tiles + s - 1) / s + 1) * kTile + kBlock + kMerge + (double)(rem * s * 256 * 1024) / kBytes;
        if (c < best) {
            best = c;
            sub = s;
        }
    }
    return sub;
}
size_t tail_bytes(i64 rem, i64 sub) { return (size_t)(rem * sub * 256) * 516u; }

// The preloaded parameters of a call (pre_args.h), or false where they cannot hold it: more than 65535 heads (the grid's
// limit too), or an address past 48 bits.
bool fill_pre(fmha_pre_args& x, const fmha_mxfp8_params& p, uint32_t flags, void* o, void* lse) {
    const uint64_t a[6] = {(uint64_t)(uintptr_t)p.q,         (uint64_t)(uintptr_t)p.k,         (uint64_t)(uintptr_t)p.v,
                           (uint64_t)(uintptr_t)p.q_descale, (uint64_t)(uintptr_t)p.k_descale, (uint64_t)(uintptr_t)p.v_descale};
    for (uint64_t u : a)
        if (u >> 48) return false;
    if (p.H > 65535) return false;
    std::memset(&x, 0, sizeof(x));
    x.q_lo = (uint32_t)a[0]; x.k_lo = (uint32_t)a[1]; x.v_lo = (uint32_t)a[2];
    x.qs_lo = (uint32_t)a[3]; x.ks_lo = (uint32_t)a[4]; x.vd_lo = (uint32_t)a[5];
    x.hi_qk = (uint32_t)(a[0] >> 32) | (uint32_t)(a[1] >> 32) << 16;
    x.hi_vqs = (uint32_t)(a[2] >> 32) | (uint32_t)(a[3] >> 32) << 16;
    x.hi_ksvd = (uint32_t)(a[4] >> 32) | (uint32_t)(a[5] >> 32) << 16;
    x.S = (uint32_t)p.S;
    x.SK = (uint32_t)p.SK;
    uint32_t sh = 0;
    while ((p.HK << sh) < p.H) ++sh;
    x.heads = (uint32_t)p.H | sh << 16 | flags << 24;
    x.scale = p.softmax_scale;
    x.o = o;
    x.lse = lse;
    x.rows_total = (uint32_t)((i64)p.B * p.S * p.H);
    return true;
}
static_assert(sizeof(fmha_pre_args) == 96 && offsetof(fmha_pre_args, o) == 56 && offsetof(fmha_pre_args, out) == 80, "preloaded kernarg");

// The preloaded kernel that runs the body of a full-sequence kernel, or -1: the short recipe (fewer than 4 key tiles), the
// per-32-key V scales, the causal pairing and the causal single-wave blocks stay with the packed ABI's kernels.
int pre_kernel(int kern, i64 tiles, uint32_t flags) {
    if (flags & (FMHA_FLAG_V_SEQ32 | FMHA_FLAG_CAUSAL_PAIR)) return -1;
    if (kern == K_T128) return (flags & FMHA_FLAG_CAUSAL) ? -1 : tiles < 4 ? K_PRE_T128_LUT : K_PRE_T128;
    if (tiles < 4) return -1;
    switch (kern) {
        case K_VS128: return K_PRE_VS128;
        case K_VS128_SC: return K_PRE_VS128_SC;
        case K_T128ST: return K_PRE_T128ST;
        case K_T128ST_SC: return K_PRE_T128ST_SC;
        default: return -1;
    }
}

// What the one-call entry runs for a shape: the resolved path, and for the packed-rows kernel its shares.
struct Plan {
    int path, splits;   // as the entry reports them
    i64 parts;          // KV-split partials (chunks x fill), 1 off the KV split
    i64 sub;            // packed-rows shares of each partial's range; 0: the path's own kernel
    bool whole;         // packed rows: the softmax reference over whole tiles
    i64 tail, tail_blocks;   // 256-row grid: ranges per split last block (0: none) and how many blocks are split
    int kern;           // the path's own kernel (full-sequence paths)
    uint32_t block, gx;
};

int kernel_of(int path, i64 B, i64 H, i64 S, i64 SK, bool causal, bool pair_asked, bool scaled, uint32_t* block, uint32_t* gx) {
    if (path == FMHA_PATH_VS128 && !vs128_on_128row_grid(B, H, S, SK, causal, pair_asked)) {
        *block = 512u;
        *gx = (uint32_t)((S + 255) / 256);
        return scaled ? K_VS128_SC : K_VS128;
    }
    // t128, or vs128 on the 128-row grid (same kernarg layout): the split-tile kernel or the 256-thread one
    const bool st = use_split_tiles(B, H, S, SK, causal);
    *block = st ? 512u : 256u;
    *gx = (uint32_t)((S + 127) / 128);
    return st ? (scaled ? K_T128ST_SC : K_T128ST) : (scaled ? K_T128_SC : K_T128);
}

// Fills the plan of a shape whose path (and, for the KV split, chunk count) is resolved. `workspace` is what the call may
// use: partials that do not fit lower the fill, then the shares. `any_path` (fmha_fwd_hd128_mxfp8_auto_ws): shares, and a
// workspace on the full-sequence paths too; the other entries run the path's own kernels.
void make_plan(Plan& pl, const fmha_mxfp8_params& p, bool scaled, size_t workspace, bool any_path) {
    const i64 B = p.B, H = p.H, HK = p.HK, S = p.S, SK = p.SK;
    fmha_pre_args fits_pre;   // the packed rows and the split last blocks exist on preloaded parameters only
    any_path = any_path && fill_pre(fits_pre, p, 0u, nullptr, nullptr);
    const size_t one = fmha_mxfp8_workspace_bytes(B, H, S, 1);
    const i64 fits = (i64)std::min<size_t>(workspace / one, 256);
    pl.parts = 1;
    pl.sub = pl.tail = pl.tail_blocks = 0;
    pl.kern = -1;
    if (pl.path == FMHA_PATH_KVSPLIT) {
        i64 fill = p.kv_fill ? 1 : kv_fill(B, H, S, SK, pl.splits);
        while (fill > 1 && fits < pl.splits * fill) fill /= 2;
        pl.parts = pl.splits * fill;
        pl.whole = false;
        // kv_fill = 1 asks for the reference's grid
        if (any_path && !p.kv_fill) pl.sub = packed_sub(B, H, HK, S, SK, pl.parts, false, true, p.f32_partials != 0, H * B * pl.parts, fits);
    } else {
        pl.kern = kernel_of(pl.path, B, H, S, SK, p.causal != 0, p.causal_pair == 1, scaled, &pl.block, &pl.gx);
        pl.whole = pl.kern != K_T128ST && pl.kern != K_T128ST_SC;
        // a forced path keeps its kernel (and its bits)
        if (any_path && p.path < 0 && p.kv_fill == 0)
            pl.sub = packed_sub(B, H, HK, S, SK, 1, pl.whole, false, true, (i64)pl.gx * H * B, fits);
        if (any_path && p.path < 0 && p.kv_fill == 0 && !p.causal && pl.sub == 0 && (pl.kern == K_VS128 || pl.kern == K_VS128_SC)) {
            const i64 blocks = (i64)pl.gx * H * B;
            pl.tail = tail_sub(blocks, (SK + 127) / 128);
            pl.tail_blocks = pl.tail ? blocks % cu_count() : 0;
            if (pl.tail && (tail_bytes(pl.tail_blocks, pl.tail) > workspace || pl.tail_blocks > 255 || blocks >= (1 << 20))) pl.tail = pl.tail_blocks = 0;
        }
    }
    if (pl.sub > 0 && (pl.parts > 255 || pl.parts * pl.sub * B * S * H * 512 >= (1LL << 32))) pl.sub = 0;   // the combines' 32-bit partial offsets
}

// path / splits as the entry resolves them from the params (no checks)
void resolve_path(Plan& pl, const fmha_mxfp8_params& p) {
    pl.splits = 0;
    pl.path = p.path;
    if (pl.path < 0) {
        pl.path = fmha_mxfp8_select_path(p.B, p.H, p.S, p.SK, &pl.splits);
        if (p.causal && pl.path == FMHA_PATH_KVSPLIT) pl.path = ((i64)(p.S + 255) / 256 * p.H * p.B <= 64) ? FMHA_PATH_T128 : FMHA_PATH_VS128;
    } else if (pl.path == FMHA_PATH_KVSPLIT) {
        pl.splits = p.splits > 0 ? p.splits : 4;
    }
}

}  // namespace

extern "C" {

int fmha_mxfp8_kv_partials(int64_t B, int64_t H, int64_t S, int64_t SK, int splits) {
    if (B < 1 || H < 1 || S < 1 || SK < 1 || splits < 1) return 0;
    return (int)(splits * kv_fill(B, H, S, SK, splits));
}

const char* fmha_mxfp8_version(void) { return "fmha_mxfp8 gfx950 1.0"; }

int fmha_mxfp8_init(char* err, size_t errlen) {
    hipFunction_t* fns = nullptr;
    return get_functions(&fns, err, errlen);
}

int fmha_mxfp8_validate_vs128(const fmha_mxfp8_args* a, const fmha_mxfp8_buffer_sizes* sz, uint32_t gx, uint32_t gy,
                              uint32_t gz, int64_t HK, char* err, size_t errlen) {
    // the causal q-tile pairing runs on the 128-row grid only
    if (a->flags & FMHA_FLAG_CAUSAL_PAIR) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x280) outside contract");
    return validate_base(*a, *sz, gx, gy, (i64)gz, HK, 256, err, errlen);
}

int fmha_mxfp8_validate_t128(const fmha_mxfp8_args* a, const fmha_mxfp8_buffer_sizes* sz, uint32_t gx, uint32_t gy,
                             uint32_t gz, int64_t HK, char* err, size_t errlen) {
    return validate_base(*a, *sz, gx, gy, (i64)gz, HK, 128, err, errlen);
}

int fmha_mxfp8_validate_kvsplit(const fmha_mxfp8_kvsplit_args* ka, const fmha_mxfp8_buffer_sizes* sz, uint32_t gx,
                                uint32_t gy, uint32_t gz, int64_t B, int64_t HK, int64_t KL, char* err, size_t errlen) {
    // kvsplit_abi.h: the base rules with the symbol B, the split extension inserted into each group
    fmha_mxfp8_args a;
    std::memcpy(&a, ka, 0x270);
    std::memset(reinterpret_cast<uint8_t*>(&a) + 0x270, 0, sizeof(a) - 0x270);
    // the split count is the low 16 bits; bit 16 is the f32-partials extension (FMHA_KVS_F32_PARTIALS)
    const i64 splits = ka->kvs_splits & 0xffffu, rows = ka->kvs_rows_total;
    const i64 row_bytes = 512;   // the workspace rows are fp32-sized in both formats
    int rc;
    if ((rc = rules_extent(a, *sz, B, (ka->kvs_splits & FMHA_KVS_V_SEQ32) != 0, err, errlen)) != FMHA_OK) return rc;
    if (sz->ptr_ohat < (uint64_t)(splits * rows * row_bytes)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_ohat: buffer ptr_ohat smaller than declared allocation");
    if (splits * rows * row_bytes >= (1LL << 32)) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x284) outside contract (partials of 4 GiB or more)");
    if (sz->ptr_lse < (uint64_t)(splits * rows * 4)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_lse: buffer ptr_lse smaller than declared allocation");
    if ((rc = rules_range(a, err, errlen)) != FMHA_OK) return rc;
    if (splits < 1 || (ka->kvs_splits & ~(0xffffu | FMHA_KVS_F32_PARTIALS | FMHA_KVS_V_SEQ32 | FMHA_KVS_SCALE)) != 0)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x280) outside contract");
    if ((rc = rules_scale(a, (ka->kvs_splits & FMHA_KVS_SCALE) != 0, err, errlen)) != FMHA_OK) return rc;
    if (rows < 1) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x284) outside contract");
    if ((rc = rules_is(a, HK, err, errlen)) != FMHA_OK) return rc;
    if (rows != B * (i64)a.s_seq_len * (i64)a.s_q_head_num) return fail(err, errlen, FMHA_ERR_KA_IS, "GV-HOST-KA-IS", "ka(0x284) relation failed");
    if ((rc = rules_grid(a, gx, gy, 256, err, errlen)) != FMHA_OK) return rc;
    if ((i64)gz != B * splits) return fail(err, errlen, FMHA_ERR_GRID, "GV-HOST-GRID", "grid axis 2 relation failed");
    if (KL < 0) return fail(err, errlen, FMHA_ERR_SYM, "GV-HOST-SYM", "symbol KL outside contract");
    return FMHA_OK;
}

int fmha_mxfp8_validate_combine(const fmha_mxfp8_combine_args* a, const fmha_mxfp8_buffer_sizes* sz, uint32_t gx,
                                uint32_t gy, uint32_t gz, char* err, size_t errlen) {
    // combine8h_abi.h:56-65
    (void)gx; (void)gy; (void)gz;
    const i64 rows = a->rows_total, splits = a->splits & 0xffffu;
    if (sz->ptr_ohat < (uint64_t)(splits * rows * 512)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_ohat: buffer ptr_ohat smaller than declared allocation");
    if (sz->ptr_lse < (uint64_t)(splits * rows * 4)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_lse: buffer ptr_lse smaller than declared allocation");
    if (splits * rows * 512 >= (1LL << 32)) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x18) outside contract (partials of 4 GiB or more)");
    if (sz->ptr_o < (uint64_t)(rows * 256)) return fail(err, errlen, FMHA_ERR_EXTENT, "GV-HOST-EXTENT", "ptr_out: buffer ptr_out smaller than declared allocation");
    if (rows < 1) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x18) outside contract");
    if (a->d != 128) return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x1C) outside contract");
    if (splits < 1 || (a->splits & ~(0xffffu | FMHA_KVS_F32_PARTIALS)) != 0)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x20) outside contract");
    return FMHA_OK;
}

int fmha_mxfp8_uses_split_tiles(int path, int64_t B, int64_t H, int64_t S, int64_t SK, int causal) {
    if (path == FMHA_PATH_T128) return use_split_tiles(B, H, S, SK, causal != 0) ? 1 : 0;
    if (path == FMHA_PATH_VS128)
        return vs128_on_128row_grid(B, H, S, SK, causal != 0) && use_split_tiles(B, H, S, SK, causal != 0) ? 1 : 0;
    return 0;
}

int fmha_mxfp8_select_path(int64_t B, int64_t H, int64_t S, int64_t SK, int* splits) {
    // dispatch.rs:494-511
    const i64 blocks256 = (S + 255) / 256 * H * B;
    const i64 ntiles = (SK + 127) / 128;
    i64 sp = 0;
    if (ntiles >= 16 && blocks256 <= 64) sp = 4;
    else if (ntiles >= 32 && blocks256 <= 128) sp = 2;
    if (sp > 0 && !empty_split(SK, sp)) {
        if (splits) *splits = (int)sp;
        return FMHA_PATH_KVSPLIT;
    }
    if (splits) *splits = 0;
    return blocks256 <= 64 ? FMHA_PATH_T128 : FMHA_PATH_VS128;
}

void fmha_mxfp8_fill_args(fmha_mxfp8_args* a, void* o, const void* q, const void* k, const void* v, const void* q_descale,
                          const void* k_descale, const void* v_descale, int B, int H, int HK, int S, int SK) {
    // the values tests/gpu/ref_host.cpp:342-360 writes
    (void)B;
    std::memset(a, 0, sizeof(*a));
    const uint32_t D = 128;
    a->ptr_o = o;
    a->ptr_q = const_cast<void*>(q);
    a->ptr_k = const_cast<void*>(k);
    a->ptr_v = const_cast<void*>(v);
    a->s_seq_len = (uint32_t)S;
    a->s_Seqs = (uint32_t)H * D;
    a->s_Hs = D;
    a->s_Bs = (uint32_t)((uint64_t)S * H * D);
    a->s_gqa = (uint32_t)(H / HK);
    a->s_k_Seqs = (uint32_t)HK * D;
    a->s_k_Hs = D;
    a->s_k_Bs = (uint32_t)((uint64_t)SK * HK * D);
    a->s_kv_seq_len = (uint32_t)SK;
    a->s_q_head_num = (uint32_t)H;
    a->s_v_Seqs = (uint32_t)HK * D;
    a->s_v_Hs = D;
    a->s_v_Bs = (uint32_t)((uint64_t)SK * HK * D);
    a->s_o_Seqs = (uint32_t)H * D * 2;
    a->s_o_Hs = D * 2;
    a->s_o_Bs = (uint32_t)((uint64_t)S * H * D * 2);
    a->ptr_q_descale = const_cast<void*>(q_descale);
    a->ptr_k_descale = const_cast<void*>(k_descale);
    a->ptr_v_descale = const_cast<void*>(v_descale);
    a->s_descale_q_Bs = (uint32_t)((uint64_t)S * H * 4);
    a->s_descale_q_Hs = 4;
    a->s_descale_k_Bs = (uint32_t)((uint64_t)SK * HK * 4);
    a->s_descale_k_Hs = 4;
    const float scale = 0.08838834764831845f;   // 1/sqrt(128), written as the reference host does (ignored)
    std::memcpy(&a->softmax_scale, &scale, 4);
}

size_t fmha_mxfp8_workspace_bytes(int64_t B, int64_t H, int64_t S, int splits) {
    if (splits <= 0) return 0;
    const uint64_t rows = (uint64_t)B * (uint64_t)S * (uint64_t)H;
    return (size_t)((uint64_t)splits * rows * (512u + 4u));
}

int fmha_mxfp8_launch_vs128(const fmha_mxfp8_args* a, uint32_t gx, uint32_t gy, uint32_t gz, void* stream) {
    return launch_raw((a->flags & FMHA_FLAG_SCALE) ? K_VS128_SC : K_VS128, a, sizeof(*a), gx, gy, gz, 512, stream, nullptr, 0);
}
int fmha_mxfp8_launch_t128(const fmha_mxfp8_args* a, uint32_t gx, uint32_t gy, uint32_t gz, void* stream) {
    // the reference-named kernel under its own contract: 256 threads (t128_abi.h)
    return launch_raw((a->flags & FMHA_FLAG_SCALE) ? K_T128_SC : K_T128, a, sizeof(*a), gx, gy, gz, 256, stream, nullptr, 0);
}
int fmha_mxfp8_launch_t128_split_tiles(const fmha_mxfp8_args* a, uint32_t gx, uint32_t gy, uint32_t gz, void* stream) {
    return launch_raw((a->flags & FMHA_FLAG_SCALE) ? K_T128ST_SC : K_T128ST, a, sizeof(*a), gx, gy, gz, 512, stream, nullptr, 0);
}
int fmha_mxfp8_launch_kvsplit(const fmha_mxfp8_kvsplit_args* a, uint32_t gx, uint32_t gy, uint32_t gz, void* stream) {
    return launch_raw((a->kvs_splits & FMHA_KVS_SCALE) ? K_KVSPLIT_SC : K_KVSPLIT, a, sizeof(*a), gx, gy, gz, 512, stream, nullptr, 0);
}
int fmha_mxfp8_launch_combine(const fmha_mxfp8_combine_args* a, uint32_t gx, void* stream) {
    return launch_raw(K_COMBINE, a, sizeof(*a), gx, 1, 1, 256, stream, nullptr, 0);
}
int fmha_mxfp8_launch_combine_wide(const fmha_mxfp8_combine_args* a, uint32_t gx, void* stream) {
    return launch_raw(K_COMBINE_WIDE, a, sizeof(*a), gx, 1, 1, 256, stream, nullptr, 0);
}

// The slot of the workspace that this call's partials go to, and the caller's turn word advanced.
// Workspace slots: a workspace of k >= 2 times the need (rounded to 256 B) holds min(k, FMHA_WORKSPACE_SLOTS) sets
// of partials, and consecutive calls take them in turn. The split kernel then writes lines that the previous
// call's combine did not just read: writing over partials that the combine read in the kernel before cost
// B1H8S2048 (4 splits) 25.6 -> 19.1 us per call with 4 slots (2 slots: 21.2, 8: 19.1, 16: 20.0).
static uint8_t* workspace_slot(const fmha_mxfp8_params& p, void* workspace, size_t workspace_bytes, size_t need) {
    const size_t stride = (need + 255u) & ~(size_t)255u;
    size_t nslots = workspace_bytes / stride;
    if (nslots < 1) nslots = 1;
    if (nslots > FMHA_WORKSPACE_SLOTS) nslots = FMHA_WORKSPACE_SLOTS;
    size_t slot = 0;
    if (nslots > 1 && p.ws_turn) slot = (size_t)((*p.ws_turn)++ % nslots);
    return (uint8_t*)workspace + slot * stride;
}

// The merge of `parts` partials per row into the output rows (and the LSE, when `lse` is not null).
static int run_combine(const fmha_mxfp8_params& p, const uint8_t* ohat, const uint8_t* lse, i64 parts, bool f32, float* lse_out, void* stream,
                       char* err, size_t errlen) {
    const i64 rows_total = (i64)p.B * p.S * p.H;
    struct LseArgs {
        fmha_mxfp8_combine_args c;
        uint32_t pad;
        float* lse_out;
        uint32_t S, H;
    } la;
    static_assert(sizeof(LseArgs) == 56 && offsetof(LseArgs, lse_out) == 40, "combine_lse kernarg");
    fmha_mxfp8_combine_args& ca = la.c;
    ca.ptr_ohat = const_cast<uint8_t*>(ohat);
    ca.ptr_lse = const_cast<uint8_t*>(lse);
    ca.ptr_out = p.o;
    ca.rows_total = (uint32_t)rows_total;
    ca.d = 128;
    ca.splits = (uint32_t)parts | (f32 ? FMHA_KVS_F32_PARTIALS : 0u);
    if (!p.no_check) {
        fmha_mxfp8_buffer_sizes csz;
        std::memset(&csz, 0, sizeof(csz));
        csz.ptr_ohat = (uint64_t)parts * rows_total * 512;
        csz.ptr_lse = (uint64_t)parts * rows_total * 4;
        csz.ptr_o = p.bytes_o;
        const int rc = fmha_mxfp8_validate_combine(&ca, &csz, 0, 1, 1, err, errlen);
        if (rc != FMHA_OK) return rc;
    }
    // more than 8 partials per row: the combine with the splits spread over 4 waves (64 groups per block)
    const bool wide = parts > 8 || lse_out;
    const uint64_t cgrid = ((uint64_t)rows_total * 128 / 8 + (wide ? 63 : 255)) / (wide ? 64 : 256);
    const uint32_t gx = (uint32_t)(cgrid ? cgrid : 1);
    if (lse_out) {
        la.pad = 0;
        la.lse_out = lse_out;
        la.S = (uint32_t)p.S;
        la.H = (uint32_t)p.H;
        return launch_raw(K_COMBINE_LSE, &la, sizeof(la), gx, 1, 1, 256, stream, err, errlen);
    }
    return launch_raw(wide ? K_COMBINE_WIDE : K_COMBINE, &ca, sizeof(ca), gx, 1, 1, 256, stream, err, errlen);
}

// The packed-rows kernel and its merge, for a plan with pl.sub > 0 (make_plan checked that the workspace holds the
// partials, and the caller the extents).
static int run_packed(const fmha_mxfp8_params& p, const Plan& pl, const fmha_mxfp8_args& a, void* workspace, size_t workspace_bytes, void* stream,
                      char* err, size_t errlen) {
    const i64 rows_total = (i64)p.B * p.S * p.H, parts = pl.parts * pl.sub;
    // the full-sequence paths hold O and the row sums in f32 to the end, so their partials stay in f32
    const bool f32 = pl.path != FMHA_PATH_KVSPLIT || p.f32_partials;
    uint8_t* ohat = workspace_slot(p, workspace, workspace_bytes, fmha_mxfp8_workspace_bytes(p.B, p.H, p.S, (int)parts));
    uint8_t* lse = ohat + (size_t)parts * rows_total * 512;
    fmha_pre_args ka;
    if (!fill_pre(ka, p, a.flags & (FMHA_FLAG_CAUSAL | FMHA_FLAG_V_SEQ32), ohat, lse)) return FMHA_ERR_KA_RANGE;   // (make_plan checked)
    ka.extra = (uint32_t)pl.parts | (uint32_t)pl.sub << 8 | (f32 ? kPreF32 : 0u) | (pl.whole ? kPreWhole : 0u) |
               ((p.B * parts) % 8 == 0 ? kPreByXcd : 0u);
    const i64 qtiles = ((i64)p.S * (p.H / p.HK) + 127) / 128;
    const int rc = launch_raw(p.v_seq32 ? ((a.flags & FMHA_FLAG_SCALE) ? K_PACKED_SC_VS : K_PACKED_VS)
                                       : ((a.flags & FMHA_FLAG_SCALE) ? K_PACKED_SC : K_PACKED), &ka, sizeof(ka), (uint32_t)(qtiles * p.HK * p.B * parts), 1, 1,
                              512, stream, err, errlen);
    if (rc != FMHA_OK) return rc;
    return run_combine(p, ohat, lse, parts, f32, pl.path == FMHA_PATH_KVSPLIT ? nullptr : (float*)p.lse, stream, err, errlen);
}

// The 256-row kernel with split last blocks and their merge, for a plan with pl.tail > 0 (make_plan checked the workspace).
static int run_tail(const fmha_mxfp8_params& p, const Plan& pl, const fmha_mxfp8_args& a, void* workspace, size_t workspace_bytes, void* stream,
                    char* err, size_t errlen) {
    const i64 blocks = (i64)pl.gx * p.H * p.B, nfull = blocks - pl.tail_blocks;
    uint8_t* ohat = workspace_slot(p, workspace, workspace_bytes, tail_bytes(pl.tail_blocks, pl.tail));
    uint8_t* lse = ohat + (size_t)(pl.tail_blocks * pl.tail * 256) * 512u;
    fmha_pre_args ta;
    if (!fill_pre(ta, p, a.flags & FMHA_FLAG_V_SEQ32, ohat, lse)) return FMHA_ERR_KA_RANGE;   // (make_plan checked)
    ta.extra = (uint32_t)nfull << 12 | (uint32_t)pl.tail_blocks << 4 | (uint32_t)pl.tail;
    ta.out = p.o;
    ta.lse_out = p.lse;
    const int rc = launch_raw(p.v_seq32 ? (pl.kern == K_VS128_SC ? K_TAIL_SC_VS : K_TAIL_VS) : (pl.kern == K_VS128_SC ? K_TAIL_SC : K_TAIL), &ta, sizeof(ta), (uint32_t)(nfull + pl.tail_blocks * pl.tail), 1, 1,
                              512, stream, err, errlen);
    if (rc != FMHA_OK) return rc;
    struct {
        const void *ohat, *lse;
        void *out, *lse_out;
        uint32_t ntail, sub, nfull, S, H, pad;
    } ca = {ohat, lse, p.o, p.lse, (uint32_t)pl.tail_blocks, (uint32_t)pl.tail, (uint32_t)nfull, (uint32_t)p.S, (uint32_t)p.H, 0u};
    return launch_raw(K_TAIL_COMBINE, &ca, sizeof(ca), (uint32_t)(pl.tail_blocks * 16), 1, 1, 256, stream, err, errlen);
}

// any_path: as in make_plan
static int run_entry(const fmha_mxfp8_params* p, void* workspace, size_t workspace_bytes, bool any_path, void* stream, int* path_out,
                     int* splits_out, char* err, size_t errlen) {
    if (!p) return fail(err, errlen, FMHA_ERR_PATH, "GV-HOST-ARGS", "null params");
    const i64 B = p->B, H = p->H, HK = p->HK, S = p->S, SK = p->SK;
    if (B < 1 || H < 1 || HK < 1 || S < 1 || SK < 1)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "B, H, HK, S, SK must be >= 1");
    if (H % HK != 0 || ((H / HK) & (H / HK - 1)) != 0 || H / HK > 16)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "H must be a power-of-two multiple (<= 16) of HK");
    Plan pl;
    resolve_path(pl, *p);
    const int path = pl.path, splits = pl.splits;
    if (path != FMHA_PATH_VS128 && path != FMHA_PATH_T128 && path != FMHA_PATH_KVSPLIT)
        return fail(err, errlen, FMHA_ERR_PATH, "GV-HOST-PATH", "unknown path");
    if (path == FMHA_PATH_KVSPLIT) {
        if (splits != 2 && splits != 4 && splits != 8) return fail(err, errlen, FMHA_ERR_PATH, "GV-HOST-PATH", "KV split count must be 2, 4 or 8");
        if (empty_split(SK, splits)) return fail(err, errlen, FMHA_ERR_PATH, "GV-HOST-PATH", "KV split leaves a split without a key tile");
        if (p->causal) return fail(err, errlen, FMHA_ERR_PATH, "GV-HOST-PATH", "the causal mask is not supported on the KV-split path");
    }
    if (p->f32_partials != 0 && p->f32_partials != 1)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "f32_partials must be 0 or 1");
    if (p->v_seq32 != 0 && p->v_seq32 != 1)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "v_seq32 must be 0 or 1");
    if (p->causal_pair < 0 || p->causal_pair > 2)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "causal_pair must be 0, 1 or 2");
    if (p->kv_fill != 0 && p->kv_fill != 1)
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "kv_fill must be 0 or 1");
    const bool scaled = p->softmax_scale != 0.0f;
    if (scaled && !scale_ok(p->softmax_scale))
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "softmax_scale must be 0 or positive with a normal f32 scale x log2(e)");
    fmha_mxfp8_args a;
    fmha_mxfp8_fill_args(&a, p->o, p->q, p->k, p->v, p->q_descale, p->k_descale, p->v_descale, (int)B, (int)H, (int)HK, (int)S, (int)SK);
    a.flags = (p->causal ? FMHA_FLAG_CAUSAL : 0u) | (p->v_seq32 ? FMHA_FLAG_V_SEQ32 : 0u) | (scaled ? FMHA_FLAG_SCALE : 0u);
    if (scaled) std::memcpy(&a.softmax_scale, &p->softmax_scale, 4);
    fmha_mxfp8_buffer_sizes sz;
    std::memset(&sz, 0, sizeof(sz));
    sz.ptr_q = p->bytes_q; sz.ptr_k = p->bytes_k; sz.ptr_v = p->bytes_v; sz.ptr_o = p->bytes_o;
    sz.ptr_q_descale = p->bytes_q_descale; sz.ptr_k_descale = p->bytes_k_descale; sz.ptr_v_descale = p->bytes_v_descale;
    // the KV split's partial count: the chunks times the fill, as far as the workspace holds it; the packed-rows shares
    make_plan(pl, *p, scaled, workspace ? workspace_bytes : 0, any_path);
    i64 parts = pl.parts;
    if (path == FMHA_PATH_KVSPLIT && parts * B * S * H * 512 >= (1LL << 32))
        // a kernel-contract limit (32-bit partial offsets), checked with or without no_check
        return fail(err, errlen, FMHA_ERR_KA_RANGE, "GV-HOST-KA-RANGE", "ka(0x284) outside contract (partials of 4 GiB or more)");
    if (path_out) *path_out = path;
    if (splits_out) *splits_out = path == FMHA_PATH_KVSPLIT ? splits : 0;
    if (p->partials_out) *p->partials_out = path == FMHA_PATH_KVSPLIT ? (int32_t)parts : 0;
    const uint32_t gy = (uint32_t)H;
    if (path == FMHA_PATH_VS128 || path == FMHA_PATH_T128) {
        a.ptr_lse = p->lse;
        const int rows = path == FMHA_PATH_VS128 ? 256 : 128;
        const uint32_t gx = (uint32_t)((S + rows - 1) / rows);
        if (!p->no_check) {
            const int rc = path == FMHA_PATH_VS128 ? fmha_mxfp8_validate_vs128(&a, &sz, gx, gy, (uint32_t)B, HK, err, errlen)
                                                   : fmha_mxfp8_validate_t128(&a, &sz, gx, gy, (uint32_t)B, HK, err, errlen);
            if (rc != FMHA_OK) return rc;
        }
        if (pl.sub > 0) return run_packed(*p, pl, a, workspace, workspace_bytes, stream, err, errlen);
        if (pl.tail > 0) return run_tail(*p, pl, a, workspace, workspace_bytes, stream, err, errlen);
        const int kern = pl.kern;
        const uint32_t block = pl.block;
        uint32_t kgx = pl.gx;
        // the causal q-tile pairing when the grid would take more than one wave of blocks (the extension's flag; the
        // reference pairs its causal kernels' tiles always, grid.rs:94-111), or when the caller asks for it
        const bool pair = p->causal && kern != K_VS128 && kern != K_VS128_SC && kgx > 1 &&
                          (p->causal_pair == 1 || (p->causal_pair == 0 && (i64)kgx * H * B > (i64)cu_count()));
        if (pair) {
            a.flags |= FMHA_FLAG_CAUSAL_PAIR;
            kgx = (kgx + 1) / 2;
        }
        const int pk = pre_kernel(kern, (SK + 127) / 128, a.flags);
        fmha_pre_args pre;
        if (pk >= 0 && fill_pre(pre, *p, a.flags, p->o, p->lse)) return launch_raw(pk, &pre, sizeof(pre), kgx, gy, (uint32_t)B, block, stream, err, errlen);
        return launch_raw(kern, &a, sizeof(a), kgx, gy, (uint32_t)B, block, stream, err, errlen);
    }
    // KV split: partials (fp32-sized rows, as ref_host.cpp:149 / ops.py:133) then the LSE, both in the workspace
    const i64 rows_total = B * S * H;
    const size_t need = fmha_mxfp8_workspace_bytes(B, H, S, (int)parts);
    if (!workspace || workspace_bytes < need) {
        set_err(err, errlen, "GV-HOST-WORKSPACE: KV split needs %zu workspace bytes, got %zu", need, workspace_bytes);
        return FMHA_ERR_WORKSPACE;
    }
    uint8_t* ohat = pl.sub > 0 ? (uint8_t*)workspace : workspace_slot(*p, workspace, workspace_bytes, need);
    uint8_t* lse = ohat + (size_t)parts * rows_total * 512;
    fmha_mxfp8_kvsplit_args ka;
    std::memcpy(&ka, &a, 0x270);
    ka.ptr_ohat = ohat;
    ka.ptr_lse = lse;
    const uint32_t part_fmt = p->f32_partials ? FMHA_KVS_F32_PARTIALS : 0u;
    ka.kvs_splits = (uint32_t)parts | part_fmt | (p->v_seq32 ? FMHA_KVS_V_SEQ32 : 0u) | (scaled ? FMHA_KVS_SCALE : 0u);
    ka.kvs_rows_total = (uint32_t)rows_total;
    sz.ptr_ohat = (uint64_t)parts * rows_total * 512;
    sz.ptr_lse = (uint64_t)parts * rows_total * 4;
    const uint32_t gx = (uint32_t)((S + 255) / 256), gz = (uint32_t)(B * parts);
    int rc = p->no_check ? FMHA_OK : fmha_mxfp8_validate_kvsplit(&ka, &sz, gx, gy, gz, B, HK, 0, err, errlen);
    if (rc != FMHA_OK) return rc;
    if (pl.sub > 0) return run_packed(*p, pl, a, workspace, workspace_bytes, stream, err, errlen);
    fmha_pre_args pre;
    if (!scaled && !p->v_seq32 && (SK + 127) / 128 >= 4 && fill_pre(pre, *p, 0u, ohat, lse)) {
        pre.extra = (uint32_t)parts | (p->f32_partials ? kPreF32 : 0u) | (gx == 1u && gz % 8u == 0u ? kPreByXcd : 0u);
        rc = launch_raw(K_PRE_KVSPLIT, &pre, sizeof(pre), gx, gy, gz, 512, stream, err, errlen);
    } else {
        rc = launch_raw(scaled ? K_KVSPLIT_SC : K_KVSPLIT, &ka, sizeof(ka), gx, gy, gz, 512, stream, err, errlen);
    }
    if (rc != FMHA_OK) return rc;
    return run_combine(*p, ohat, lse, parts, p->f32_partials != 0, nullptr, stream, err, errlen);
}

int fmha_fwd_hd128_mxfp8_auto(const fmha_mxfp8_params* p, void* workspace, size_t workspace_bytes, void* stream, int* path_out,
                              int* splits_out, char* err, size_t errlen) {
    return run_entry(p, workspace, workspace_bytes, false, stream, path_out, splits_out, err, errlen);
}

int fmha_fwd_hd128_mxfp8_auto_ws(const fmha_mxfp8_params* p, void* workspace, size_t workspace_bytes, void* stream, int* path_out,
                                 int* splits_out, char* err, size_t errlen) {
    return run_entry(p, workspace, workspace_bytes, true, stream, path_out, splits_out, err, errlen);
}

size_t fmha_mxfp8_auto_workspace_bytes(const fmha_mxfp8_params* p) {
    if (!p || p->B < 1 || p->H < 1 || p->HK < 1 || p->S < 1 || p->SK < 1 || p->H % p->HK != 0) return 0;
    Plan pl;
    resolve_path(pl, *p);
    if (pl.path != FMHA_PATH_VS128 && pl.path != FMHA_PATH_T128 && pl.path != FMHA_PATH_KVSPLIT) return 0;
    make_plan(pl, *p, p->softmax_scale != 0.0f, ~(size_t)0, true);
    if (pl.sub > 0) return fmha_mxfp8_workspace_bytes(p->B, p->H, p->S, (int)(pl.parts * pl.sub));
    if (pl.tail > 0) return tail_bytes(pl.tail_blocks, pl.tail);
    return pl.path == FMHA_PATH_KVSPLIT ? fmha_mxfp8_workspace_bytes(p->B, p->H, p->S, (int)pl.parts) : 0;
}

}  // extern "C"
