// w8a8_internal.hpp -- launchers shared between the kernel files and the C ABI.
// Callers (capi.cpp) have validated every argument before these run.
#pragma once

#include "../../include/w8a8.h"

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace w8a8 {

// Describes where quantizer row `i` reads from and writes to.
struct QuantRows {
    const uint16_t* x;        // fp16 source
    const float*    s;        // smooth scale (dense: [N]; moe: [experts, N])
    int8_t*         q;        // int8 destination
    float*          r;        // row scales
    uint32_t        rows;     // number of logical rows (dense: M, moe: tokens*topk)
    uint32_t        n;        // row length
    uint32_t        ldx, ldq; // strides in elements
    float           qmax;
    // MoE gather (all NULL / 0 for the dense quantizer)
    const int32_t* topk_ids;
    const int32_t* dst_row;
    uint32_t       rows_out; // destination rows (bound for dst_row entries)
    uint32_t       topk;
    uint32_t       experts;
};

hipError_t launch_smoothquant(const QuantRows& p, hipStream_t stream);
// How the MoE form runs: 16-byte chunks per lane, waves per row (0: two passes),
// and whether a group of waves takes a token with all its slots or one pair.
struct QuantPlan {
    uint32_t chunks, waves;
    bool     tokens;
};
QuantPlan moe_quant_plan(uint32_t pairs, uint32_t n, uint32_t topk);

// RMSNorm (+ residual add) fused with the quantizer (rmsnorm_sq.hip).  x,
// residual and x_out share the row stride ldx; residual, x_out, y, s, q and r
// may be NULL as w8a8_add_rmsnorm_smoothquant documents.
struct NormRows {
    const uint16_t* x;
    const uint16_t* res;
    const float*    gamma;
    const float*    s;
    uint16_t*       x_out;
    uint16_t*       y;
    int8_t*         q;
    float*          r;
    uint32_t        rows, n, ldx, ldy, ldq;
    float           eps, qmax;
};
hipError_t launch_rmsnorm_sq(const NormRows& p, hipStream_t stream);
// Rows of any alignment and length: 16-byte chunks per lane and waves per row (0: the
// generic kernel).
struct NormPlan {
    uint32_t chunks, waves;
};
NormPlan norm_rows_plan(uint32_t rows, uint32_t n);

struct GemmArgs {
    uint32_t       m, n, k;
    const int8_t*  a;
    const int8_t*  b;
    void*          c;
    uint32_t       lda, ldb, ldc;
    const float*   scale_a;
    const float*   scale_b;
    float          tsa, tsb;
    int            out_type; // W8A8_OUT_*
};

// A row-major [m,k], B [n,k] K-contiguous.  Fast path requirements (checked by
// the caller through gemm_fast_path_ok): 16-byte aligned a/b, lda/ldb % 16 == 0,
// k % 16 == 0.
// Small m (decode) is routed to the decode kernel inside launch_gemm_nk.
bool       gemm_fast_path_ok(const GemmArgs& g);
// ws (optional): int32 partials of a K split, where a plan whose partials fit
// ws_bytes is estimated to be faster; gemm_nk_workspace_bytes allows them all.
hipError_t launch_gemm_nk(const GemmArgs& g, void* ws, size_t ws_bytes, hipStream_t stream);
size_t     gemm_nk_workspace_bytes(const GemmArgs& g);
// sizes: m, n, k, workspace bytes -> plan: tile rows, tile columns, K pieces
// (0 x 32: the decode kernel).  Packed weights: m > 64.
void       gemm_plan(const uint32_t* sizes, bool packed, uint32_t* plan);
void       grouped_plan(const uint32_t* sizes, uint32_t* plan); // groups, their m, n, k
void       gemm_any_plan(const uint32_t* sizes, uint32_t* plan); // m, n, k, sample layout
// Explicit stream-K over every tile (w8a8_gemm_streamk): `blocks` blocks (0:
// one per CU, never more than the problem's k-tiles); ws: 16-byte aligned,
// streamk_workspace_bytes.  Needs gemm_fast_path_ok and A, B under 2 GiB
// (streamk_shape_ok).
bool       streamk_shape_ok(const GemmArgs& g);
size_t     streamk_workspace_bytes(uint32_t m, uint32_t n, uint32_t k, uint32_t blocks);
uint32_t   streamk_blocks(uint32_t m, uint32_t n, uint32_t k, uint32_t blocks);
hipError_t launch_gemm_streamk(const GemmArgs& g, uint32_t blocks, void* ws, hipStream_t stream);
// The current device's stream-K status word (gemm::kSkWaitExpired bits),
// read after a device-wide synchronisation, cleared when `clear`.
hipError_t streamk_status(uint32_t* flags, bool clear);
// Test hook of the stream-K wait: polls before giving up (0: the default)
// and phantom pieces the last piece also waits for (0: none).
void       streamk_debug_wait(uint32_t spin, uint32_t phantom);
// Device address of the current GPU's W8A8_NOALLOC_SCRATCH_BYTES scratch
// array (resolved once per device; gemm_i8.hip).
hipError_t noalloc_scratch(void** ptr);

// Decode kernel (m <= kDecodeMaxM): weights streamed once, split-K across the
// waves of a block.  `packed`: g.b holds packed weights (g.ldb unused).
constexpr uint32_t kDecodeMaxM = 64;
bool       gemm_decode_ok(const GemmArgs& g);
// The decode kernel with the activation quantization folded in (packed
// weights, fp16 output, m = 1 when decode_fuse_ok): x fp16 [m, ldx] (16-byte
// aligned rows), s [k] (16-byte aligned); q [m, k] and r [m] are written as
// by the quantizer, and g.a = q, g.scale_a = r.
struct FuseArgs {
    const uint16_t* x;
    const float*    s;
    int8_t*         q;
    float*          r;
    uint32_t        ldx;
    float           qmax;
};
bool       decode_fuse_ok(uint32_t m, uint32_t k);
hipError_t launch_gemm_decode_fused(const GemmArgs& g, const FuseArgs& f, hipStream_t stream);
hipError_t launch_gemm_decode(const GemmArgs& g, bool packed, void* ws, size_t ws_bytes,
                              hipStream_t stream);

// Packed weights: [n, k] int8 rearranged into MFMA register order, 64-row
// slabs x 128-deep k-tiles of 8 KiB, zero padded (n to 64, k to 128).
size_t     packed_weight_bytes(uint32_t n, uint32_t k);
hipError_t launch_pack_weights(const int8_t* w, uint32_t n, uint32_t k, uint32_t ldw,
                               int8_t* packed, hipStream_t stream);
// Fold + per-channel quantization of fp16 weights (weights.hip); packed:
// write the packed layout (zero padding included), else row-major [n, ldq].
struct WeightQuant {
    const uint16_t* w;
    const float*    s;
    int8_t*         q;
    float*          sb;
    uint32_t        n, k, ldw, ldq;
    float           qmax;
};
hipError_t launch_quantize_weights(const WeightQuant& p, bool divide, bool packed,
                                   hipStream_t stream);

// GEMM over packed weights (g.ldb unused).  gemm_packed_ok: 16-byte aligned
// A, lda % 16 == 0, k % 16 == 0 and every A panel addressable (< 2 GiB).
bool       gemm_packed_ok(const GemmArgs& g);
hipError_t launch_gemm_packed(const GemmArgs& g, void* ws, size_t ws_bytes, hipStream_t stream);
// Split-K workspace the packed path can use for this problem (m > 32); 0 when
// none is used.  A smaller (or no) workspace falls back to the unsplit decode
// kernel (m <= 64) or to a plan whose partials fit.
size_t     packed_workspace_bytes(const GemmArgs& g);

// Tile GEMM over any pointers, strides and K (gemm_i8_direct_kernel.hpp): the
// primary layout, or the sample layout in place (kn; gemm_direct_kn_ok: at
// least 4 rows and columns).  direct_kn_pays: sizes where that beats the repack.
hipError_t launch_gemm_direct(const GemmArgs& g, bool kn, hipStream_t stream);
bool       gemm_direct_kn_ok(const GemmArgs& g);
bool       direct_kn_pays(const GemmArgs& g);

// Generic strided GEMM: A(m,k) = a[m*sam + k*sak], B(n,k) = b[n*sbn + k*sbk].
// One output per thread: where generic_pays (few products of short K; kn: the
// sample layout), and the sample layout with m < 4 or n < 4 and no workspace.
bool       generic_pays(const GemmArgs& g, bool kn);
hipError_t launch_gemm_generic(const GemmArgs& g, size_t sam, size_t sak, size_t sbn,
                               size_t sbk, hipStream_t stream);

// Repack of the sample layout's operands (A [k, lda], B [k, ldb]) into K-contiguous
// rows of kp bytes (a multiple of 16, zero past k), one launch.
hipError_t launch_repack_kn(const GemmArgs& g, int8_t* at, int8_t* bt, uint32_t kp,
                            hipStream_t stream);

// ---- MoE (moe.hip) ----------------------------------------------------------
hipError_t launch_topk_softmax(const void* logits, bool f16, float* w, int32_t* ids,
                               uint32_t tokens, uint32_t experts, uint32_t topk,
                               hipStream_t stream);

size_t     moe_sort_lds_bytes(uint32_t experts);
// ws (optional, moe_sort_workspace_bytes): the multi-block sort for inputs of
// more than one block of pairs; NULL or smaller: one workgroup.
size_t     moe_sort_workspace_bytes(uint32_t tokens, uint32_t topk, uint32_t experts);
hipError_t launch_moe_sort(const int32_t* ids, uint32_t tokens, uint32_t topk, uint32_t experts,
                           uint32_t unit, int32_t* count, int32_t* start, int32_t* padded,
                           int32_t* sorted_ids, uint32_t sorted_cap, int32_t* dst_row, void* ws,
                           size_t ws_bytes, hipStream_t stream);

hipError_t launch_silu_mul_quant(const uint16_t* gu, uint32_t ld_gu, const float* s2,
                                 const int32_t* expert_start, const int32_t* expert_count,
                                 uint32_t experts, uint32_t rows, uint32_t inter, int8_t* q,
                                 uint32_t ldq, float* r, float qmax, hipStream_t stream);

hipError_t launch_moe_combine(const uint16_t* y, uint32_t ldy, uint32_t rows_y, const float* w,
                              const int32_t* dst_row, uint32_t tokens, uint32_t topk, uint32_t n,
                              uint16_t* out, uint32_t ldo, hipStream_t stream);

// Grouped GEMM (moe.hip).  grouped_gemm_tile: one tile for all groups, of the
// least estimated time (gemm_i8.hip), and the total tile count with it; tiles =
// 0 for empty groups only.  groups: the validated host descriptors; groups_dev:
// their copy, read only for more than kGroupedInline groups.
constexpr uint32_t kGroupedInline = W8A8_GROUPED_INLINE_GROUPS;
struct GroupedTile {
    uint32_t bm, bn, tiles;
};
GroupedTile grouped_gemm_tile(const w8a8_group_desc* groups, uint32_t ngroups);
hipError_t  launch_grouped_gemm(const w8a8_group_desc* groups, const void* groups_dev,
                                uint32_t ngroups, const GroupedTile& tile, int out_type,
                                hipStream_t stream);

struct MoeGemmArgs {
    const int8_t*  a;
    const int8_t*  w;
    void*          c;
    const float*   scale_a;
    const float*   scale_w;
    const int32_t* expert_start;
    const int32_t* expert_count;
    uint32_t       rows, experts, n, k, lda, ldw, ldc;
    uint64_t       w_stride;
    float          tsa, tsb;
    int            out_type;
    void*          ws;       // tail-split partials, or null (no split)
    size_t         ws_bytes;
};
hipError_t launch_moe_gemm(const MoeGemmArgs& a, hipStream_t stream);
// sizes: experts, rows, n, k -> plan: tile rows, tile columns, whether a tail that
// fills few CUs is cut along K (given the workspace).
void       moe_gemm_plan(const uint32_t* sizes, uint32_t* plan);
// sizes: rows, inter, block -> plan: rows a block, the block's first row
void       moe_requant_plan(const uint32_t* sizes, uint32_t* plan);
// Workspace that lets launch_moe_gemm split its last partial round of tiles
// along K (one int32 tile partial per CU of the current device).
size_t moe_gemm_workspace_bytes();

// The gate_up expert GEMM with the SiLU(gate) * up epilogue, then the
// requantization of the fp16 activation (w8a8_moe_gate_up_silu).  w: the
// interleaved gate_up weights [experts, 2 * inter, k]; ws: 256-byte aligned,
// moe_gate_up_silu_workspace_bytes (activation, row maxima, split partials).
struct MoeSiluArgs {
    const int8_t*  a;
    const int8_t*  w;
    const float*   scale_a;
    const float*   scale_w; // [experts, 2 * inter], interleaved like w
    const float*   s2;      // [experts, inter] or null
    const int32_t* expert_start;
    const int32_t* expert_count;
    uint32_t       rows, experts, inter, k, lda;
    float          tsa, tsb;
    int8_t*        q;
    uint32_t       ldq;
    float*         r;
    float          qmax;
    void*          ws;
};
size_t     moe_gate_up_silu_workspace_bytes(uint32_t rows, uint32_t inter);
hipError_t launch_moe_gate_up_silu(const MoeSiluArgs& a, hipStream_t stream);
hipError_t launch_moe_interleave_gate_up(const int8_t* w, const float* sw, uint32_t experts,
                                         uint32_t inter, uint32_t k, uint32_t ldw, int8_t* wo,
                                         float* swo, hipStream_t stream);

} // namespace w8a8
