// smoothquant.hip -- row-wise smooth-scale + absmax int8 quantizer for gfx950.
//
// Computation (kernel_smoothquant, rocwmma_smoothquant.cpp:58-122, and
// kernel_moe_smoothquant, rocwmma_moe_smoothquant.cpp:69-131):
//   p = float(x[row, n]) * s[n];  r = max|p| / qmax;  inv = r > 0 ? 1/r : 0
//   q[row, n] = int8(clamp(rint(p * inv), -qmax, qmax))
//
// The kernels, all with the same per-element operations (bit-identical results):
//   * sq_stream_kernel (dense rows, 16-byte aligned, N % 8 == 0, N <= 32768):
//     s staged once per block in LDS, one block per CU walking the rows with
//     a grid stride and double-buffering them in registers (described at the
//     kernel);
//   * sq_rows_kernel: a dense row, or one (token, slot) pair of the MoE form, of
//     any alignment and length to 32768;
//   * sq_tokens_kernel: the MoE form where reading a token once for all of its
//     experts pays (moe_quant_plan says where);
//   * sq_twopass_kernel: longer rows.
//
// sq_rows_kernel (HBM-bound: 3 bytes moved per element):
//   * One wavefront owns a row segment of CPL*512 elements; WPR wavefronts
//     share a row.  Each lane issues CPL 16-byte loads (8 fp16) at whatever
//     address the row has (the hardware takes unaligned global accesses), so a
//     wave instruction reads 1 KiB contiguous and the whole segment is in
//     flight at once; only the chunk that straddles N goes element by element.
//     15000 x 1337, odd rows: 71 -> 15 us.
//   * The products stay in VGPRs: x is read from HBM exactly once (the
//     reference re-reads it in its second pass, :101-117).
//   * absmax: DPP quad/mirror steps inside each 16-lane row + 4 readlanes;
//     rows spread over several waves merge through 16 bytes of LDS.
//   * Output: each lane packs 8 int8 and stores 8 bytes (a wave writes 512
//     contiguous bytes), straight into the row-major A operand of the GEMM.
#include "w8a8_device.hpp"
#include "w8a8_internal.hpp"

#include <algorithm>
#include <mutex>

namespace w8a8 {
namespace {

constexpr int kSqThreads = 256; // 4 waves
// Cache-policy operand of the buffer builtins: the NT (non-temporal) bit.
constexpr int kCpolNt = 2;
constexpr int kSqWaves   = kSqThreads / kWave;

struct RowSrc {
    const uint16_t* x;
    const float*    s;
    long            dst;
    bool            valid;
};

template <bool MOE>
__device__ __forceinline__ RowSrc resolve_row(const QuantRows& p, uint32_t row)
{
    RowSrc rs{nullptr, nullptr, -1, false};
    if(row >= p.rows) return rs;
    if constexpr(MOE) {
        uint32_t tok = row / p.topk;
        int32_t  e   = p.topk_ids[row];
        if(e < 0 || (uint32_t)e >= p.experts) return rs;
        long dst = p.dst_row ? (long)p.dst_row[row] : (long)row;
        if(dst < 0 || dst >= (long)p.rows_out) return rs;
        rs.x   = p.x + (size_t)tok * p.ldx;
        rs.s   = p.s + (size_t)e * p.n;
        rs.dst = dst;
    } else {
        rs.x   = p.x + (size_t)row * p.ldx;
        rs.s   = p.s;
        rs.dst = row;
    }
    rs.valid = true;
    return rs;
}

constexpr int sq_rows_threads(int wpr) { return wpr * kWave > kSqThreads ? wpr * kWave : kSqThreads; }
// Waves per SIMD that a lane's products leave room for; without it the compiler
// takes 82 VGPRs for CPL = 8 and a wave fewer fits.
constexpr int sq_rows_waves(int cpl) { return cpl == 4 ? 8 : cpl == 8 ? 6 : 1; }

// CPL: 16-byte chunks per lane; WPR: waves per row.  A chunk's x and s are
// loaded and multiplied together, and both tails are computed in their own
// branch: x ahead of s, or the packing ahead of the branch, costs 12-34 VGPRs and
// with them two waves a SIMD (8192 pairs of 4096, top 1: 22.4 us, 18.7 as it is).
template <int CPL, int WPR, bool MOE>
__global__ void __launch_bounds__(sq_rows_threads(WPR), sq_rows_waves(CPL))
    sq_rows_kernel(QuantRows p)
{
    constexpr int kWaves        = sq_rows_threads(WPR) / kWave;
    constexpr int kRowsPerBlock = kWaves / WPR;
    constexpr int kSpan         = CPL * 8 * kWave;

    const int      wave = threadIdx.x / kWave;
    const int      lane = threadIdx.x % kWave;
    const int      rib  = wave / WPR; // row in block
    const int      part = wave % WPR; // segment of the row
    const RowSrc   src  = resolve_row<MOE>(p, blockIdx.x * kRowsPerBlock + rib);
    const uint32_t n    = p.n;
    const uint32_t base = part * kSpan + lane * 8;

    float pv[CPL * 8];
    float amax = 0.f;
    if(src.valid) {
#pragma unroll
        for(int j = 0; j < CPL; ++j) {
            const uint32_t c = base + j * (8 * kWave);
            if(c + 8 <= n) {
                uint32_t w[4];
                float    sv[8];
                __builtin_memcpy(w, src.x + c, 16);
                __builtin_memcpy(sv, src.s + c, 16);
                __builtin_memcpy(sv + 4, src.s + c + 4, 16);
#pragma unroll
                for(int e = 0; e < 4; ++e) {
                    pv[j * 8 + 2 * e]     = mul_h16_f32<false>(w[e], sv[2 * e]);
                    pv[j * 8 + 2 * e + 1] = mul_h16_f32<true>(w[e], sv[2 * e + 1]);
                }
            } else {
#pragma unroll
                for(int e = 0; e < 8; ++e)
                    pv[j * 8 + e] = e < 7 && c + e < n
                                        ? half_bits_to_float(src.x[c + e]) * src.s[c + e]
                                        : 0.f;
            }
#pragma unroll
            for(int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(pv[j * 8 + e]));
        }
    }

    amax = wave_max(amax);
    if constexpr(WPR > 1) {
        __shared__ float red[kWaves];
        if(lane == 0) red[wave] = amax;
        __syncthreads();
#pragma unroll
        for(int w = 0; w < WPR; ++w) amax = fmaxf(amax, red[rib * WPR + w]);
    }
    if(!src.valid) return;

    const float qmax = p.qmax;
    const float rs   = amax / qmax; // correctly rounded fp32 division
    if(part == 0 && lane == 0) p.r[src.dst] = rs;
    const float inv = (rs > 0.f) ? (1.f / rs) : 0.f;

    int8_t* qrow = p.q + (size_t)src.dst * p.ldq;
#pragma unroll
    for(int j = 0; j < CPL; ++j) {
        const uint32_t c = base + j * (8 * kWave);
        const float*   v = pv + j * 8;
        auto           pack = [&](uint32_t(&o)[2]) {
            o[0] = cvt_pack4_i8(quant_f(v[0], inv, qmax), quant_f(v[1], inv, qmax),
                                quant_f(v[2], inv, qmax), quant_f(v[3], inv, qmax));
            o[1] = cvt_pack4_i8(quant_f(v[4], inv, qmax), quant_f(v[5], inv, qmax),
                                quant_f(v[6], inv, qmax), quant_f(v[7], inv, qmax));
        };
        uint32_t packed[2];
        if constexpr(CPL == 1) pack(packed); // short rows are mostly their tail
        if(c + 8 <= n) {
            if constexpr(CPL > 1) pack(packed);
            __builtin_memcpy(qrow + c, packed, 8);
        } else {
#pragma unroll
            for(int e = 0; e < 7; ++e)
                if(c + e < n)
                    qrow[c + e] = CPL == 1 ? (int8_t)(packed[e / 4] >> (8 * (e % 4)))
                                           : (int8_t)quant_i8(v[e], inv, qmax);
        }
    }
}

// The MoE form with x read once for all of a token's experts: a group of WPR
// waves holds the token's x in VGPRs and writes its topk rows one after another,
// reading only each expert's smooth scale (2916 x 7168, top 6 92 -> 58 us).
template <int CPL, int WPR>
__global__ void __launch_bounds__(sq_rows_threads(WPR)) sq_tokens_kernel(QuantRows p)
{
    constexpr int kWaves          = sq_rows_threads(WPR) / kWave;
    constexpr int kTokensPerBlock = kWaves / WPR;
    constexpr int kSpan           = CPL * 8 * kWave;
    __shared__ float red[2][kWaves];

    const int      wave = threadIdx.x / kWave;
    const int      lane = threadIdx.x % kWave;
    const int      tib  = wave / WPR; // token in block
    const int      part = wave % WPR; // segment of the row
    const uint32_t tok  = blockIdx.x * kTokensPerBlock + tib;
    const uint32_t row0 = tok * p.topk;
    const uint32_t n    = p.n;
    const uint32_t base = part * kSpan + lane * 8;

    v4i raw[CPL]; // zeros past N and for tokens past the last
    if(row0 < p.rows) {
        const uint16_t* x = p.x + (size_t)tok * p.ldx;
#pragma unroll
        for(int j = 0; j < CPL; ++j) {
            const uint32_t c = base + j * (8 * kWave);
            raw[j]           = v4i{0};
            if(c + 8 <= n) {
                __builtin_memcpy(&raw[j], x + c, 16);
            } else if(c < n) {
                uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
                for(int e = 0; e < 7; ++e)
                    if(c + e < n) w[e / 2] |= (uint32_t)x[c + e] << (16 * (e % 2));
                raw[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
            }
        }
    }
    const float qmax = p.qmax;
    for(uint32_t slot = 0; slot < p.topk; ++slot) { // the same count in every wave
        const RowSrc src = resolve_row<true>(p, row0 + slot);
        float        pv[CPL * 8];
        float        amax = 0.f;
        if(src.valid) {
#pragma unroll
            for(int j = 0; j < CPL; ++j) {
                const uint32_t c     = base + j * (8 * kWave);
                float          sv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                if(c + 8 <= n) {
                    __builtin_memcpy(sv, src.s + c, 16);
                    __builtin_memcpy(sv + 4, src.s + c + 4, 16);
                } else if(c < n) {
#pragma unroll
                    for(int e = 0; e < 7; ++e)
                        if(c + e < n) sv[e] = src.s[c + e];
                }
                const uint32_t w[4] = {(uint32_t)raw[j].x, (uint32_t)raw[j].y, (uint32_t)raw[j].z,
                                       (uint32_t)raw[j].w};
#pragma unroll
                for(int e = 0; e < 4; ++e) {
                    pv[j * 8 + 2 * e]     = mul_h16_f32<false>(w[e], sv[2 * e]);
                    pv[j * 8 + 2 * e + 1] = mul_h16_f32<true>(w[e], sv[2 * e + 1]);
                }
#pragma unroll
                for(int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(pv[j * 8 + e]));
            }
        }
        amax = wave_max(amax);
        if constexpr(WPR > 1) {
            float* r = red[slot % 2]; // the other half may still be read from the slot before
            if(lane == 0) r[wave] = amax;
            __syncthreads();
#pragma unroll
            for(int w = 0; w < WPR; ++w) amax = fmaxf(amax, r[tib * WPR + w]);
        }
        if(!src.valid) continue;
        const float rs = amax / qmax; // correctly rounded fp32 division
        if(part == 0 && lane == 0) p.r[src.dst] = rs;
        const float inv = (rs > 0.f) ? (1.f / rs) : 0.f;

        int8_t* qrow = p.q + (size_t)src.dst * p.ldq;
#pragma unroll
        for(int j = 0; j < CPL; ++j) {
            const uint32_t c = base + j * (8 * kWave);
            const float*   v = pv + j * 8;
            uint32_t       packed[2];
            packed[0] = cvt_pack4_i8(quant_f(v[0], inv, qmax), quant_f(v[1], inv, qmax),
                                     quant_f(v[2], inv, qmax), quant_f(v[3], inv, qmax));
            packed[1] = cvt_pack4_i8(quant_f(v[4], inv, qmax), quant_f(v[5], inv, qmax),
                                     quant_f(v[6], inv, qmax), quant_f(v[7], inv, qmax));
            if(c + 8 <= n) {
                __builtin_memcpy(qrow + c, packed, 8);
            } else {
#pragma unroll
                for(int e = 0; e < 7; ++e)
                    if(c + e < n) qrow[c + e] = (int8_t)(packed[e / 4] >> (8 * (e % 4)));
            }
        }
    }
}

// Rows longer than the register-resident path covers: one block per row,
// two passes over x (the second pass re-reads x, mostly from L2).
template <bool MOE>
__global__ void __launch_bounds__(kSqThreads) sq_twopass_kernel(QuantRows p)
{
    __shared__ float red[kSqWaves];
    RowSrc src = resolve_row<MOE>(p, blockIdx.x);
    if(!src.valid) return; // uniform over the block
    float amax = 0.f;
    for(uint32_t c = threadIdx.x; c < p.n; c += kSqThreads)
        amax = fmaxf(amax, fabsf(half_bits_to_float(src.x[c]) * src.s[c]));
    amax = wave_max(amax);
    if(threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float rs = amax / p.qmax;
    if(threadIdx.x == 0) p.r[src.dst] = rs;
    const float inv  = (rs > 0.f) ? (1.f / rs) : 0.f;
    int8_t*     qrow = p.q + (size_t)src.dst * p.ldq;
    for(uint32_t c = threadIdx.x; c < p.n; c += kSqThreads)
        qrow[c] = (int8_t)quant_i8(half_bits_to_float(src.x[c]) * src.s[c], inv, p.qmax);
}

// ---------------------------------------------------------------------------
// Streaming quantizer for the dense case (aligned rows, N % 8 == 0, N <= 32768).
//   * s is staged once per block in LDS, permuted so that each ds_read_b128 of
//     a wave reads 1 KiB contiguous (conflict-free); rows then never re-read
//     s from L2, and no register holds it.
//   * A group of WPR waves owns one row at a time (CPL 16-byte chunks per
//     lane), the block's groups walk the rows with a grid stride, and each
//     wave loads its next row into a second register buffer while it reduces
//     and quantizes the current one: HBM reads stay in flight across rows.
//   * The smoothed values are recomputed from x and the LDS copy of s in the
//     quantize pass instead of being kept in registers, so a wave holds only
//     2 x CPL x 4 VGPRs of row data.
// Results are bit-identical to sq_rows_kernel: same per-element operations.
// ---------------------------------------------------------------------------

// Bytes of x or q one streaming launch addresses at most (below the kernel's
// out-of-range row offset, 0x7FFFFFF0).
constexpr uint64_t kPanelBytes = 0x7F000000ull;

// NT: x is read with the non-temporal cache policy (it is read once); NTS:
// q is stored with it too.
template <int CPL, int WPR, int THREADS, bool NT = false, bool NTS = false>
__global__ void __launch_bounds__(THREADS) sq_stream_kernel(QuantRows p, uint32_t iters)
{
    constexpr int kStreamThreads = THREADS;
    constexpr int kStreamWaves   = THREADS / kWave;
    extern __shared__ __attribute__((aligned(16))) float s_lds[]; // kSpan * WPR floats
    __shared__ float red[2][kStreamWaves];
    constexpr int      kGroups = kStreamWaves / WPR;
    static_assert(kStreamWaves % WPR == 0, "whole row groups per block");
    constexpr int      kSpan   = CPL * 8 * kWave; // columns one wave covers
    constexpr uint32_t kOobOff = 0x80000000u;     // past every buffer: loads 0, stores dropped
    const int      wave = threadIdx.x / kWave;
    const int      lane = threadIdx.x % kWave;
    const int      grp  = wave / WPR;
    const int      part = wave % WPR;
    const uint32_t n    = p.n;
    const uint32_t base = part * kSpan + lane * 8;

    // Operands through buffer resources: rows past the end and columns past N
    // use an offset beyond the buffer (loads read 0, stores are dropped), so
    // the hot loop has no branches and every wave always has exactly CPL loads
    // per row in flight; the wait before a row is processed then leaves the
    // next row's loads outstanding.
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.x), 0, (int)((p.rows - 1) * p.ldx * 2 + n * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        p.q, 0, (int)((p.rows - 1) * p.ldq + n), 0x00020000);

    // Offsets of a chunk = the row's base + the chunk's column offset.  A
    // column past N has offset kOobOff and a row past the end the base
    // kOobRow: every sum of an in-range row and column stays below the
    // buffer's size (< 2^31), and every other sum lies in [2^31, 2^32) (no
    // wrap), past the buffer: one add per chunk, no select.
    // (The host keeps both buffers under kPanelBytes < kOobRow.)
    constexpr uint32_t kOobRow = 0x7FFFFFF0u;
    uint32_t coff[CPL]; // q byte offset of each chunk in a row (its column), or kOobOff
    uint32_t xoff[CPL]; // x byte offset of each chunk in a row, or kOobOff
#pragma unroll
    for(int j = 0; j < CPL; ++j) {
        const uint32_t c = base + j * (8 * kWave);
        coff[j]          = c < n ? c : kOobOff;
        xoff[j]          = c < n ? 2 * c : kOobOff;
    }

    using Row = v4i[CPL];
    Row  xa, xb;
    auto load_row = [&](Row& dst, uint32_t r) {
        const uint32_t roff = r < p.rows ? r * p.ldx * 2 : kOobRow;
#pragma unroll
        for(int j = 0; j < CPL; ++j)
            dst[j] = __builtin_amdgcn_raw_buffer_load_b128(rx, roff + xoff[j], 0,
                                                           NT ? kCpolNt : 0);
    };
    // LDS offset of this lane's s values; made opaque once per row (below) so
    // the compiler re-reads s from LDS instead of pinning CPL*8 registers to it
    // for the whole kernel, which would cap the CU at one block
    uint32_t s_off = (part * kSpan + lane * 4) * 4;
    // the 8 products x*s of chunk j (mul_h16_f32: one instruction each)
    auto smoothed = [&](const v4i& raw, int j, float* v) {
        const float4 s0 = *reinterpret_cast<const float4*>(
            reinterpret_cast<const char*>(s_lds) + s_off + j * 2048);
        const float4 s1 = *reinterpret_cast<const float4*>(
            reinterpret_cast<const char*>(s_lds) + s_off + j * 2048 + 1024);
        v[0] = mul_h16_f32<false>((uint32_t)raw.x, s0.x);
        v[1] = mul_h16_f32<true>((uint32_t)raw.x, s0.y);
        v[2] = mul_h16_f32<false>((uint32_t)raw.y, s0.z);
        v[3] = mul_h16_f32<true>((uint32_t)raw.y, s0.w);
        v[4] = mul_h16_f32<false>((uint32_t)raw.z, s1.x);
        v[5] = mul_h16_f32<true>((uint32_t)raw.z, s1.y);
        v[6] = mul_h16_f32<false>((uint32_t)raw.w, s1.z);
        v[7] = mul_h16_f32<true>((uint32_t)raw.w, s1.w);
    };
    auto process = [&](const Row& x, uint32_t r, int parity) {
        asm volatile("" : "+v"(s_off));
        // columns past N hold x = 0 and s = 0: they add nothing to the max.
        // The products stay in registers for the quantize pass.
        float pv[CPL * 8];
        float amax = 0.f;
#pragma unroll
        for(int j = 0; j < CPL; ++j) {
            smoothed(x[j], j, pv + j * 8);
#pragma unroll
            for(int e = 0; e < 8; e += 2)
                amax = fmaxf(fmaxf(amax, fabsf(pv[j * 8 + e])), fabsf(pv[j * 8 + e + 1]));
        }
        amax = wave_max(amax);
        if constexpr(WPR > 1) {
            if(lane == 0) red[parity][wave] = amax;
            __syncthreads();
#pragma unroll
            for(int w = 0; w < WPR; ++w) amax = fmaxf(amax, red[parity][grp * WPR + w]);
        }
        const bool  valid = r < p.rows;
        const float qmax  = p.qmax;
        const float rs    = amax / qmax;
        if(valid && part == 0 && lane == 0) p.r[r] = rs;
        const float    inv  = rs > 0.f ? 1.f / rs : 0.f;
        const uint32_t qoff = valid ? r * p.ldq : kOobRow;
#pragma unroll
        for(int j = 0; j < CPL; ++j) {
            const float* v = pv + j * 8;
            v2i          pk;
            pk.x = (int)cvt_pack4_i8(quant_f(v[0], inv, qmax), quant_f(v[1], inv, qmax),
                                     quant_f(v[2], inv, qmax), quant_f(v[3], inv, qmax));
            pk.y = (int)cvt_pack4_i8(quant_f(v[4], inv, qmax), quant_f(v[5], inv, qmax),
                                     quant_f(v[6], inv, qmax), quant_f(v[7], inv, qmax));
            __builtin_amdgcn_raw_buffer_store_b64(pk, rq, qoff + coff[j], 0, NTS ? kCpolNt : 0);
        }
    };

    const uint32_t stride = gridDim.x * kGroups;
    uint32_t       row    = blockIdx.x * kGroups + grp;

    // The first row's loads go out before s is staged, so the two fetches
    // overlap.  s lands in LDS permuted so that each ds_read_b128 of a wave
    // reads 1 KiB contiguous (conflict-free): column c = part*kSpan + j*512 +
    // l*8 + e of a row sits at part*kSpan + j*512 + (e/4)*256 + l*4 + e%4.
    // Columns past N are stored as 0.
    load_row(xa, row);
    {
        constexpr int kTotal = kSpan * WPR;
        constexpr int kS4    = (kTotal + kStreamThreads * 4 - 1) / (kStreamThreads * 4);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(p.s), 0, (int)(n * 4), 0x00020000);
        v4i sv[kS4];
#pragma unroll
        for(int i = 0; i < kS4; ++i) {
            const uint32_t c4 = (i * kStreamThreads + threadIdx.x) * 4;
            sv[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, c4 < n ? c4 * 4 : kOobOff, 0, 0);
        }
#pragma unroll
        for(int i = 0; i < kS4; ++i) {
            const uint32_t c4 = (i * kStreamThreads + threadIdx.x) * 4;
            if(c4 < (uint32_t)kTotal) {
                const uint32_t c    = c4 & ~7u;
                const uint32_t slot = (c / 512) * 512 + ((c4 & 4u) ? 256u : 0u) + ((c % 512) / 8) * 4;
                *reinterpret_cast<v4i*>(s_lds + slot) = sv[i];
            }
        }
    }
    __syncthreads();

    // every wave runs the same `iters` steps, so the barriers stay uniform
    // (sched_barrier: the next row's loads are issued before the wait for the
    // current row, never sunk below it by the scheduler)
    for(uint32_t it = 0; it < iters; it += 2) {
        load_row(xb, row + stride);
        __builtin_amdgcn_sched_barrier(0);
        process(xa, row, 0);
        row += stride;
        if(it + 1 >= iters) break;
        load_row(xa, row + stride);
        __builtin_amdgcn_sched_barrier(0);
        process(xb, row, 1);
        row += stride;
    }
}

// THREADS per block, BPC resident blocks per CU (the grid is BPC x CUs, each
// block walking rows with a grid stride).
template <int CPL, int WPR, int THREADS, int BPC = 1, bool NT = false, bool NTS = false>
hipError_t launch_stream(const QuantRows& p, hipStream_t stream)
{
    constexpr int  kGroups = THREADS / kWave / WPR;
    const size_t   lds     = (size_t)CPL * 512 * WPR * sizeof(float);
    // one row group must span the whole row
    if((uint64_t)CPL * 512 * WPR < p.n) return hipErrorInvalidValue;
    static int     max_blocks = [] {
        int dev = 0, cus = 256;
        if(hipGetDevice(&dev) == hipSuccess)
            (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        return cus * BPC;
    }();
    if(lds > 65536) {
        static std::once_flag once;
        std::call_once(once, [] {
            (void)hipFuncSetAttribute(
                reinterpret_cast<const void*>(sq_stream_kernel<CPL, WPR, THREADS, NT, NTS>),
                hipFuncAttributeMaxDynamicSharedMemorySize, 131072);
            (void)hipGetLastError();
        });
    }
    // x and q are addressed through 32-bit buffer offsets: launch row panels
    // whose x and q spans both stay under kPanelBytes (the kernel's
    // out-of-range sentinels lie above it)
    const uint64_t rows_x = kPanelBytes / ((uint64_t)p.ldx * 2);
    const uint64_t rows_q = kPanelBytes / (uint64_t)p.ldq;
    // (a single row spans only its own n columns, whatever the strides)
    const uint32_t panel  = (uint32_t)std::max<uint64_t>(
        1, std::min<uint64_t>(p.rows, std::min(rows_x, rows_q)));
    for(uint32_t r0 = 0; r0 < p.rows; r0 += panel) {
        QuantRows q = p;
        q.rows      = std::min(panel, p.rows - r0);
        q.x         = p.x + (size_t)r0 * p.ldx;
        q.q         = p.q + (size_t)r0 * p.ldq;
        q.r         = p.r + r0;
        const uint32_t need   = (q.rows + kGroups - 1) / kGroups;
        const uint32_t blocks = std::max<uint32_t>(1, std::min<uint32_t>(need, (uint32_t)max_blocks));
        const uint32_t iters  = (q.rows + blocks * kGroups - 1) / (blocks * kGroups);
        hipLaunchKernelGGL((sq_stream_kernel<CPL, WPR, THREADS, NT, NTS>), dim3(blocks), dim3(THREADS), lds,
                           stream, q, iters);
        const hipError_t e = hipGetLastError();
        if(e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int CPL, int WPR, bool MOE>
hipError_t launch_rows(const QuantRows& p, hipStream_t stream)
{
    constexpr int kThreads      = sq_rows_threads(WPR);
    constexpr int kRowsPerBlock = kThreads / kWave / WPR;
    hipLaunchKernelGGL((sq_rows_kernel<CPL, WPR, MOE>),
                       dim3((p.rows + kRowsPerBlock - 1) / kRowsPerBlock), dim3(kThreads), 0,
                       stream, p);
    return hipGetLastError();
}

template <int CPL, int WPR>
hipError_t launch_tokens(const QuantRows& p, hipStream_t stream)
{
    constexpr int  kThreads        = sq_rows_threads(WPR);
    constexpr int  kTokensPerBlock = kThreads / kWave / WPR;
    const uint32_t tokens          = p.rows / p.topk;
    hipLaunchKernelGGL((sq_tokens_kernel<CPL, WPR>),
                       dim3((tokens + kTokensPerBlock - 1) / kTokensPerBlock), dim3(kThreads), 0,
                       stream, p);
    return hipGetLastError();
}

template <bool MOE>
hipError_t launch_twopass(const QuantRows& p, hipStream_t stream)
{
    hipLaunchKernelGGL((sq_twopass_kernel<MOE>), dim3(p.rows), dim3(kSqThreads), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_dense(const QuantRows& p, hipStream_t stream)
{
    const uint32_t n = p.n;
    {
        // 16-byte x loads, 32-byte aligned s loads, 8-byte q stores
        const bool vec = (reinterpret_cast<uintptr_t>(p.x) % 16 == 0) && (p.ldx % 8 == 0)
                         && (reinterpret_cast<uintptr_t>(p.s) % 16 == 0)
                         && (reinterpret_cast<uintptr_t>(p.q) % 8 == 0) && (p.ldq % 8 == 0);
        // aligned dense rows: the streaming kernel (s in LDS, rows double-buffered)
        if(vec && n % 8 == 0) {
            // (configurations chosen by a sweep on MI355X over CPL, WPR,
            // block size and blocks per CU, cache-warm and cache-cold)
            // A few rows (decode): the launch is latency-bound, so each row
            // is spread over all 16 waves of a 1024-thread block.
            if(p.rows <= 64 && n > 4096 && n <= 8192) return launch_stream<1, 16, 1024>(p, stream);
            if(p.rows <= 64 && n > 8192 && n <= 16384) return launch_stream<2, 16, 1024>(p, stream);
            if(n <= 512) return launch_stream<1, 1, 512>(p, stream);
            if(n <= 1024) return launch_stream<2, 1, 512>(p, stream);
            if(n <= 2048) return launch_stream<4, 1, 512>(p, stream);
            // Up to 4096 columns (cold, MALL-rotated buffers): below 1024
            // rows two blocks of 256 threads per CU with a row over two waves
            // (512 x 4096: 4.1 us); from 1024 rows x is read non-temporally
            // (it is read once) and one wave holds a whole row, so its max
            // needs no cross-wave merge: two blocks of 256 threads per CU
            // (2048 x 4096: 9.1 -> 7.3 us, 3328 rows 12.9 -> 10.2 us), except
            // 4096 to 32767 rows, where four blocks of 256 threads with a row
            // over two waves keep more rows in flight (8192 rows: 17.4 us
            // against 18.1), and from 32768 rows, where one 512-thread block
            // of rows over two waves walks them (131072 rows: 307 -> 275 us)
            if(n <= 4096 && p.rows < 1024) return launch_stream<4, 2, 256, 2>(p, stream);
            if(n <= 4096 && p.rows >= 4096 && p.rows < 32768)
                return launch_stream<4, 2, 256, 4, true>(p, stream);
            // (1024-4095 rows also store q non-temporally: 2048 x 4096 cold
            // 7.4 -> 6.5 us; from 4096 rows it no longer pays, 8192 rows 17.6
            // against 18.4 us)
            if(n <= 4096 && p.rows >= 32768) return launch_stream<4, 2, 512, 1, true>(p, stream);
            if(n <= 4096) return launch_stream<8, 1, 256, 2, true, true>(p, stream);
            if(n <= 8192) return launch_stream<4, 4, 512, 2>(p, stream);
            // two row groups of 8 waves per 1024-thread block (4 chunks per
            // lane), x read non-temporally: n = 14336 cold, 2048 / 8192 rows
            // 19.4 -> 16.7 / 64.2 -> 58.0 us
            if(n <= 16384) return launch_stream<4, 8, 1024, 1, true>(p, stream);
            if(n <= 32768) return launch_stream<4, 16, 1024>(p, stream);
        }
    }
    if(n <= 512) return launch_rows<1, 1, false>(p, stream);
    if(n <= 1024) return launch_rows<2, 1, false>(p, stream);
    if(n <= 2048) return launch_rows<4, 1, false>(p, stream);
    if(n <= 4096) return launch_rows<4, 2, false>(p, stream);
    if(n <= 8192) return launch_rows<4, 4, false>(p, stream);
    // Rows of more than 8192: 16 waves, but 4 for more rows than fill the chip
    // (1 / 512 / 8000 rows of 8199: 3.4 / 7.0 / 80 us by 16 waves, 5.5 / 8.2 /
    // 68 by 4; 1 / 8000 of 28671 5.0 / 192 against 8.0 / 230).
    if(n <= 16384 && p.rows > 1024) return launch_rows<8, 4, false>(p, stream);
    if(n <= 16384) return launch_rows<2, 16, false>(p, stream);
    if(n <= 32768) return launch_rows<4, 16, false>(p, stream);
    return launch_twopass<false>(p, stream);
}

hipError_t launch_moe(const QuantRows& p, hipStream_t stream)
{
    const QuantPlan d  = moe_quant_plan(p.rows, p.n, p.topk);
    auto            is = [&](uint32_t chunks, uint32_t waves) {
        return d.chunks == chunks && d.waves == waves;
    };
    if(d.tokens) {
        if(is(1, 1)) return launch_tokens<1, 1>(p, stream);
        if(is(2, 1)) return launch_tokens<2, 1>(p, stream);
        if(is(4, 4)) return launch_tokens<4, 4>(p, stream);
        if(is(2, 16)) return launch_tokens<2, 16>(p, stream);
        return launch_tokens<4, 16>(p, stream);
    }
    if(is(1, 1)) return launch_rows<1, 1, true>(p, stream);
    if(is(1, 2)) return launch_rows<1, 2, true>(p, stream);
    if(is(2, 1)) return launch_rows<2, 1, true>(p, stream);
    if(is(1, 4)) return launch_rows<1, 4, true>(p, stream);
    if(is(4, 1)) return launch_rows<4, 1, true>(p, stream);
    if(is(2, 4)) return launch_rows<2, 4, true>(p, stream);
    if(is(4, 2)) return launch_rows<4, 2, true>(p, stream);
    if(is(8, 1)) return launch_rows<8, 1, true>(p, stream);
    if(is(4, 4)) return launch_rows<4, 4, true>(p, stream);
    if(is(2, 16)) return launch_rows<2, 16, true>(p, stream);
    if(is(4, 16)) return launch_rows<4, 16, true>(p, stream);
    return launch_twopass<true>(p, stream);
}

} // namespace

// By pairs each row is on its own, in as few waves as keep the chip full; by
// tokens x is read once but a token's slots run one after another, which pays
// only where many pairs share few tokens and x is most of the traffic.  Measured
// over 40-8192 tokens, top 1-8, hidden 512-28672 (us by pairs / by tokens):
//   512: 32000 pairs 11.5 / 12.9, 49152 17.0 / 16.4
//   881: 2400 pairs 4.7 / 10.7, 12000 9.9 / 13.7, 19800 16.0 / 17.3, 32000 23.4 / 21.3;
//   1024 (whole 16 bytes): 19800 13.4 / 15.6, 48000 24.1 / 25.8
//   2048: 600 pairs, top 6 3.7 / 7.1, 12000 12.3 / 16.1, 65536 47.1 / 47.6
//   4096: 4200 pairs, top 6 10.7 / 12.3, 16000 25.6 / 29.1, 49152 68.3 / 71.0
//   7168: 2400 pairs, top 8 13.1 / 18.8, 4200 19.6 / 19.0, 24000 87 / 66;
//         top 2 8000 28.5 / 30.0
//   14336: 800 pairs, top 8 13.0 / 18.1, 1400, top 2 15.1 / 13.3, 9000 87 / 61; 176
//         tokens, fewer than the CUs, top 8 16.9 / 18.1, 400, top 4 18.6 / 16.6
//   20000: 2800 pairs, top 4 38 / 39, 6000 69 / 74; 28672: 47 / 42, 95 / 81; top 2
//         3000 44 / 50
QuantPlan moe_quant_plan(uint32_t pairs, uint32_t n, uint32_t topk)
{
    if(n <= 512) return {1, 1, pairs > 36000};
    if(n <= 1024 && pairs <= 1536) return {1, 2, false};
    if(n <= 1024) return {2, 1, pairs > 24576 && n % 8 != 0};
    if(n <= 2048) return pairs <= 1536 ? QuantPlan{1, 4, false} : QuantPlan{4, 1, false};
    if(n <= 4096 && pairs <= 1024) return {2, 4, false};
    if(n <= 4096) return pairs <= 10240 ? QuantPlan{4, 2, false} : QuantPlan{8, 1, false};
    if(n <= 8192) return {4, 4, pairs > 3584 && topk > 2};
    if(n <= 16384) return {2, 16, pairs > 1280 && pairs >= 256 * topk};
    if(n <= 32768) return {4, 16, pairs > 2048 && topk > 2};
    return {0, 0, false};
}

hipError_t launch_smoothquant(const QuantRows& p, hipStream_t stream)
{
    if(p.rows == 0) return hipSuccess;
    return p.topk_ids ? launch_moe(p, stream) : launch_dense(p, stream);
}

} // namespace w8a8
