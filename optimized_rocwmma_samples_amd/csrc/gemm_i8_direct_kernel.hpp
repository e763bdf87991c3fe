// gemm_i8_direct_kernel.hpp -- int8 tile GEMM for gfx950 over operands the
// LDS-DMA tile kernels cannot load: any pointer, row stride and K of the
// primary layout, and the sample layout (A column-major, B [K, N]) in place.
//
// Same MFMA body, LDS tile layout and epilogues as gemm_i8_kernel.hpp; only
// the way in differs.  A load to LDS writes 16 bytes per lane from a 16-byte
// aligned address along K, which these operands do not have, so a k-tile comes
// through registers, kAhead k-tiles before it is used:
//   * K-contiguous rows (RowPair): 16-byte loads at any byte address (eight
//     lanes a row, so a wave load still covers 8 rows x 128 contiguous bytes);
//     only the last k-tile looks at K (a chunk that straddles it is the row's last
//     16 bytes, shifted).
//   * K-major operands (ColPair): a thread loads 4 columns of 16
//     consecutive k rows as dwords (128 contiguous bytes per half wave) and
//     transposes the 16 x 4 bytes with v_perm_b32 into the four 16-byte
//     k-chunks that the tile's rows take.
// Rows past the matrix are clamped to the last one (their outputs are never
// stored), so every load is inside the operand.
//
// What bounds it: the loads' issue and the LDS writes beside the MFMAs, and
// latency where a launch has few tiles.  64 x 64 and 128 x 128 tiles with two
// LDS stages leave room for several blocks per CU, whose barriers overlap.
// Measured: 1000^3 int32 1320 -> 8.0 us, against the one-output-per-thread
// kernel that took these shapes before; 4000 x 4000 x 4001 84 us.
#pragma once

#include "gemm_i8_kernel.hpp"

namespace w8a8 {
namespace gemm {

// x[j]: 4 columns' bytes of k row j (16 of them, `shift` bits too low in each).
// o[c]: column c's 16 bytes along k.
__device__ __forceinline__ void transpose_quad(const uint32_t (&x)[16], uint32_t shift, v4i (&o)[4])
{
#pragma unroll
    for(int g = 0; g < 4; ++g) {
        uint32_t y[4];
#pragma unroll
        for(int j = 0; j < 4; ++j) y[j] = x[4 * g + j] >> shift;
        // 4 x 4 bytes: perm takes bytes 0-3 from its second operand, 4-7 from its first
        const uint32_t lo01 = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u);
        const uint32_t hi01 = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
        const uint32_t hi23 = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
        o[0][g]             = (int)__builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
        o[1][g]             = (int)__builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
        o[2][g]             = (int)__builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
        o[3][g]             = (int)__builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    }
}

// Rows [r0, r0 + R) of a K-contiguous operand, 16-byte chunk (r, c) per thread
// and step.
template <int R, int THREADS>
struct RowLoader {
    static constexpr int kN = R * 8 / THREADS; // chunks per thread and k-tile
    static_assert(kN * THREADS == R * 8, "whole chunks per thread");
    struct Regs {
        v4i v[kN];
    };
    const int8_t* src[kN];
    int           chunk; // the same c for every step (THREADS % 8 == 0)
    uint32_t      k;

    __device__ __forceinline__ RowLoader(const int8_t* p, uint32_t ld, uint32_t rows, uint32_t r0,
                                         uint32_t k_)
        : chunk(threadIdx.x % 8), k(k_)
    {
#pragma unroll
        for(int i = 0; i < kN; ++i) {
            const uint32_t r = min(r0 + (i * THREADS + threadIdx.x) / 8, rows - 1);
            src[i]           = p + (size_t)r * ld + chunk * 16;
        }
    }
    __device__ __forceinline__ void load(Regs& d, uint32_t kt) const
    {
        const uint32_t k0 = kt * 128;
        if(k0 + 128 <= k) { // uniform
#pragma unroll
            for(int i = 0; i < kN; ++i) __builtin_memcpy(&d.v[i], src[i] + k0, 16);
            return;
        }
        const uint32_t kk = k0 + chunk * 16;
        if(k >= 16) { // uniform: the chunk that straddles K is the row's last 16 bytes, shifted
            const bool     part = kk + 16 > k;
            const uint32_t back = part ? 16 - k % 16 : 0; // used where kk < k
#pragma unroll
            for(int i = 0; i < kN; ++i) {
                d.v[i] = v4i{0};
                if(kk < k) {
                    unsigned __int128 x;
                    __builtin_memcpy(&x, src[i] + k0 - back, 16);
                    x >>= 8 * back;
                    __builtin_memcpy(&d.v[i], &x, 16);
                }
            }
            return;
        }
#pragma unroll
        for(int i = 0; i < kN; ++i) { // rows of fewer than 16 bytes
            uint32_t x[4] = {0, 0, 0, 0};
            if(chunk == 0)
                for(uint32_t e = 0; e < k; ++e) x[e / 4] |= (uint32_t)(uint8_t)src[i][e] << (8 * (e % 4));
            d.v[i] = v4i{(int)x[0], (int)x[1], (int)x[2], (int)x[3]};
        }
    }
    __device__ __forceinline__ void store(const Regs& d, int8_t* tile) const
    {
#pragma unroll
        for(int i = 0; i < kN; ++i) {
            const int r = (i * THREADS + threadIdx.x) / 8;
            *reinterpret_cast<v4i*>(tile + r * 128 + (chunk ^ ((r >> 1) & 7)) * 16) = d.v[i];
        }
    }
};

// The A and B tiles' rows of the primary layout.
template <class C>
struct RowPair {
    using LoadA = RowLoader<C::kBM, C::kThreads>;
    using LoadB = RowLoader<C::kBN, C::kThreads>;
    struct Regs {
        typename LoadA::Regs a;
        typename LoadB::Regs b;
    };
    LoadA a;
    LoadB b;
    __device__ __forceinline__ RowPair(const KArgs& p, uint32_t m0, uint32_t n0)
        : a(p.a, p.lda, p.m, m0, p.k), b(p.b, p.ldb, p.n, n0, p.k)
    {
    }
    __device__ __forceinline__ void load(Regs& d, uint32_t kt) const
    {
        a.load(d.a, kt);
        b.load(d.b, kt);
    }
    __device__ __forceinline__ void store(const Regs& d, int8_t* stage) const
    {
        a.store(d.a, stage);
        b.store(d.b, stage + C::kABytes);
    }
};

// The A and B tiles' columns of K-major operands (at least 4 columns each).
// Units of 4 columns x 16 k rows, those of A first; a unit's side is the same
// for a whole wave.  Eight consecutive lanes hold 4 column quads x 2 k-chunks:
// their four rows' LDS writes then fall on the 8 distinct 16-byte slots of
// the swizzled rows.
template <class C>
struct ColPair {
    static constexpr int kUnitsA = C::kBM / 4 * 8, kUnitsB = C::kBN / 4 * 8;
    static constexpr int kN      = (kUnitsA + kUnitsB) / C::kThreads; // per thread and k-tile
    static_assert(kN * C::kThreads == kUnitsA + kUnitsB && kUnitsA % kWave == 0,
                  "whole units per thread, one side per wave");
    struct Regs {
        uint32_t v[kN][16];
    };
    const int8_t* src[kN];
    uint32_t      ld[kN], shift[kN]; // shift: bits to drop where a quad was moved inside
    int           row[kN], chunk[kN], base[kN];
    uint32_t      k;

    __device__ __forceinline__ ColPair(const KArgs& p, uint32_t m0, uint32_t n0) : k(p.k)
    {
#pragma unroll
        for(int i = 0; i < kN; ++i) {
            const int  wid  = i * C::kThreads + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * kWave;
            const bool in_b = wid >= kUnitsA; // wave-uniform
            const int  id   = wid + threadIdx.x % kWave - (in_b ? kUnitsA : 0);
            const int  hi   = (in_b ? C::kBN : C::kBM) / 16; // quads / 4
            row[i]          = ((id & 3) | ((id >> 3) % hi) << 2) * 4;
            chunk[i]        = ((id >> 2) & 1) | ((id >> 3) / hi) << 1;
            base[i]         = in_b ? C::kABytes : 0;
            ld[i]           = in_b ? p.ldb : p.lda;
            const uint32_t rows = in_b ? p.n : p.m, col = (in_b ? n0 : m0) + row[i];
            const uint32_t in   = min(col, rows - 4);
            shift[i]            = min(col - in, 3u) * 8;
            src[i]              = (in_b ? p.b : p.a) + (size_t)chunk[i] * 16 * ld[i] + in;
        }
    }
    __device__ __forceinline__ void load(Regs& d, uint32_t kt) const
    {
        const uint32_t k0   = kt * 128;
        const bool     full = k0 + 128 <= k; // uniform
#pragma unroll
        for(int i = 0; i < kN; ++i) {
            const int8_t* s = src[i] + (size_t)k0 * ld[i];
#pragma unroll
            for(int j = 0; j < 16; ++j) {
                d.v[i][j] = 0;
                if(full || k0 + chunk[i] * 16 + j < k)
                    __builtin_memcpy(&d.v[i][j], s + (size_t)j * ld[i], 4);
            }
        }
    }
    __device__ __forceinline__ void store(const Regs& d, int8_t* stage) const
    {
#pragma unroll
        for(int i = 0; i < kN; ++i) {
            v4i o[4];
            transpose_quad(d.v[i], shift[i], o);
#pragma unroll
            for(int c = 0; c < 4; ++c) {
                const int r = row[i] + c;
                *reinterpret_cast<v4i*>(stage + base[i] + r * 128 + (chunk[i] ^ ((r >> 1) & 7)) * 16)
                    = o[c];
            }
        }
    }
};

// COLS: both operands K-major (the sample layout), else both K-contiguous.
// AHEAD: k-tiles held in registers beyond the one in LDS.
template <class C, int OUT, bool COLS, int AHEAD>
__global__ void __launch_bounds__(C::kThreads) gemm_i8_direct_kernel(KArgs p)
{
    static_assert(C::kStages == 2 && C::kBK == 128 && C::kSubK == 2, "two stages of 128-deep k-tiles");
    static_assert(AHEAD == 1 || AHEAD == 2, "register ring of one or two k-tiles");
    using Pair = std::conditional_t<COLS, ColPair<C>, RowPair<C>>;
    using Regs = typename Pair::Regs;
    extern __shared__ __attribute__((aligned(1024))) int8_t lds[];
    const uint32_t tiles_m = (p.m + C::kBM - 1) / C::kBM;
    const uint32_t tiles_n = (p.n + C::kBN - 1) / C::kBN;
    uint32_t       tm, tn;
    tile_coords<C::kGroupM>(xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    const uint32_t m0 = tm * C::kBM, n0 = tn * C::kBN;
    const uint32_t nk = (p.k + C::kBK - 1) / C::kBK;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;

    const Pair ops(p, m0, n0);
    Regs       regs[AHEAD];
    auto load = [&](Regs& r, uint32_t kt) {
        if(kt < nk) ops.load(r, kt); // uniform
    };
    auto store = [&](const Regs& r, uint32_t kt) { ops.store(r, lds + kt % 2 * C::kStageBytes); };
    FragPipe<C> fp(wave / C::kWavesN, wave % C::kWavesN, lane);
    Acc<C>      acc;
    acc.zero();

    load(regs[0], 0);
    store(regs[0], 0);
#pragma unroll
    for(int d = 0; d < AHEAD; ++d) load(regs[d], 1 + d);
    __syncthreads();
    // k-tile kt is in its stage; slot holds kt + 1 and is refilled with the
    // k-tile AHEAD later.  The stage written here was last read before the
    // previous barrier.
    auto step = [&](uint32_t kt, Regs& slot) {
        const int8_t* s = lds + kt % 2 * C::kStageBytes;
        fp.first(s);
        fp.template step<0>(acc, 0, s, 1);
        fp.last(acc, 1);
        if(kt + 1 < nk) { // uniform
            store(slot, kt + 1);
            load(slot, kt + 1 + AHEAD);
        }
        __syncthreads();
    };
    for(uint32_t kt = 0; kt < nk; kt += AHEAD) {
        step(kt, regs[0]);
        if constexpr(AHEAD == 2)
            if(kt + 1 < nk) step(kt + 1, regs[1]);
    }
    tile_epilogue<C, OUT>(p, m0, n0, lds, acc);
}

// Preconditions (host): COLS needs m >= 4 and n >= 4; every operand and C of
// any size and alignment.
template <class C, bool COLS, int AHEAD>
hipError_t launch_direct(const KArgs& p, int out_type, hipStream_t stream)
{
    static_assert(C::kLdsBytes <= 65536 || C::kStages == 2, "dynamic LDS");
    const dim3 grid(((p.m + C::kBM - 1) / C::kBM) * ((p.n + C::kBN - 1) / C::kBN));
    if constexpr(C::kLdsBytes > 65536) {
        static std::once_flag once;
        std::call_once(once, [] {
            (void)hipFuncSetAttribute(
                reinterpret_cast<const void*>(gemm_i8_direct_kernel<C, W8A8_OUT_I32, COLS, AHEAD>),
                hipFuncAttributeMaxDynamicSharedMemorySize, C::kLdsBytes);
            (void)hipFuncSetAttribute(
                reinterpret_cast<const void*>(gemm_i8_direct_kernel<C, W8A8_OUT_F16, COLS, AHEAD>),
                hipFuncAttributeMaxDynamicSharedMemorySize, C::kLdsBytes);
            (void)hipGetLastError();
        });
    }
    if(out_type == W8A8_OUT_I32)
        hipLaunchKernelGGL((gemm_i8_direct_kernel<C, W8A8_OUT_I32, COLS, AHEAD>), grid,
                           dim3(C::kThreads), C::kLdsBytes, stream, p);
    else
        hipLaunchKernelGGL((gemm_i8_direct_kernel<C, W8A8_OUT_F16, COLS, AHEAD>), grid,
                           dim3(C::kThreads), C::kLdsBytes, stream, p);
    return hipGetLastError();
}

} // namespace gemm
} // namespace w8a8
