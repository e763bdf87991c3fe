// gemm_i8_pack.hpp -- the packed weight layout of the int8 GEMMs.
//
// The "pre-shuffled B" the reference describes for FlatMM
// (rocwmma_flatmm.cpp:12-16) but leaves unimplemented: weights stored once in
// MFMA register order, so that every wave-load of a GEMM reads 1 KiB
// contiguous.
//
// Packed weight layout (w8a8_pack_weights):
//   N is padded to a multiple of 64 (a "slab"), K to a multiple of 128 (a
//   "k-tile"), pad bytes are zero.  For slab s, k-tile t, the 8 KiB block
//   ((s * nKT + t) * 8) KiB holds 8 fragments of 1 KiB, fragment f = nt*4 + g
//   (nt = 32-row half of the slab, g = 32-deep k group).  Inside a fragment,
//   lane l = h*32 + r owns 16 bytes: row s*64 + nt*32 + r, k = t*128 + g*32 +
//   h*16 + [0, 16).  That is exactly the v_mfma_i32_32x32x32_i8 operand a wave
//   holds, so one buffer_load_dwordx4 per fragment reads 1 KiB contiguous (the
//   decode kernels).  Seen by 16-byte chunk c = 2g + h of a row, the block is
//   [nt][c][r]: copied to LDS as it is, the 16 rows x 4 chunks a
//   v_mfma_i32_16x16x64_i8 operand takes are four runs of 256 contiguous
//   bytes, which ds_read_b128 reads without bank conflicts (the tile kernels,
//   gemm_i8_kernel.hpp).
#pragma once

#include "w8a8_device.hpp"

namespace w8a8 {
namespace gemm {

constexpr int kSlab      = 64;   // packed-weight rows per slab (one wave's N extent)
constexpr int kPackK     = 128;  // packed-weight k-tile
constexpr int kPackFrags = 8;    // 1 KiB fragments per (slab, k-tile)

__host__ __device__ inline uint32_t packed_ktiles(uint32_t k) { return (k + kPackK - 1) / kPackK; }
__host__ __device__ inline uint32_t packed_slabs(uint32_t n) { return (n + kSlab - 1) / kSlab; }
__host__ __device__ inline size_t   packed_bytes(uint32_t n, uint32_t k)
{
    return (size_t)packed_slabs(n) * packed_ktiles(k) * kPackFrags * 1024;
}

} // namespace gemm
} // namespace w8a8
