// gemm_i8.hip -- launchers of the int8 GEMM: the gfx950 MFMA tile kernel
// (gemm_i8_kernel.hpp) over row-major or packed weights (gemm_i8_pack.hpp), the
// decode kernels for m <= 64 (gemm_i8_decode_kernel.hpp), the tile kernel for
// operands those do not take (k % 16 != 0, unaligned: gemm_i8_direct_kernel.hpp)
// and the repack used for the reference sample's A col-major / B [K,N] layout.
#include "gemm_i8_decode_kernel.hpp"
#include "gemm_i8_decode_wide_kernel.hpp"
#include "gemm_i8_direct_kernel.hpp"
#include "gemm_i8_kernel.hpp"
#include "gemm_i8_persist_kernel.hpp"
#include "gemm_i8_streamk_kernel.hpp"
#include "w8a8_internal.hpp"

#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <numeric>
#include <tuple>

namespace w8a8 {

namespace {

using gemm::KArgs;

// Production tile configuration, and the smaller tiles of launches that
// would leave most CUs idle with it (plan_tiles).  All on the
// 16 x 16 x 64 MFMA (gemm::Cfg): against the 32 x 32 x 32 form, GEMM-only,
// cold weights, cfg3 projections: M = 8192 1448 -> 1389 µs, M = 2048 411 ->
// 398 µs, M = 512 144 -> 132 µs (sum of the four).
// PB: over packed weights.
// 3 LDS stages in the next two: these launches have few tiles per CU and
// read their panels from HBM, where a third k-tile in flight hides the latency
// (cold weights, M = 512: 128 x 128 o_proj 32 -> 22 µs, down 100 -> 66 µs;
// M = 2048, 128 x 256: o_proj 47 -> 40 µs, down 146 -> 116 µs).
// The last three are short enough that a CU holds two or three blocks, whose
// barriers and waits then overlap: what a launch of few or short tiles lacks
// (plan_tiles says where each wins).
template <bool PB>
struct Tiles {
    using Main   = gemm::Cfg<256, 256, 128, 2, 2, 4, 4, 16, PB>;
    using MidM   = gemm::Cfg<128, 256, 128, 3, 2, 4, 4, 16, PB>; // 8 waves of 64 x 64, 144 KiB LDS
    using Small  = gemm::Cfg<128, 128, 128, 3, 2, 4, 4, 16, PB>; // 8 waves of 64 x 32, 96 KiB LDS
    using Narrow = gemm::Cfg<64, 128, 128, 3, 2, 4, 4, 16, PB>;  // 8 waves of 32 x 32, 72 KiB LDS
    using Tiny   = gemm::Cfg<64, 64, 128, 4, 2, 2, 4, 16, PB>;   // 4 waves of 32 x 32, 64 KiB LDS
    using Row    = gemm::Cfg<32, 64, 128, 4, 1, 2, 4, 16, PB>;   // 2 waves of 32 x 32, 48 KiB LDS
};
using GemmMain    = Tiles<false>::Main;
using GemmMidM    = Tiles<false>::MidM;
using GemmSmall   = Tiles<false>::Small;
// Decode configurations: <32-row m tiles, 32-row weight tiles, waves, ring>.
using DecSmall   = gemm::DecCfg<1, 1, 4, 3>; // m <= 32, or <= 16 packed
using DecSmallW  = gemm::DecCfg<1, 2, 8, 3>; // packed, 8 <= m <= 32, many slabs
using DecMid     = gemm::DecCfg<2, 1, 8, 3>; // 32 < m <= 64
using DecMidW    = gemm::DecCfg<2, 2, 8, 2>; // packed, 32 < m <= 64, many slabs
// packed, 32 < m <= 64 with a split-K workspace: 8 half slabs per block share
// the A k-tile through LDS
using DecWide    = gemm::DecWideCfg<8, 3>;
// 4 waves of 32 weight rows: twice the blocks of DecWide, so half its K
// splits for the same fill (fewer partials; none where DecWide needs 2):
// M = 64, W [28672, 8192] 55.5 -> 49.9 us, W [8192, 28672] 59.0 -> 56.3 us.
using DecWide4   = gemm::DecWideCfg<4, 4>;
// A packed GEMM with at least this many 64-row slabs has enough blocks at
// 64 rows per block to fill the chip; fewer slabs run 32 rows per block.
constexpr uint32_t kWideSlabs = 384;

// ---------------------------------------------------------------------------
// Generic strided kernel: one thread per output (generic_pays, and the sample
// layout with fewer than 4 rows or columns and no workspace to repack into).
// ---------------------------------------------------------------------------
template <int OUT>
__global__ void __launch_bounds__(256) gemm_i8_generic_kernel(KArgs p, size_t sam, size_t sak,
                                                              size_t sbn, size_t sbk)
{
    const uint32_t n = blockIdx.x * 16 + (threadIdx.x & 15);
    const uint32_t m = blockIdx.y * 16 + (threadIdx.x >> 4);
    if(m >= p.m || n >= p.n) return;
    int32_t acc = 0;
    for(uint32_t k = 0; k < p.k; ++k)
        acc += (int32_t)p.a[m * sam + k * sak] * (int32_t)p.b[n * sbn + k * sbk];
    if constexpr(OUT == W8A8_OUT_I32) {
        reinterpret_cast<int32_t*>(p.c)[(size_t)m * p.ldc + n] = acc;
    } else {
        float f = (float)acc;
        if(p.sa == nullptr && p.sb == nullptr)
            f = f * (p.tsa * p.tsb);
        else
            f = (f * (p.sa ? p.sa[m] : p.tsa)) * (p.sb ? p.sb[n] : p.tsb);
        reinterpret_cast<uint16_t*>(p.c)[(size_t)m * p.ldc + n] = float_to_half_bits_2step(f);
    }
}

// Repack of the sample layout: dst[r, c] = src[c * ld + r] for both operands in
// one launch, 0 for c in [cols, ldd) (the K padding).  A block moves a tile of
// 128 rows r x 128 columns c: each thread loads 4 bytes (4 rows) of 16
// consecutive source rows, 128 contiguous bytes per half wave, transposes them
// with v_perm_b32 (gemm::transpose_quad) into 16-byte pieces of 4 destination
// rows, and the tile goes through LDS (swizzled as the GEMM's tiles, no bank
// conflicts) so that 8 lanes store 128 contiguous bytes of a row.  HBM-bound;
// any pointer and ld.  3840 x 4096 x 4096, both operands: 18.4 -> 11.1 us (6 TB/s);
// 4095^3 67.6 -> 16.4 us (two launches whose edge and unaligned loads went byte by
// byte).
struct Repack {
    const int8_t* src;
    int8_t*       dst;
    uint32_t      ld, rows; // source leading dimension; rows of dst
};

__global__ void __launch_bounds__(256) repack_i8_kernel(Repack a, Repack b, uint32_t blocks_a,
                                                        uint32_t cols, uint32_t ldd)
{
    __shared__ __attribute__((aligned(16))) int8_t tile[128 * 128];
    const bool     in_b = blockIdx.x >= blocks_a; // uniform
    const Repack   p    = in_b ? b : a;
    const uint32_t id   = blockIdx.x - (in_b ? blocks_a : 0);
    const uint32_t rt   = (p.rows + 127) / 128;
    const uint32_t r0 = id % rt * 128, c0 = id / rt * 128;
    const uint32_t t = threadIdx.x;
    {
        const uint32_t row = ((t & 3) | ((t >> 3) % 8) << 2) * 4;
        const uint32_t ch  = ((t >> 2) & 1) | ((t >> 3) / 8) << 1;
        const uint32_t in  = p.rows < 4 ? 0 : min(r0 + row, p.rows - 4); // a quad past the end moves inside
        const uint32_t sh  = min(r0 + row - in, 3u) * 8;
        uint32_t       x[16];
        if(p.rows < 4) { // uniform: 1-3 source columns, byte by byte, all in flight
#pragma unroll
            for(int j = 0; j < 16; ++j) {
                const uint32_t c = c0 + ch * 16 + j;
                uint32_t       e[3];
#pragma unroll
                for(uint32_t i = 0; i < 3; ++i) // past the end: the last row or column
                    e[i] = (uint8_t)p.src[(size_t)min(c, cols - 1) * p.ld + min(i, p.rows - 1)];
                x[j] = c < cols ? e[0] | e[1] << 8 | e[2] << 16 : 0;
            }
        } else if(c0 + 128 <= cols) { // uniform
            const int8_t* s = p.src + (size_t)(c0 + ch * 16) * p.ld + in;
#pragma unroll
            for(int j = 0; j < 16; ++j) __builtin_memcpy(&x[j], s + (size_t)j * p.ld, 4);
        } else {
#pragma unroll
            for(int j = 0; j < 16; ++j) {
                const uint32_t c = c0 + ch * 16 + j;
                x[j]             = 0;
                if(c < cols) __builtin_memcpy(&x[j], p.src + (size_t)c * p.ld + in, 4);
            }
        }
        v4i o[4];
        gemm::transpose_quad(x, sh, o);
#pragma unroll
        for(int i = 0; i < 4; ++i) {
            const uint32_t r = row + i;
            *reinterpret_cast<v4i*>(tile + r * 128 + (ch ^ ((r >> 1) & 7)) * 16) = o[i];
        }
    }
    __syncthreads();
#pragma unroll
    for(int i = 0; i < 4; ++i) {
        const uint32_t r = (i * 256 + t) / 8, ch = t % 8;
        const v4i      v = *reinterpret_cast<const v4i*>(tile + r * 128 + (ch ^ ((r >> 1) & 7)) * 16);
        // ldd is a multiple of 16: a chunk is inside the row or past it
        if(r0 + r < p.rows && c0 + ch * 16 < ldd)
            *reinterpret_cast<v4i*>(p.dst + (size_t)(r0 + r) * ldd + c0 + ch * 16) = v;
    }
}

// One thread per 16-byte packed chunk.
__global__ void __launch_bounds__(256) pack_weights_kernel(const int8_t* __restrict__ w,
                                                           uint32_t n, uint32_t k, uint32_t ldw,
                                                           int8_t* __restrict__ out,
                                                           size_t nchunks)
{
    const size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if(idx >= nchunks) return;
    const uint32_t nkt   = gemm::packed_ktiles(k);
    const uint32_t lane  = idx % 64;
    const uint32_t frag  = (idx / 64) % gemm::kPackFrags;
    const size_t   blk   = idx / (64 * gemm::kPackFrags); // slab * nkt + ktile
    const uint32_t kt    = blk % nkt;
    const uint32_t slab  = blk / nkt;
    const uint32_t row   = slab * gemm::kSlab + (frag / 4) * 32 + lane % 32;
    const uint32_t k0    = kt * gemm::kPackK + (frag % 4) * 32 + (lane / 32) * 16;
    int4           v     = make_int4(0, 0, 0, 0);
    if(row < n) {
        const int8_t* src = w + (size_t)row * ldw + k0;
        if(k0 + 16 <= k && (reinterpret_cast<uintptr_t>(src) % 16) == 0) {
            v = *reinterpret_cast<const int4*>(src);
        } else {
            int8_t tmp[16];
            for(int e = 0; e < 16; ++e) tmp[e] = (k0 + e < k) ? src[e] : 0;
            v = *reinterpret_cast<const int4*>(tmp);
        }
    }
    reinterpret_cast<int4*>(out)[idx] = v;
}

KArgs make_kargs(const GemmArgs& g)
{
    return KArgs{g.a,   g.b,   g.c,   g.scale_a, g.scale_b, g.m,   g.n,
                 g.k,   g.lda, g.ldb, g.ldc,     g.tsa,     g.tsb};
}

// Sub-problem of rows [n0, n0 + nn) of the weights.  For packed weights n0 is
// a multiple of the 64-row slab and b points at the slab's packed block.
KArgs n_panel(const GemmArgs& g, uint32_t n0, uint32_t nn, bool packed)
{
    const size_t esz = g.out_type == W8A8_OUT_I32 ? 4 : 2;
    KArgs        p   = make_kargs(g);
    p.n              = nn;
    p.b = packed ? g.b + (size_t)(n0 / gemm::kSlab) * gemm::packed_ktiles(g.k) * gemm::kPackFrags * 1024
                 : g.b + (size_t)n0 * g.ldb;
    p.c  = static_cast<int8_t*>(g.c) + (size_t)n0 * esz;
    p.sb = g.scale_b ? g.scale_b + n0 : nullptr;
    return p;
}

// Weight rows per launch so that every buffer resource stays under 2 GiB
// (a multiple of the 64-row slab).
uint32_t weight_panel_rows(const GemmArgs& g, bool packed)
{
    constexpr size_t kLimit = 0x7FFFFFFFull;
    size_t           rows;
    if(packed)
        rows = kLimit / ((size_t)gemm::packed_ktiles(g.k) * gemm::kPackFrags * 1024) * gemm::kSlab;
    else
        rows = (kLimit - g.k) / g.ldb + 1;
    rows = std::max<size_t>(gemm::kSlab, rows / gemm::kSlab * gemm::kSlab);
    return (uint32_t)std::min<size_t>(g.n, rows);
}

uint32_t device_cus()
{
    static const uint32_t cus = [] {
        int dev = 0, c = 256;
        if(hipGetDevice(&dev) == hipSuccess)
            (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
        return (uint32_t)c;
    }();
    return cus;
}

// ---------------------------------------------------------------------------
// Plan of one tile launch: the configuration and the number of K pieces.
// ---------------------------------------------------------------------------
enum class TileCfg { kMain, kMidM, kSmall, kNarrow, kTiny, kRow, kDecode };

struct TilePlan {
    TileCfg cfg;
    uint32_t parts; // K pieces per tile (gemm_i8_split_kernel + fixup when > 1)
    size_t   bytes; // int32 partials of the pieces
};

// Time of a launch in µs, fitted per configuration to launches of random sizes
// (m 1-4096, n 64-28672, k 512-28672) with weights cold and in the MALL:
//   fixed + sum over a CU's blocks of k-tiles x step[blocks resident together]
//   + round x rounds of resident blocks after the first
//   + out_mb x output MB + w_mb x weight MB
//   + (pieces > 1) (split + split_mb x partial MB)
// with step x cross where row-major operands' rows cross 128-byte lines (K no
// multiple of 128: a 128-byte row piece off a line is two requests).  The
// shortest tiles make the most requests for their sums, and with the chip full
// of them the requests are what their k-steps wait for: there the factor rises
// to 1 + full x share of the rows off a line, from `from` blocks a CU to `to`
// (181 x 19016 x 9488: 64 x 64 tiles, 3.5 blocks a CU, 122 us against 99 in 128 x
// 256 ones; one factor for every load had said 81 against 88).  Fitted on 193
// sizes with such K, every configuration and 1-8 pieces measured.
// m <= 64 (kDecodeMaxM) never fills taller tiles, larger m never needs shorter
// ones.  64 x 128 tiles in more rows than one have costs of their own: each
// weight panel is read by several blocks, and cold weights keep a k-step waiting
// longer (529 x 1984 x 8192: 32.6 us in one round of them, 24 estimated with the
// one row's costs; 22.9 in 128 x 128 tiles).  Their and the 128 x 128 tiles' step and
// all `round`s: every plan of 1600 sizes of 65-3000 rows measured, row-major and
// packed, cold and in the MALL; the plan is on average 0.75% slower than the best and
// for 2% of the sizes by more than 10% (1.6 and 6% with one row's costs and no
// round).  500 more of K 64-1024 and up to 70000 columns: 1.3% against 4.1%.
struct CfgCost {
    TileCfg  cfg;
    uint32_t bm, bn, resident; // resident: blocks a CU holds (LDS)
    uint32_t least, most;      // the m it serves
    double   fixed, step[3], round, split, split_mb, out_mb, w_mb, cross, full, from, to;
};
constexpr uint32_t kAnyM    = 0xFFFFFFFFu;
constexpr CfgCost  kCosts[] = {
    {TileCfg::kMain, 256, 256, 1, 65, kAnyM, 6.2, {1.19}, 1.0, 6.5, 0.45, 0.27, 0.044, 1.06, 0.0, 0.0, 1.0},
    {TileCfg::kMidM, 128, 256, 1, 65, kAnyM, 4.9, {0.71}, 0.0, 4.7, 0.38, 0.34, 0.043, 1.25, 0.0, 0.0, 1.0},
    {TileCfg::kSmall, 128, 128, 1, 65, kAnyM, 3.6, {0.45}, 0.7, 3.8, 0.40, 0.40, 0.023, 1.25, 0.0, 0.0, 1.0},
    {TileCfg::kNarrow, 64, 128, 2, 1, 64, 3.2, {0.30, 0.63}, 0.0, 3.7, 0.32, 0.23, 0.061, 1.40, 0.0, 0.0, 1.0},
    {TileCfg::kNarrow, 64, 128, 2, 65, kAnyM, 3.2, {0.375, 0.745}, 0.7, 3.7, 0.32, 0.30, 0.061, 1.40, 0.0, 0.0, 1.0},
    {TileCfg::kTiny, 64, 64, 2, 1, kAnyM, 3.3, {0.24, 0.42}, 0.3, 3.3, 0.47, 0.37, 0.030, 1.10, 0.8, 0.8, 2.0},
    {TileCfg::kRow, 32, 64, 3, 1, 64, 3.4, {0.23, 0.36, 0.59}, 0.0, 3.0, 0.41, 0.0, 0.048, 1.02, 0.6, 0.9, 1.5},
};
static_assert(kDecodeMaxM == 64, "the rows that kCosts' entries serve");
constexpr uint32_t kMinKtPlan    = 6;        // k-tiles of a K piece, at least
constexpr size_t   kMaxPlanBytes = 64 << 20; // partials of a plan, at most
// A split call launches twice, and the host needs about 3.5 µs a launch and
// 4 µs around it: an eager caller does not see a GPU time below that (25 x 784 x
// 2944, split 15.0 -> 19.8 µs a layer although its kernels take 2 µs less).
constexpr double kSplitHostUs = 11.0;

uint32_t ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// seen: what the caller waits for, at least the host's time of a split call; gpu
// decides between plans that are alike in it (a replayed graph or a caller with
// other work in flight sees the GPU's time).
struct PlanTime {
    double seen, gpu;
    bool   operator<(const PlanTime& o) const
    {
        return seen != o.seen ? seen < o.seen : gpu < o.gpu;
    }
};

// What a k-step of row-major operands takes against one of whole 128-byte lines.
double line_factor(const CfgCost& c, uint32_t k, uint64_t blocks)
{
    if(k % 128 == 0) return 1.0;
    const double ramp
        = std::clamp(((double)blocks / device_cus() - c.from) / (c.to - c.from), 0.0, 1.0);
    const double off = 1.0 - std::gcd(k, 128u) / 128.0; // rows off a line
    return std::max(c.cross, 1.0 + c.full * off * ramp);
}

PlanTime plan_cost(const CfgCost& c, uint32_t m, uint32_t n, uint32_t k, uint32_t parts,
                   bool packed)
{
    const uint32_t cus    = device_cus();
    const uint32_t tm     = ceil_div(m, c.bm);
    const uint64_t blocks = (uint64_t)tm * ceil_div(n, c.bn) * parts;
    const double   factor = packed ? 1.0 : line_factor(c, k, blocks);
    const double   steps  = ceil_div(ceil_div(k, 128), parts) * factor;
    uint64_t       per_cu = (blocks + cus - 1) / cus;
    double         t      = c.fixed + 2e-6 * m * n * c.out_mb + 1e-6 * n * (double)k * c.w_mb;
    // launch_main runs a last round of at most half the CUs as smaller tiles
    if(c.cfg == TileCfg::kMain && per_cu > 1 && blocks % cus != 0 && blocks % cus * 2 <= cus
       && blocks / cus * cus % tm == 0) {
        t += steps * kCosts[1].step[0];
        --per_cu;
    }
    t += steps * (per_cu / c.resident * c.step[c.resident - 1]
                  + (per_cu % c.resident ? c.step[per_cu % c.resident - 1] : 0.0))
         + c.round * ((per_cu - 1) / c.resident);
    if(parts == 1) return {t, t};
    t += c.split + 4e-6 * blocks * c.bm * c.bn * c.split_mb;
    return {std::max(t, kSplitHostUs), t};
}

// The row-major decode kernel (32 weight rows a block, its waves splitting K
// inside the block): the fewest microseconds where the whole launch is a few
// k-tiles per wave, e.g. 2 x 784 x 1472 5.3 µs against 6.2 for the best tiles.
double decode_cost(uint32_t m, uint32_t n, uint32_t k)
{
    const double nk = ceil_div(k, 128), blocks = ceil_div(n, 32);
    return 2.1 + nk * (0.29 * std::ceil(blocks / device_cus())
                       + 0.11 * (m <= 32 ? 1 : 2) * blocks / device_cus());
}

// The plan of least estimated time among those whose partials fit ws_bytes.
// 256 x 256 tiles where the persistent kernel may run them (two whole rounds,
// K <= 4096) and from four rounds on, unless a quarter of their rows or more would
// be padding: 151936 columns of K = 4096 1 / 64 / 100 / 300 rows 159 / 172 /
// 179 / 267 us in 256 x 256 tiles, 113 / 129 / 157 / 252 in the searched ones (64 x
// 64, 64 x 128, 128 x 128, 128 x 256).  Otherwise what the launch lacks
// decides: blocks, k-tiles per block or both.  m <= 64: row-major weights also have
// the decode kernel.  Against the fixed rules this replaced (largest tile
// that fills 3/4 of the CUs, K split when half of them idle): 128 x 4096 x
// 4096 15.0 -> 11.4 µs, 512 x 4096 x 4096 20.0 -> 14.7, 226 x 384 x 12224
// 17.3 -> 13.6, 24 x 16480 x 12672 113 -> 49, 1 x 19584 x 7680 71 -> 33; the
// plan's time is within 2% of the best plan's on average.
TilePlan search_plan(uint32_t m, uint32_t n, uint32_t k, size_t ws_bytes, bool decode, bool packed)
{
    TilePlan best{TileCfg::kMain, 1, 0};
    if((uint64_t)ceil_div(m, 256) * ceil_div(n, 256) >= (k <= 4096 ? 2ull : 4ull) * device_cus()
       && m * 4ull > ceil_div(m, 256) * 768ull)
        return best;
    const double   dec  = decode ? decode_cost(m, n, k) : 1e300;
    PlanTime       cost{dec, dec};
    const uint32_t most = std::min(gemm::kMaxParts, ceil_div(k, 128) / kMinKtPlan);
    if(decode) best.cfg = TileCfg::kDecode;
    for(const CfgCost& c : kCosts) {
        if(m < c.least || m > c.most) continue;
        const uint64_t tiles = (uint64_t)ceil_div(m, c.bm) * ceil_div(n, c.bn);
        for(uint32_t p = 1; p <= std::max(1u, most); ++p) {
            const uint64_t bytes = p == 1 ? 0 : tiles * p * c.bm * c.bn * 4;
            if(bytes > std::min(ws_bytes, kMaxPlanBytes)
               || (p > 1 && tiles * p > (uint64_t)device_cus() * c.resident))
                break;
            const PlanTime t = plan_cost(c, m, n, k, p, packed);
            if(t < cost) {
                cost = t;
                best = TilePlan{c.cfg, p, (size_t)bytes};
            }
        }
    }
    // Up to 16 rows of whole 128-byte lines (K 1536-4000) the decode kernel keeps what
    // tiles neither cut along K nor are estimated 10% faster for: 231 sizes within that
    // run through it 15% faster with weights in L2, 3.5% in the MALL, 1.5% cold (1 x 752
    // x 2816 5.7 us warm, 8.4 in 32 x 64 tiles).  Off the lines it is 18% faster warm but
    // 3-4% slower elsewhere (37 sizes), and below 1536 slower in all three.  Weights of
    // fewer than 256 rows, a megabyte or less, it always keeps: 1 x 21 x 3856 5.5 us,
    // 11.2 in 32 x 64 tiles; 19 sizes 1.85 times as fast in L2, 1.5 in the MALL, 2% slower cold.
    if(m <= 16 && k >= 1536 && best.parts == 1
       && decode && (n < 256 || (k % 128 == 0 && dec < 1.1 * cost.seen)))
        best.cfg = TileCfg::kDecode;
    return best;
}

// search_plan, with the last plans of each host thread kept: a call asks for
// its plan two or three times (the workspace size, the route, the launch) and
// the search takes half a microsecond of a 4 µs call.
TilePlan plan_tiles(uint32_t m, uint32_t n, uint32_t k, size_t ws_bytes, bool decode, bool packed)
{
    struct Entry {
        uint32_t m = 0, n = 0, k = 0; // m = 0: empty
        bool     decode = false, packed = false;
        size_t   ws     = 0;
        TilePlan plan{};
    };
    constexpr uint32_t        kEntries = 64;
    static thread_local Entry seen[kEntries];
    ws_bytes = std::min(ws_bytes, kMaxPlanBytes);
    Entry& e = seen[(m * 31 + n * 17 + k * 7 + (ws_bytes != 0) * 4 + decode * 2 + packed)
                    % kEntries];
    if(e.m != m || e.n != n || e.k != k || e.decode != decode || e.packed != packed
       || e.ws != ws_bytes)
        e = Entry{m,      n,        k, decode, packed,
                  ws_bytes, search_plan(m, n, k, ws_bytes, decode, packed)};
    return e.plan;
}

} // namespace

// One tile for a grouped launch: the plan's costs over the groups' tiles, each
// CU's blocks at the tiles' mean k-tiles (the longest group's where no CU has
// two blocks).  Against the tallest tile that fills 3/4 of the CUs: 13 groups
// of 1-901 rows, 3584 x 3776, 116 -> 82 us a call; 7 and 67 rows, 1280 x 576,
// kernel 7.4 -> 5.2 us; 256 / 512 / 128 / 768 rows, 4096^2, stays on 208 tiles
// of 128 x 256 (35 -> 34 us).  Rows off a 128-byte line count as in plan_cost: 60 groups of
// 622 rows, 3968 x 3568, 875 -> 746 us, 16 of 288, 5600 x 4448, 224 -> 199.
GroupedTile grouped_gemm_tile(const w8a8_group_desc* groups, uint32_t ngroups)
{
    GroupedTile best{0, 0, 0};
    double      cost = 1e300;
    for(const CfgCost& c : kCosts) {
        if(c.most != kAnyM) continue;
        // this runs on each call: shifts for the tile's divisions, and one loop, [1] the
        // groups with rows off a line, whose factor the last of them gives
        const int sm = __builtin_ctz(c.bm), sn = __builtin_ctz(c.bn);
        uint64_t  tiles = 0, steps[2] = {0, 0}, most[2] = {0, 0};
        uint32_t  off_k = 0;
        double    out = 0, w = 0;
        for(uint32_t i = 0; i < ngroups; ++i) {
            const w8a8_group_desc& g = groups[i];
            if(g.m == 0) continue;
            const uint64_t t   = (uint64_t)((g.m + c.bm - 1) >> sm) * ((g.n + c.bn - 1) >> sn);
            const uint64_t k   = ceil_div(g.k, 128);
            const int      off = g.k % 128 != 0;
            tiles += t;
            steps[off] += t * k;
            most[off] = std::max(most[off], k);
            if(off) off_k = g.k;
            out += 2e-6 * g.m * g.n;
            w += 1e-6 * g.n * (double)g.k;
        }
        if(tiles == 0 || tiles > 0x7FFFFFFFull) continue;
        const double   f      = off_k ? line_factor(c, off_k, tiles) : 1.0;
        const uint64_t per_cu = (tiles + device_cus() - 1) / device_cus();
        const double   nk     = per_cu == 1 ? std::max<double>(most[0], most[1] * f)
                                            : (steps[0] + steps[1] * f) / tiles;
        const double   t      = c.fixed + out * c.out_mb + w * c.w_mb
                         + nk * (per_cu / c.resident * c.step[c.resident - 1]
                                 + (per_cu % c.resident ? c.step[per_cu % c.resident - 1] : 0.0))
                         + c.round * ((per_cu - 1) / c.resident);
        if(t < cost) {
            cost = t;
            best = GroupedTile{c.bm, c.bn, (uint32_t)tiles};
        }
    }
    return best;
}

// sizes: groups alike (up to 64), their m, n, k.
void grouped_plan(const uint32_t* sizes, uint32_t* plan)
{
    w8a8_group_desc groups[64] = {};
    for(auto& g : groups) g.m = sizes[1], g.n = sizes[2], g.k = sizes[3];
    const GroupedTile t = grouped_gemm_tile(groups, std::min(sizes[0], 64u));
    plan[0] = t.bm, plan[1] = t.bn, plan[2] = 1;
}

uint32_t direct_tile(uint32_t m, uint32_t n);

// The plan of a GEMM over row-major (with at least 16-byte aligned operands) or
// packed weights, for tests: tile rows and columns, K pieces; the decode kernel
// as 0 x 32.
void gemm_plan(const uint32_t* sizes, bool packed, uint32_t* plan)
{
    const TilePlan p = plan_tiles(sizes[0], sizes[1], sizes[2], sizes[3],
                                  !packed && sizes[0] <= kDecodeMaxM, packed);
    plan[0] = 0, plan[1] = 32, plan[2] = p.parts;
    for(const CfgCost& c : kCosts)
        if(c.cfg == p.cfg) plan[0] = c.bm, plan[1] = c.bn;
}

// The same for operands of any alignment and K (sizes[3] = 0) or the sample layout
// in place (1): the direct kernel's tile, or 0 x 0 for the generic kernel.
void gemm_any_plan(const uint32_t* sizes, uint32_t* plan)
{
    GemmArgs g{};
    g.m = sizes[0], g.n = sizes[1], g.k = sizes[2];
    const bool kn = sizes[3] != 0, one = generic_pays(g, kn) || (kn && !gemm_direct_kn_ok(g));
    plan[0] = plan[1] = one ? 0 : direct_tile(g.m, g.n);
    plan[2]           = 1;
}

namespace {

// K splits of the wide decode kernel for one weight panel: the count that
// minimises the weight bytes of the busiest CU, ceil(blocks / CUs) / splits
// (the fewest splits among equals), at least 8 k-tiles per split; 1 = no
// split.  E.g. 112 panels of W1 on 256 CUs: 2 splits (224 blocks, one per
// CU) rather than 3 (336 blocks: 80 CUs would stream two).
uint32_t decode_wide_splits(const GemmArgs& g, uint32_t n)
{
    const uint32_t cus  = device_cus();
    const uint32_t nblk = (n + DecWide::kRows - 1) / DecWide::kRows;
    const uint32_t nkt  = gemm::packed_ktiles(g.k);
    const uint32_t most = std::max<uint32_t>(1, std::min<uint32_t>(nkt / 8, 8));
    uint32_t       best = 1;
    double         cost = 1e30;
    for(uint32_t s = 1; s <= most; ++s) {
        const double c = (double)((nblk * s + cus - 1) / cus) / s;
        if(c < cost * (1 - 1e-9)) {
            cost = c;
            best = s;
        }
    }
    return best;
}

bool decode_wide_shape(const GemmArgs& g) { return g.m > 32 && g.m <= kDecodeMaxM; }

} // namespace

size_t packed_workspace_bytes(const GemmArgs& g)
{
    if(g.m > kDecodeMaxM) return plan_tiles(g.m, g.n, g.k, kMaxPlanBytes, false, true).bytes;
    if(!decode_wide_shape(g) || !gemm_decode_ok(g)) return 0;
    const uint32_t step = weight_panel_rows(g, true);
    size_t         most = 0;
    for(uint32_t n0 = 0; n0 < g.n; n0 += step) {
        const uint32_t nn = std::min(step, g.n - n0);
        most = std::max(most, gemm::decode_ws_bytes(g.m, nn, decode_wide_splits(g, nn)));
    }
    return most;
}

bool gemm_decode_ok(const GemmArgs& g)
{
    return g.m <= kDecodeMaxM && (uint64_t)(g.m - 1) * g.lda + g.k < 0x7FFFFFFFull;
}

// The row quantized inside the decode kernel (w8a8_fused_sq_gemm_packed at
// m <= kFuseRows = 1 and k <= kFuseMaxK): every block quantizes the row
// before its A-dependent MFMAs, a prologue that grows with K.  It pays where
// it is short and saves the quantizer launch: M = 1, N = K = 4096 8.9 ->
// 7.2 us, N = K = 1024 5.7 -> 4.1 us, [14336, 4096] 13.8 -> 12.0 us, W1
// [28672, 8192] level (41.8 / 41.7 us); at W2 [8192, 28672] (one block per
// CU, 28672-element rows) it cost 48.9 -> 54.5 us, so longer rows keep the
// separate quantizer.
constexpr uint32_t kFuseMaxK = 8192;
bool decode_fuse_ok(uint32_t m, uint32_t k)
{
    const uint64_t pitch = (uint64_t)gemm::packed_ktiles(k) * gemm::kPackK + gemm::kFusePad;
    return m >= 1 && m <= gemm::kFuseRows && k <= kFuseMaxK
           && DecSmall::kLdsBytes + m * pitch <= 160 * 1024;
}

hipError_t launch_gemm_decode_fused(const GemmArgs& g, const FuseArgs& f, hipStream_t stream)
{
    const uint32_t    ka = gemm::packed_ktiles(g.k) * gemm::kPackK;
    const gemm::FuseQ fq{f.x, f.s, f.q, f.r, f.ldx, ka, ka + gemm::kFusePad, f.qmax};
    const uint32_t step   = weight_panel_rows(g, true);
    for(uint32_t n0 = 0; n0 < g.n; n0 += step) {
        const KArgs      p = n_panel(g, n0, std::min(step, g.n - n0), true);
        const hipError_t e = gemm::launch_decode_fused<DecSmall>(p, fq, stream);
        if(e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_gemm_decode(const GemmArgs& g, bool packed, void* ws, size_t ws_bytes,
                              hipStream_t stream)
{
    if(g.m == 0 || g.n == 0) return hipSuccess;
    const uint32_t step   = weight_panel_rows(g, packed);
    const bool     wide   = packed && gemm::packed_slabs(g.n) >= kWideSlabs;
    for(uint32_t n0 = 0; n0 < g.n; n0 += step) {
        const KArgs p = n_panel(g, n0, std::min(step, g.n - n0), packed);
        hipError_t  e;
        if(packed && decode_wide_shape(g) && ws != nullptr) {
            // the workspace holds every panel's partials (panels run in stream order)
            const uint32_t splits = decode_wide_splits(g, p.n);
            // the 4-wave form: twice the blocks, so half the splits for the
            // same fill (1 = unsplit, no reduce launch)
            const uint64_t b4 = (uint64_t)(p.n + DecWide4::kRows - 1) / DecWide4::kRows * (splits / 2);
            if(splits % 2 == 0 && b4 * 4 >= (uint64_t)device_cus() * 3 && b4 <= device_cus()
               && gemm::decode_ws_bytes(g.m, p.n, splits / 2) <= ws_bytes) {
                e = gemm::launch_decode_wide<DecWide4>(p, g.out_type,
                                                       static_cast<int32_t*>(ws), splits / 2,
                                                       stream);
                if(e != hipSuccess) return e;
                continue;
            }
            if(gemm::decode_ws_bytes(g.m, p.n, splits) <= ws_bytes) {
                e = gemm::launch_decode_wide<DecWide>(p, g.out_type,
                                                      static_cast<int32_t*>(ws), splits, stream);
                if(e != hipSuccess) return e;
                continue;
            }
        }
        if(packed) {
            // 8 <= m <= 16 on many slabs: 64 weight rows per block halve the
            // re-reads of the activation rows (M=16 N=28672: 54 -> 52 us)
            if((g.m <= 16 && (!wide || g.m < 8)) || (g.m <= 32 && !wide))
                e = gemm::launch_decode<DecSmall, true>(p, g.out_type, stream);
            else if(g.m <= 32)
                e = gemm::launch_decode<DecSmallW, true>(p, g.out_type, stream);
            else if(!wide)
                e = gemm::launch_decode<DecMid, true>(p, g.out_type, stream);
            else
                e = gemm::launch_decode<DecMidW, true>(p, g.out_type, stream);
        } else {
            if(g.m <= 32)
                e = gemm::launch_decode<DecSmall, false>(p, g.out_type, stream);
            else
                e = gemm::launch_decode<DecMid, false>(p, g.out_type, stream);
        }
        if(e != hipSuccess) return e;
    }
    return hipSuccess;
}

size_t packed_weight_bytes(uint32_t n, uint32_t k) { return gemm::packed_bytes(n, k); }

hipError_t launch_pack_weights(const int8_t* w, uint32_t n, uint32_t k, uint32_t ldw,
                               int8_t* packed, hipStream_t stream)
{
    const size_t chunks = gemm::packed_bytes(n, k) / 16;
    hipLaunchKernelGGL(pack_weights_kernel, dim3((chunks + 255) / 256), dim3(256), 0, stream, w, n,
                       k, ldw, packed, chunks);
    return hipGetLastError();
}

bool gemm_fast_path_ok(const GemmArgs& g)
{
    // every launch addresses A and B panels of at least one tile of rows
    // through buffer resources: a tile's rows must fit in 2 GiB
    constexpr uint64_t kLimit = 0x7FFFFFFFull;
    return (reinterpret_cast<uintptr_t>(g.a) % 16 == 0)
           && (reinterpret_cast<uintptr_t>(g.b) % 16 == 0) && (g.lda % 16 == 0)
           && (g.ldb % 16 == 0) && (g.k % 16 == 0)
           && (uint64_t)g.lda * GemmMain::kBM <= kLimit && (uint64_t)g.ldb * GemmMain::kBN <= kLimit;
}

bool gemm_packed_ok(const GemmArgs& g)
{
    constexpr uint64_t kLimit = 0x7FFFFFFFull;
    if(reinterpret_cast<uintptr_t>(g.a) % 16 != 0 || g.lda % 16 != 0 || g.k % 16 != 0) return false;
    // one packed k-row of a 64-row slab must fit in 2 GiB
    if((uint64_t)gemm::packed_ktiles(g.k) * gemm::kPackFrags * 1024 > kLimit) return false;
    return g.m <= kDecodeMaxM ? gemm_decode_ok(g) : (uint64_t)g.lda * GemmMain::kBM <= kLimit;
}

// The persistent tile kernel for a 256 x 256 launch: fp16 output, at least
// two tiles per CU and at most 32 k-tiles per tile.  It saves a fixed cost
// per tile (workgroup launch, cold prologue, store burst), which pays where
// tiles are short: 2-4% at M=8192 K=4096 N=28672, 10-20% at K <= 1024,
// nothing measurable at K=14336 with two tiles per CU.
template <class C>
bool persist_pays(const KArgs& p, int out_type)
{
    return out_type == W8A8_OUT_F16 && (p.k + C::kBK - 1) / C::kBK <= 32
           && gemm::persist_ok<C>(p, device_cus());
}

size_t gemm_nk_workspace_bytes(const GemmArgs& g)
{
    if(g.m == 0 || g.n == 0 || g.k == 0) return 0;
    return plan_tiles(g.m, g.n, g.k, kMaxPlanBytes, g.m <= kDecodeMaxM, false).bytes;
}

// The weights of rows [n0, ...) of a panel (packed: n0 a multiple of the slab).
template <bool PB>
const int8_t* weight_rows(const KArgs& p, uint32_t n0)
{
    return PB ? p.b + (size_t)(n0 / gemm::kSlab) * gemm::packed_ktiles(p.k) * gemm::kPackFrags * 1024
              : p.b + (size_t)n0 * p.ldb;
}

// One 256 x 256 launch (a panel).  When its tiles make whole rounds over the
// CUs plus a last round at most half full, and the whole rounds are whole
// columns of tiles, the columns of the last round run as 128 x 256 tiles in
// a launch of their own: twice the tiles, each half the work, so that round
// keeps every CU busy for about half as long (cfg3 gate_up at M = 2048:
// 8 x 112 tiles = 3 rounds + 128 tiles; the last 16 columns become one
// round of 256 tiles of 128 x 256).  The same k-order per output, so the
// result is bit-identical to the single launch.
template <bool PB>
hipError_t launch_main(const KArgs& p, int out_type, hipStream_t stream)
{
    using Main           = typename Tiles<PB>::Main;
    using MidM           = typename Tiles<PB>::MidM;
    const uint32_t cus   = device_cus();
    const uint32_t tm    = (p.m + Main::kBM - 1) / Main::kBM;
    const uint32_t tiles = tm * ((p.n + Main::kBN - 1) / Main::kBN);
    const uint32_t full = tiles / cus, rest = tiles % cus;
    const uint32_t mid_rows = (p.m + MidM::kBM - 1) / MidM::kBM;
    auto whole = [&](const KArgs& q) {
        return persist_pays<Main>(q, out_type)
                   ? gemm::launch_cfg_persist<Main>(q, cus, stream)
                   : gemm::launch_cfg<Main>(q, out_type, stream);
    };
    if(full >= 1 && rest > 0 && rest * 2 <= cus && (full * cus) % tm == 0) {
        const uint32_t n1   = full * cus / tm * Main::kBN; // < p.n: rest > 0
        const uint32_t n2   = p.n - n1;
        const size_t   esz  = out_type == W8A8_OUT_I32 ? 4 : 2;
        if((uint64_t)mid_rows * ((n2 + MidM::kBN - 1) / MidM::kBN) <= cus) {
            KArgs head = p, tail = p;
            head.n     = n1;
            tail.n     = n2;
            tail.b     = weight_rows<PB>(p, n1);
            tail.c     = static_cast<int8_t*>(p.c) + (size_t)n1 * esz;
            tail.sb    = p.sb ? p.sb + n1 : nullptr;
            hipError_t e = whole(head);
            if(e != hipSuccess) return e;
            return gemm::launch_cfg<MidM>(tail, out_type, stream);
        }
    }
    return whole(p);
}

// One planned launch of a panel.
template <bool PB>
hipError_t launch_plan(const KArgs& p, const TilePlan& d, int out_type, void* ws,
                       hipStream_t stream)
{
    using T = Tiles<PB>;
    auto go = [&](auto c) {
        using C = decltype(c);
        if(d.parts > 1)
            return gemm::launch_cfg_split<C>(p, out_type, static_cast<int32_t*>(ws),
                                             d.parts, stream);
        return gemm::launch_cfg<C>(p, out_type, stream);
    };
    switch(d.cfg) {
    case TileCfg::kMain:
        return d.parts > 1 ? go(typename T::Main{})
                           : launch_main<PB>(p, out_type, stream);
    case TileCfg::kMidM: return go(typename T::MidM{});
    case TileCfg::kSmall: return go(typename T::Small{});
    case TileCfg::kNarrow: return go(typename T::Narrow{});
    case TileCfg::kTiny: return go(typename T::Tiny{});
    default: return go(typename T::Row{});
    }
}

// The tile kernels over a whole problem, row-major (PB = false) or packed
// weights, in row and column panels where an operand exceeds 2 GiB.
template <bool PB>
hipError_t launch_tiles(const GemmArgs& g, void* ws, size_t ws_bytes, hipStream_t stream)
{
    const size_t esz    = g.out_type == W8A8_OUT_I32 ? 4 : 2;
    // The tile kernel addresses each operand through a buffer resource whose
    // out-of-range offsets read as zero; keep every launch's A and B under
    // 2 GiB by splitting M and N into row panels (multiples of the tile).
    constexpr size_t kLimit = 0x7FFFFFFFull;
    const uint32_t   mstep  = (uint32_t)std::min<size_t>(
        g.m, std::max<size_t>(GemmMain::kBM, kLimit / g.lda / GemmMain::kBM * GemmMain::kBM));
    // weight rows under 2 GiB: ldb bytes a row, or packed rows of whole k-tiles
    const size_t   row   = PB ? (size_t)gemm::packed_ktiles(g.k) * gemm::kPackK : g.ldb;
    const uint32_t nstep = (uint32_t)std::min<size_t>(
        g.n, std::max<size_t>(GemmMain::kBN, kLimit / row / GemmMain::kBN * GemmMain::kBN));
    for(uint32_t m0 = 0; m0 < g.m; m0 += mstep) {
        for(uint32_t n0 = 0; n0 < g.n; n0 += nstep) {
            KArgs p = make_kargs(g);
            p.m     = std::min(mstep, g.m - m0);
            p.n     = std::min(nstep, g.n - n0);
            p.a     = g.a + (size_t)m0 * g.lda;
            p.b     = weight_rows<PB>(p, n0);
            p.c     = static_cast<int8_t*>(g.c) + ((size_t)m0 * g.ldc + n0) * esz;
            p.sa    = g.scale_a ? g.scale_a + m0 : nullptr;
            p.sb    = g.scale_b ? g.scale_b + n0 : nullptr;
            // panels run in stream order, so they share the workspace
            const TilePlan   d = plan_tiles(p.m, p.n, p.k, ws ? ws_bytes : 0, false, PB);
            const hipError_t e = launch_plan<PB>(p, d, g.out_type, ws, stream);
            if(e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

hipError_t launch_gemm_nk(const GemmArgs& g, void* ws, size_t ws_bytes, hipStream_t stream)
{
    if(g.m == 0 || g.n == 0) return hipSuccess;
    if(gemm_decode_ok(g)
       && plan_tiles(g.m, g.n, g.k, ws ? ws_bytes : 0, true, false).cfg == TileCfg::kDecode)
        return launch_gemm_decode(g, false, nullptr, 0, stream);
    return launch_tiles<false>(g, ws, ws_bytes, stream);
}

// Packed weights: m <= 64 streams them through the decode kernels; larger m
// runs the row-major GEMM's tile kernels and rules over the packed layout.
// (A kernel that loaded B fragments straight to registers, 32 x 32 x 32 MFMA,
// no K split, was 5-10% slower at M = 8192 and far behind below: 300 x 6144 x
// 4096 24.0 -> 18.5 us, 1000 x 1024 x 26576 120 -> 94 us, 322 x 566 x 3936
// 50 -> 20 us, where it also cut N into two launches.)
hipError_t launch_gemm_packed(const GemmArgs& g, void* ws, size_t ws_bytes, hipStream_t stream)
{
    if(g.m == 0 || g.n == 0) return hipSuccess;
    if(gemm_decode_ok(g)) return launch_gemm_decode(g, true, ws, ws_bytes, stream);
    return launch_tiles<true>(g, ws, ws_bytes, stream);
}

namespace {

// Explicit stream-K (w8a8_gemm_streamk): every tile of the problem in the
// stream-K schedule over `blocks` blocks (0: one per CU), the reference
// sample's decomposition (rocwmma_streamk_gemm.cpp:223-226).  The tile is
// the largest of 256 x 256, 128 x 256 and 128 x 128 that leaves each block
// at least 8 k-tiles (else 128 x 128); never more blocks than k-tiles.
struct ExplicitSk {
    TileCfg      cfg;
    gemm::SkPlan plan;
    size_t       bytes;
};

// Estimated critical path of a stream-K plan on tile configuration C: the
// longest block's k-tiles at C's rate per CU (`tops`, whole chip, measured on
// the dense kernels: the smaller tiles sustain less), plus the partials the
// last piece of the most-split tile reads back at `xbw` bytes/s (device-scope
// loads; fitted to the square and cfg3 CLI shapes, lower for the larger
// tiles, whose kernels spill around the exchange).  Splitting a tile over P
// blocks costs its last block P - 1 partials, so fewer, larger tiles win
// only where their pieces stay few: 2048^3 ran 75 µs on 256 x 256 tiles (4
// pieces each) against 26 µs on 128 x 128 tiles (one block per tile).
template <class C>
double sk_cost(const gemm::SkPlan& s, double tops, double xbw)
{
    const uint64_t u    = (s.total() + s.blocks - 1) / s.blocks;
    const uint32_t pmax = s.max_pieces();
    const double unit_s = 2.0 * C::kBM * C::kBN * C::kBK / (tops / device_cus());
    return (double)u * unit_s + (pmax - 1) * (double)gemm::Partial<C>::kBytes / xbw;
}

// blocks = 0: the block count is chosen too, among one per CU and 1/2, 1/4,
// 1/8 of that: a few tiles cut into many pieces cost their last blocks more
// partials than the extra blocks save (512^3: 16 pieces per tile on 256
// blocks, 4 on 64).
ExplicitSk plan_streamk(uint32_t m, uint32_t n, uint32_t k, uint32_t blocks)
{
    const uint32_t nk = (k + 127) / 128;
    ExplicitSk     e{TileCfg::kMain, {}, 0};
    double         best = 1e300;
    for(uint32_t div = 1; div <= (blocks ? 1u : 8u); div *= 2) {
        const uint32_t G = blocks ? blocks : std::max(1u, device_cus() / div);
        auto plan = [&](uint32_t bm, uint32_t bn) {
            const uint32_t tiles = ((m + bm - 1) / bm) * ((n + bn - 1) / bn);
            return gemm::SkPlan{nk, tiles, (uint32_t)std::min<uint64_t>(G, (uint64_t)tiles * nk)};
        };
        const ExplicitSk cand[3] = {
            {TileCfg::kMain, plan(GemmMain::kBM, GemmMain::kBN), 0},
            {TileCfg::kMidM, plan(GemmMidM::kBM, GemmMidM::kBN), 0},
            {TileCfg::kSmall, plan(GemmSmall::kBM, GemmSmall::kBN), 0}};
        const double cost[3] = {sk_cost<GemmMain>(cand[0].plan, 2.5e15, 13e9),
                                sk_cost<GemmMidM>(cand[1].plan, 2.1e15, 15e9),
                                sk_cost<GemmSmall>(cand[2].plan, 1.7e15, 35e9)};
        for(int c = 0; c < 3; ++c)
            if(cost[c] < best * (1 - 1e-9)) {
                best = cost[c];
                e    = cand[c];
            }
    }
    e.bytes = e.cfg == TileCfg::kMain   ? gemm::sk_workspace_bytes<GemmMain>(e.plan)
              : e.cfg == TileCfg::kMidM ? gemm::sk_workspace_bytes<GemmMidM>(e.plan)
                                        : gemm::sk_workspace_bytes<GemmSmall>(e.plan);
    return e;
}

// plan_streamk memoized per (m, n, k, blocks): every w8a8_gemm_streamk call
// needs the plan twice (the workspace check, then the launch) and a caller
// sizing its workspace a third time; the plan depends on nothing else (the CU
// count is the process's first device's).  The table is bounded: a caller
// cycling through more shapes than kMaxPlans starts it over.
ExplicitSk explicit_streamk(uint32_t m, uint32_t n, uint32_t k, uint32_t blocks)
{
    constexpr size_t kMaxPlans = 1024;
    struct Key {
        uint32_t m, n, k, blocks;
        bool     operator<(const Key& o) const
        {
            return std::tie(m, n, k, blocks) < std::tie(o.m, o.n, o.k, o.blocks);
        }
    };
    static std::mutex               mu;
    static std::map<Key, ExplicitSk> plans;
    const Key                        key{m, n, k, blocks};
    {
        std::lock_guard<std::mutex> lock(mu);
        const auto                  it = plans.find(key);
        if(it != plans.end()) return it->second;
    }
    const ExplicitSk e = plan_streamk(m, n, k, blocks);
    std::lock_guard<std::mutex> lock(mu);
    if(plans.size() >= kMaxPlans) plans.clear();
    plans.emplace(key, e);
    return e;
}

} // namespace

bool streamk_shape_ok(const GemmArgs& g)
{
    constexpr uint64_t kLimit = 0x7FFFFFFFull;
    return gemm_fast_path_ok(g) && (uint64_t)g.m * g.lda <= kLimit
           && (uint64_t)g.n * g.ldb <= kLimit;
}

size_t streamk_workspace_bytes(uint32_t m, uint32_t n, uint32_t k, uint32_t blocks)
{
    if(m == 0 || n == 0 || k == 0) return 0;
    return explicit_streamk(m, n, k, blocks).bytes;
}

uint32_t streamk_blocks(uint32_t m, uint32_t n, uint32_t k, uint32_t blocks)
{
    if(m == 0 || n == 0 || k == 0) return 0;
    return explicit_streamk(m, n, k, blocks).plan.blocks;
}

// ---------------------------------------------------------------------------
// The stream-K wait's status word (gemm::SkWatch): one per GPU, a file-scope
// device array like the no-allocation scratch below, reached from the host
// only through the address hipGetSymbolAddress returns for the current
// device.  Zero-initialised when the code object loads; a kernel only ORs
// bits into it; streamk_status reads (and optionally clears) it.
// ---------------------------------------------------------------------------
static __device__ __align__(256) uint32_t sk_status[64];

namespace {

hipError_t sk_status_ptr(uint32_t** ptr)
{
    constexpr int     kMaxDevices = 64;
    static std::mutex mu;
    static void*      addr[kMaxDevices] = {};
    int               dev               = 0;
    hipError_t        e                 = hipGetDevice(&dev);
    if(e != hipSuccess) return e;
    if(dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if(addr[dev] == nullptr) {
        void* p = nullptr;
        e       = hipGetSymbolAddress(&p, HIP_SYMBOL(sk_status));
        if(e != hipSuccess) return e;
        addr[dev] = p;
    }
    *ptr = static_cast<uint32_t*>(addr[dev]);
    return hipSuccess;
}

// the wait's poll limit and phantom piece count (test hook only)
std::atomic<uint32_t> g_sk_spin{gemm::kSkSpinLimit};
std::atomic<uint32_t> g_sk_phantom{0};

} // namespace

void streamk_debug_wait(uint32_t spin, uint32_t phantom)
{
    g_sk_spin.store(spin ? spin : gemm::kSkSpinLimit);
    g_sk_phantom.store(phantom);
}

hipError_t streamk_status(uint32_t* flags, bool clear)
{
    uint32_t*  ptr = nullptr;
    hipError_t e   = sk_status_ptr(&ptr);
    if(e != hipSuccess) return e;
    // every launch that may set the word has finished, on any stream
    if((e = hipDeviceSynchronize()) != hipSuccess) return e;
    if((e = hipMemcpy(flags, ptr, sizeof(uint32_t), hipMemcpyDeviceToHost)) != hipSuccess) return e;
    if(clear && *flags) {
        const uint32_t zero = 0;
        e = hipMemcpy(ptr, &zero, sizeof(uint32_t), hipMemcpyHostToDevice);
    }
    return e;
}

hipError_t launch_gemm_streamk(const GemmArgs& g, uint32_t blocks, void* ws, hipStream_t stream)
{
    if(g.m == 0 || g.n == 0) return hipSuccess;
    gemm::SkWatch watch{nullptr, g_sk_spin.load(), g_sk_phantom.load()};
    const hipError_t err = sk_status_ptr(&watch.status);
    if(err != hipSuccess) return err;
    const ExplicitSk e      = explicit_streamk(g.m, g.n, g.k, blocks);
    const KArgs      p      = make_kargs(g);
    if(e.plan.blocks == e.plan.ntiles) {
        // one whole tile per block, no pieces: the schedule is the tile
        // kernel's one-block-per-tile grid (the same logical block -> tile
        // order), which runs it without the counters' clear launch and with
        // the epilogue's scales loaded under the last k-tile
        switch(e.cfg) {
        case TileCfg::kMain: return gemm::launch_cfg<GemmMain>(p, g.out_type, stream);
        case TileCfg::kMidM: return gemm::launch_cfg<GemmMidM>(p, g.out_type, stream);
        default: return gemm::launch_cfg<GemmSmall>(p, g.out_type, stream);
        }
    }
    switch(e.cfg) {
    case TileCfg::kMain:
        return gemm::launch_cfg_streamk<GemmMain>(p, g.out_type, 0, e.plan, ws, watch,
                                                  stream);
    case TileCfg::kMidM:
        return gemm::launch_cfg_streamk<GemmMidM>(p, g.out_type, 0, e.plan, ws, watch,
                                                  stream);
    default:
        return gemm::launch_cfg_streamk<GemmSmall>(p, g.out_type, 0, e.plan, ws, watch,
                                                   stream);
    }
}

hipError_t launch_gemm_generic(const GemmArgs& g, size_t sam, size_t sak, size_t sbn, size_t sbk,
                               hipStream_t stream)
{
    if(g.m == 0 || g.n == 0) return hipSuccess;
    const KArgs p = make_kargs(g);
    dim3        grid((g.n + 15) / 16, (g.m + 15) / 16);
    if(g.out_type == W8A8_OUT_I32)
        hipLaunchKernelGGL(gemm_i8_generic_kernel<W8A8_OUT_I32>, grid, dim3(256), 0, stream, p,
                           sam, sak, sbn, sbk);
    else
        hipLaunchKernelGGL(gemm_i8_generic_kernel<W8A8_OUT_F16>, grid, dim3(256), 0, stream, p,
                           sam, sak, sbn, sbk);
    return hipGetLastError();
}

hipError_t launch_repack_kn(const GemmArgs& g, int8_t* at, int8_t* bt, uint32_t kp,
                            hipStream_t stream)
{
    const Repack   a{g.a, at, g.lda, g.m}, b{g.b, bt, g.ldb, g.n};
    const uint32_t kt = (kp + 127) / 128;
    const uint64_t na = (uint64_t)ceil_div(g.m, 128) * kt, nb = (uint64_t)ceil_div(g.n, 128) * kt;
    if(na + nb > 0x7FFFFFFFull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(repack_i8_kernel, dim3((uint32_t)(na + nb)), dim3(256), 0, stream, a, b,
                       (uint32_t)na, g.k, kp);
    return hipGetLastError();
}

// Tiles of the direct kernel: 256 x 256 and 128 x 128 from 5/8 of a round of
// them on, else 64 x 64.  4000 x 4000 x 4001 (256 / 1024 / 3969 tiles) 84 /
// 113 / 212 us; 3000^3 (144 of 256 x 256) 65 / 65; 2000^3 (256 of 128 x 128)
// 45 / 21 / 30; 847 x 2388 x 92 (133 of 128 x 128) 19 / 10.9 / 10.2; 1000^3
// 22 / 9.5 / 7.9.  The sample layout's lie alike: 4095^3 149 / 221 / 407,
// 2000^3 53 / 25 / 36, 912 x 563 x 2138 (40 of 128 x 128) 64 / 28 / 21.
uint32_t direct_tile(uint32_t m, uint32_t n)
{
    const uint64_t enough = (uint64_t)device_cus() * 5 / 8;
    for(uint32_t b : {256u, 128u})
        if((uint64_t)ceil_div(m, b) * ceil_div(n, b) >= enough) return b;
    return 64;
}

template <bool COLS>
hipError_t launch_direct_tiles(const GemmArgs& g, hipStream_t stream)
{
    if(g.m == 0 || g.n == 0) return hipSuccess;
    using Big    = gemm::Cfg<256, 256, 128, 2, 2, 4, 4, 16>;
    using Middle = gemm::Cfg<128, 128, 128, 2, 2, 4, 4, 16>;
    using Little = gemm::Cfg<64, 64, 128, 2, 2, 2, 4, 16>;
    constexpr int  kAhead = COLS ? 1 : 2; // k-tiles in registers (a quad unit is 16 VGPRs)
    const KArgs    p      = make_kargs(g);
    if((uint64_t)ceil_div(g.m, 64) * ceil_div(g.n, 64) > 0x7FFFFFFFull) return hipErrorInvalidValue;
    switch(direct_tile(g.m, g.n)) {
    case 256: return gemm::launch_direct<Big, COLS, 1>(p, g.out_type, stream);
    case 128: return gemm::launch_direct<Middle, COLS, kAhead>(p, g.out_type, stream);
    default: return gemm::launch_direct<Little, COLS, kAhead>(p, g.out_type, stream);
    }
}

hipError_t launch_gemm_direct(const GemmArgs& g, bool kn, hipStream_t stream)
{
    return kn ? launch_direct_tiles<true>(g, stream) : launch_direct_tiles<false>(g, stream);
}

// Primary layout, K below 32: a tile's k-step is mostly zeros, loaded byte by byte
// below 16, and one output per thread is done sooner while there are few products.
// Microseconds of either, fitted to 110 sizes: 300 x 300 x 9 3.3 against 7.4, 640 x 640
// x 13 6.4 / 8.4, 1000 x 1000 x 9 8.7 / 7.5, 1500 x 900 x 3 6.5 / 5.7, 55 x 1307 x 17
// 3.8 / 4.6, 100 x 1000 x 25 5.2 / 4.5.  The sample layout in place, whose tiles load
// quads of either operand: 120 sizes, 218 x 252 x 1 3.1 / 4.4, 123 x 75 x 14 3.9 / 4.3,
// 557 x 1018 x 12 5.8 / 4.5, 12 x 755 x 30 5.3 / 4.2.
bool generic_pays(const GemmArgs& g, bool kn)
{
    const double k = g.k, outputs = (double)g.m * g.n;
    if(g.k >= 32 || ceil_div(g.m, 16) > 65535) return false; // its grid's rows
    if(kn) return 2.8 + 0.07 * k + 1e-6 * outputs * (1.0 + 0.15 * k) < 4.25;
    return 2.6 + 0.05 * k + 1e-6 * outputs * (1.7 + 0.47 * k) < 4.4 + (g.k < 16 ? 0.33 * k : 0.0);
}

bool gemm_direct_kn_ok(const GemmArgs& g) { return g.m >= 4 && g.n >= 4; }

// The sample layout in place, where it beats the repack and its second
// launch: a direct k-tile costs about 1 us, so up to 8 of them in one round
// of 64 x 64 tiles (130 x 2767 x 996: 11.7 us against 17.7 with the repack;
// 186 x 1044 x 3394, 27 k-tiles: 28.8 against 25.7).
bool direct_kn_pays(const GemmArgs& g)
{
    return gemm_direct_kn_ok(g)
           && (uint64_t)ceil_div(g.m, 64) * ceil_div(g.n, 64) <= device_cus()
           && ceil_div(g.k, 128) <= 8;
}

// ---------------------------------------------------------------------------
// Scratch of w8a8_gemm_noalloc: a file-scope device array.  Every GPU that
// loads this code object holds its own copy until the process ends; host code
// uses it only through the device address hipGetSymbolAddress returns, looked
// up once per device with that device current (the array's name is a host
// stand-in, not a device address).  The K-split partials that live in it are
// written in full before they are read, so nothing is cleared between calls;
// calls that overlap on one GPU share the array and race.
// ---------------------------------------------------------------------------
static __device__ __align__(256) int8_t scratch[W8A8_NOALLOC_SCRATCH_BYTES];

hipError_t noalloc_scratch(void** ptr)
{
    constexpr int      kMaxDevices = 64;
    static std::mutex  mu;
    static void*       addr[kMaxDevices] = {};
    int                dev               = 0;
    hipError_t         e                 = hipGetDevice(&dev);
    if(e != hipSuccess) return e;
    if(dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if(addr[dev] == nullptr) {
        void* p = nullptr;
        e       = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if(e != hipSuccess) return e;
        addr[dev] = p;
    }
    *ptr = addr[dev];
    return hipSuccess;
}

} // namespace w8a8
