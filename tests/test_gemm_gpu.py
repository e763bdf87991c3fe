"""GPU parity of the int8 GEMM: int32 accumulators bit-exact against the
oracle (gemm_cpu_h semantics), fp16 dequant bit-exact against the oracle's
epilogue (and within the 1e-2 rel / 1e-3 abs tolerance the path requires),
for the fast kernel, its edge handling, the generic kernel and the sample
(A col-major / B [K,N]) layout."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from checks import assert_f16_bitexact, assert_i32_equal, dev, host, plan
from optimized_rocwmma_samples_amd import _lib as L
from optimized_rocwmma_samples_amd import datagen as G

pytestmark = pytest.mark.gpu


def inputs(m, n, k, seed):
    a = G.int8(seed, G.TID_A, (m, k))
    b = G.int8(seed, G.TID_B, (n, k))
    sa = G.uniform(seed, G.TID_SA, (m,), 1e-3, 1e-2)
    sb = G.uniform(seed, G.TID_SB, (n,), 1e-3, 1e-2)
    return a, b, sa, sb


SHAPES = [
    (256, 256, 64), (512, 512, 512), (1, 1, 16), (300, 200, 80), (257, 513, 144),
    (100, 1000, 4096), (256, 256, 48), (384, 640, 4112), (33, 4096, 1024), (4096, 64, 256),
    (1000, 1000, 1000),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_int32_exact(w8a8, gpu, m, n, k):
    import torch
    a, b, _, _ = inputs(m, n, k, m * 7 + n * 3 + k)
    c = w8a8.gemm(dev(a, gpu), dev(b, gpu), out_dtype=torch.int32)
    assert_i32_equal(host(c), O.gemm_i32(a, b))


@pytest.mark.parametrize("m,n,k", [(512, 768, 512), (300, 200, 80), (64, 4096, 4096)])
def test_f16_dequant_mode2(w8a8, gpu, m, n, k):
    a, b, sa, sb = inputs(m, n, k, 17 + m)
    c = w8a8.gemm(dev(a, gpu), dev(b, gpu), dev(sa, gpu), dev(sb, gpu))
    assert_f16_bitexact(host(c), O.dequant_f16(O.gemm_i32(a, b), sa, sb))


# Every tile of the plan (rows x columns; 0 x 32: the decode kernel), unsplit, with
# partial tiles on both edges and a K tail; the last eight with odd rows of C.
TILE_CFG_SHAPES = [
    (4100, 3000, 160, (256, 256)), (2048, 4096, 512, (128, 256)), (1500, 4000, 272, (128, 256)),
    (700, 1100, 400, (64, 64)), (2, 107, 144, (0, 32)), (3, 373, 3520, (32, 64)),
    (90, 123, 144, (64, 64)), (771, 1051, 144, (64, 64)), (549, 2785, 240, (64, 128)),
    (713, 2883, 656, (128, 128)), (1746, 4227, 688, (128, 256)), (1497, 8675, 400, (256, 256)),
]


def unsplit_tile(w8a8, m, n, k, packed=False):
    kind = L.PLAN_GEMM_PACKED if packed else L.PLAN_GEMM
    rows, cols, pieces = plan(w8a8, kind, m, n, k, 64 << 20)
    assert pieces == 1
    return rows, cols


@pytest.mark.parametrize("m,n,k,tile", TILE_CFG_SHAPES)
def test_tile_configs_exact(w8a8, gpu, m, n, k, tile):
    import torch
    assert unsplit_tile(w8a8, m, n, k) == tile
    a, b, sa, sb = inputs(m, n, k, m + 3 * n + 5 * k)
    ad, bd = dev(a, gpu), dev(b, gpu)
    acc = O.gemm_i32(a, b)
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32)), acc)
    c = w8a8.gemm(ad, bd, dev(sa, gpu), dev(sb, gpu))
    assert_f16_bitexact(host(c), O.dequant_f16(acc, sa, sb))


# 256 x 256 launches of whole rounds plus a last round at most half full,
# whose whole rounds are whole tile columns: the last round's columns run as
# 128 x 256 tiles in a second launch (tile counts for 256 CUs).
COLUMN_TAIL_SHAPES = [
    (2048, 28672, 256),  # 8 x 112 tiles = 3 rounds + 128: columns 24576.. as 16 x 16 tiles
    (2000, 17000, 272),  # 8 x 67 = 2 rounds + 24, ragged edges, a K tail: columns 16384..
]


@pytest.mark.parametrize("m,n,k", COLUMN_TAIL_SHAPES)
def test_column_tail_exact(w8a8, gpu, m, n, k):
    import torch
    a, b, sa, sb = inputs(m, n, k, m + n + k)
    ad, bd = dev(a, gpu), dev(b, gpu)
    acc = O.gemm_i32(a, b)
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32)), acc)
    c = w8a8.gemm(ad, bd, dev(sa, gpu), dev(sb, gpu))
    assert_f16_bitexact(host(c), O.dequant_f16(acc, sa, sb))


# Launches of at least two 256 x 256 tiles per CU with K <= 4096 and an fp16
# output run the persistent kernel: one block per CU walks its tiles, the
# stage ring runs across tile boundaries and each tile's epilogue stores stay
# in flight into the next tile.  Tile counts are for a 256-CU device.
PERSIST_SHAPES = [
    (4100, 8200, 160),   # 561 tiles, ragged edges, 2 k-tiles (K tail)
    (8192, 8192, 128),   # 1024 tiles, one k-tile per tile
    (4096, 8200, 2000),  # 528 tiles, 16 k-tiles (K tail)
    (8192, 16400, 128),  # 2080 tiles, a 269 MB output (over the 256 MB MALL): non-temporal stores
]


@pytest.mark.parametrize("m,n,k", PERSIST_SHAPES)
def test_persistent_tiles_exact(w8a8, gpu, m, n, k):
    a, b, sa, sb = inputs(m, n, k, 7 * m + n + 3 * k)
    ad, bd = dev(a, gpu), dev(b, gpu)
    acc = O.gemm_i32(a, b)
    c = w8a8.gemm(ad, bd, dev(sa, gpu), dev(sb, gpu))
    assert_f16_bitexact(host(c), O.dequant_f16(acc, sa, sb))
    c1 = w8a8.gemm(ad, bd, tensor_scale_a=0.5, tensor_scale_b=0.25)
    assert_f16_bitexact(host(c1), O.dequant_f16(acc, tsa=0.5, tsb=0.25))


def test_persistent_tiles_strided_output(w8a8, gpu):
    # the persistent kernel's stores into rows of ldc > n: columns past n keep
    # what they held (every store past the matrix is dropped)
    import torch
    m, n, k, ldc = 4100, 8200, 160, 8208
    a, b, sa, sb = inputs(m, n, k, 99)
    big = torch.full((m, ldc), 7.0, dtype=torch.float16, device=gpu)
    w8a8.gemm(dev(a, gpu), dev(b, gpu), dev(sa, gpu), dev(sb, gpu), out=big[:, :n])
    hb = host(big)
    assert_f16_bitexact(np.ascontiguousarray(hb[:, :n]), O.dequant_f16(O.gemm_i32(a, b), sa, sb))
    assert (hb[:, n:] == 7.0).all()


# The K split (workspace given) of every tile, tile rows x columns: ragged edges, odd
# rows of C, a K tail in the last piece.
SPLIT_SHAPES = [
    (10, 107, 4128, (32, 64)), (64, 1000, 8208, (32, 64)), (83, 107, 4176, (64, 64)),
    (257, 851, 7104, (64, 64)), (300, 600, 8192, (64, 64)), (512, 512, 16384, (64, 128)),
    (305, 1097, 9744, (64, 128)),
    (204, 2739, 8512, (128, 128)), (512, 4096, 14336, (128, 128)),
    (1200, 1067, 21200, (128, 256)), (2062, 2099, 15296, (256, 256)),
]


@pytest.mark.parametrize("m,n,k,tile", SPLIT_SHAPES)
def test_k_split_exact(w8a8, gpu, m, n, k, tile):
    import torch
    size = w8a8.gemm_workspace_size(m, n, k)
    split = plan(w8a8, L.PLAN_GEMM, m, n, k, size)
    assert split[:2] == tile and split[2] > 1 and plan(w8a8, L.PLAN_GEMM, m, n, k, 0)[2] == 1
    a, b, sa, sb = inputs(m, n, k, 2 * m + n + k)
    ad, bd, sad, sbd = dev(a, gpu), dev(b, gpu), dev(sa, gpu), dev(sb, gpu)
    none = torch.empty(0, dtype=torch.uint8, device=gpu)
    ci = host(w8a8.gemm(ad, bd, out_dtype=torch.int32))           # split (workspace allocated)
    cf = host(w8a8.gemm(ad, bd, sad, sbd))
    assert_i32_equal(ci, host(w8a8.gemm(ad, bd, out_dtype=torch.int32, workspace=none)))
    assert_f16_bitexact(cf, host(w8a8.gemm(ad, bd, sad, sbd, workspace=none)))
    rows = np.unique(np.concatenate([np.arange(min(m, 16)), np.arange(max(0, m - 16), m),
                                     np.random.default_rng(m).integers(0, m, 64)]))
    acc = O.gemm_i32(a[rows], b)
    assert_i32_equal(ci[rows], acc)
    assert_f16_bitexact(cf[rows], O.dequant_f16(acc, sa[rows], sb))
    if m > 64:
        assert plan(w8a8, L.PLAN_GEMM_PACKED, m, n, k, size)[2] > 1
        pw = w8a8.pack_weights(bd)
        ws = torch.empty(size, dtype=torch.uint8, device=gpu)
        assert_i32_equal(host(w8a8.gemm_packed(ad, pw, out_dtype=torch.int32, workspace=ws)), ci)
        assert_f16_bitexact(host(w8a8.gemm_packed(ad, pw, sad, sbd, workspace=ws)), cf)


# Outputs at odd rows and addresses, channel scales 4 bytes off: 16-byte accesses of
# interior tiles, and the elements around the matrix untouched, for each tile over
# row-major and packed weights and the decode kernels.
@pytest.mark.parametrize("m,n,k,tile", [
    (4100, 3001, 160, (256, 256)), (990, 1621, 368, (64, 128)), (100, 1003, 1040, (64, 64)),
    (40, 515, 400, (0, 32)), (3, 77, 64, (0, 32)), (3, 373, 3520, (32, 64)),
    (713, 2883, 656, (128, 128)), (1746, 4227, 688, (128, 256)), (1497, 8675, 400, (256, 256))])
def test_unaligned_outputs_exact(w8a8, gpu, m, n, k, tile):
    assert unsplit_tile(w8a8, m, n, k) == tile
    assert m <= 64 or unsplit_tile(w8a8, m, n, k, packed=True) == tile
    import torch
    a, b, sa, sb = inputs(m, n, k, m + 2 * n + k)
    ad, bd = dev(a, gpu), dev(b, gpu)
    sbd = torch.empty(n + 1, dtype=torch.float32, device=gpu)[1:].copy_(dev(sb, gpu))
    pw = w8a8.pack_weights(bd)
    acc = O.gemm_i32(a, b)
    want = O.dequant_f16(acc, sa, sb)
    for packed in (False, True):
        for dt in (torch.float16, torch.int32):
            buf = torch.full((m * (n + 2) + 1,), 7, dtype=dt, device=gpu)
            out = buf[1:].view(m, n + 2)[:, :n]
            sc = (dev(sa, gpu), sbd) if dt == torch.float16 else (None, None)
            if packed:
                w8a8.gemm_packed(ad, pw, *sc, out=out)
            else:
                w8a8.gemm(ad, bd, *sc, out=out)
            got = host(buf)
            assert got[0] == 7 and (got[1:].reshape(m, n + 2)[:, n:] == 7).all()
            got = np.ascontiguousarray(got[1:].reshape(m, n + 2)[:, :n])
            assert_f16_bitexact(got, want) if dt == torch.float16 else assert_i32_equal(got, acc)


# Any pointer, row stride and K: tails of 1, 15 and 16 bytes either side of a
# k-tile, single rows and columns, K below 16, operands 1-7 bytes off alignment, in
# the generic kernel (tile 0) and each tile of the direct kernel (64, 128 and 256
# rows), one k-tile and several (the register ring's refills and both LDS stages).
DIRECT_SHAPES = [(1, 1, 1, 0), (3, 5, 15, 0), (65, 63, 17, 0), (900, 1050, 11, 64),
                 (300, 290, 31, 64), (64, 129, 127, 64), (130, 66, 129, 64), (200, 100, 255, 64),
                 (1, 300, 1001, 64), (300, 200, 641, 64), (1700, 1650, 100, 128),
                 (1700, 1650, 257, 128), (1650, 1700, 529, 128), (3400, 3330, 33, 256),
                 (3400, 3330, 385, 256), (3330, 3400, 527, 256)]


def _at_offset(a, ld, off, gpu):
    import torch
    buf = torch.full((a.shape[0] * ld + off,), 77, dtype=torch.int8, device=gpu)
    view = buf[off:].view(a.shape[0], ld)[:, :a.shape[1]]
    view.copy_(dev(a, gpu))
    return view


@pytest.mark.parametrize("pad,off", [(0, 0), (1, 3), (16, 8)])
@pytest.mark.parametrize("m,n,k,tile", DIRECT_SHAPES)
def test_any_alignment_exact(w8a8, gpu, m, n, k, tile, pad, off):
    import torch
    assert plan(w8a8, L.PLAN_GEMM_ANY, m, n, k) == (tile, tile, 1)
    a, b, sa, sb = inputs(m, n, k, 3 * m + 5 * n + k)
    ad, bd = _at_offset(a, k + pad, off, gpu), _at_offset(b, k + pad, off + 4, gpu)
    acc = O.gemm_i32(a, b)
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32)), acc)
    assert_f16_bitexact(host(w8a8.gemm(ad, bd, dev(sa, gpu), dev(sb, gpu))),
                        O.dequant_f16(acc, sa, sb))


# The sample layout: in place (few products of a short K one per thread; few tiles,
# short K), repacked (with and without
# the room for 128-byte rows), in place for want of a workspace (each tile size,
# several k-tiles and a tail), and 1-3 rows or columns, each with ragged sizes and
# leading dimensions.
@pytest.mark.parametrize("m,n,k", [(4, 4, 1), (130, 767, 996), (186, 1044, 1394), (2, 300, 200),
                                   (300, 3, 77), (700, 900, 2051), (1, 1, 5), (1700, 1650, 403),
                                   (3330, 3400, 527), (123, 75, 14), (5, 6, 31),
                                   (3, 2, 1466)])
def test_sample_layout_routes_exact(w8a8, gpu, m, n, k):
    import torch
    a, b, _, _ = inputs(m, n, k, m + 7 * n + 3 * k)
    at = _at_offset(np.ascontiguousarray(a.T), m + 1, 3, gpu)
    bt = _at_offset(np.ascontiguousarray(b.T), n + 5, 1, gpu)
    acc = O.gemm_i32(a, b)
    full = w8a8.gemm_workspace_size(m, n, k, w8a8.LAYOUT_A_COL_B_KN)
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    kp = (k + 15) // 16 * 16
    for size in (full, up(m * kp) + up(n * kp), 0):
        ws = torch.empty(size, dtype=torch.uint8, device=gpu)
        c = w8a8.gemm(at, bt, layout=w8a8.LAYOUT_A_COL_B_KN, out_dtype=torch.int32, workspace=ws,
                      m=m, n=n, k=k)
        assert_i32_equal(host(c), acc)


# More rows than one output per thread has a grid for, with and without the room to
# repack: K below 32 and few products all the same.
@pytest.mark.parametrize("m,n", [(1100000, 1), (1048560, 1)])
def test_sample_layout_of_very_many_rows(w8a8, gpu, m, n):
    import torch
    a, b, _, _ = inputs(m, n, 1, 5)
    at = _at_offset(np.ascontiguousarray(a.T), m + 1, 0, gpu)
    bt = _at_offset(np.ascontiguousarray(b.T), n + 1, 0, gpu)
    c = w8a8.gemm(at, bt, layout=w8a8.LAYOUT_A_COL_B_KN, out_dtype=torch.int32)
    assert_i32_equal(host(c), O.gemm_i32(a, b))
    prim = w8a8.gemm(_at_offset(a, 1, 0, gpu), _at_offset(b, 1, 0, gpu), out_dtype=torch.int32)
    assert_i32_equal(host(prim), O.gemm_i32(a, b))


# The short tiles (several blocks a CU) and their K pieces, row-major and packed
# weights: edges of 32 / 64 rows and 64 / 128 columns, K tails, one k-tile.
SHORT_TILE_SHAPES = [
    (1, 5000, 4096, (32, 64, 3)), (33, 4104, 2064, (32, 64, 1)),
    (31, 520, 17152, (32, 64, 8)), (64, 1000, 8208, (32, 64, 7)),
    (65, 4096, 16, (64, 64, 1)), (191, 1001, 1040, (64, 64, 1)),
    (70, 512, 17072, (64, 64, 8)), (226, 380, 12224, (64, 64, 8)),
    (549, 2785, 240, (64, 128, 1)), (418, 885, 9152, (64, 128, 5)), (512, 4096, 2048, (64, 128, 1)),
]


@pytest.mark.parametrize("m,n,k,kernel", SHORT_TILE_SHAPES)
def test_short_tiles_exact(w8a8, gpu, m, n, k, kernel):
    import torch
    assert plan(w8a8, L.PLAN_GEMM, m, n, k, w8a8.gemm_workspace_size(m, n, k)) == kernel
    a, b, sa, sb = inputs(m, n, k, 11 * m + n + k)
    ad, bd, sad, sbd = dev(a, gpu), dev(b, gpu), dev(sa, gpu), dev(sb, gpu)
    pw = w8a8.pack_weights(bd)
    none = torch.empty(0, dtype=torch.uint8, device=gpu)
    acc = O.gemm_i32(a, b)
    want = O.dequant_f16(acc, sa, sb)
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32)), acc)
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32, workspace=none)), acc)
    assert_i32_equal(host(w8a8.gemm_packed(ad, pw, out_dtype=torch.int32)), acc)
    assert_f16_bitexact(host(w8a8.gemm(ad, bd, sad, sbd)), want)
    assert_f16_bitexact(host(w8a8.gemm_packed(ad, pw, sad, sbd)), want)


# Few rows of many columns (more than two rounds of 256 x 256 tiles): short tiles.
@pytest.mark.parametrize("m,n,k", [(3, 131100, 160), (100, 131100, 144), (257, 66001, 512)])
def test_few_rows_of_many_columns_exact(w8a8, gpu, m, n, k):
    import torch
    a, b, sa, sb = inputs(m, n, k, m + n + k)
    ad, bd = dev(a, gpu), dev(b, gpu)
    acc = O.gemm_i32(a, b)
    assert plan(w8a8, L.PLAN_GEMM, m, n, k, w8a8.gemm_workspace_size(m, n, k))[0] < 256
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32)), acc)
    if m > 64:
        assert plan(w8a8, L.PLAN_GEMM_PACKED, m, n, k, 0)[0] < 256
        c = w8a8.gemm_packed(ad, w8a8.pack_weights(bd), dev(sa, gpu), dev(sb, gpu))
        assert_f16_bitexact(host(c), O.dequant_f16(acc, sa, sb))


def test_k_split_strided(w8a8, gpu):
    # split path with row strides on A, B and C (64 tiles of 64 x 64 x 4 pieces)
    import torch
    m, n, k = 256, 1024, 4096
    assert plan(w8a8, L.PLAN_GEMM, m, n, k, w8a8.gemm_workspace_size(m, n, k)) == (64, 64, 4)
    a, b, sa, sb = inputs(m, n, k + 32, 77)
    ad = dev(a, gpu)[:, :k]
    bd = dev(b, gpu)[:, :k]
    acc = O.gemm_i32(a[:, :k], b[:, :k])
    for dt in (torch.int32, torch.float16):
        big = torch.full((m, n + 8), -3, dtype=dt, device=gpu)
        w8a8.gemm(ad, bd, dev(sa, gpu) if dt == torch.float16 else None,
                  dev(sb, gpu) if dt == torch.float16 else None, out=big[:, :n])
        got = host(big)
        if dt == torch.int32:
            assert_i32_equal(got[:, :n], acc)
        else:
            assert_f16_bitexact(np.ascontiguousarray(got[:, :n]), O.dequant_f16(acc, sa, sb))
        assert (got[:, n:] == -3).all()


def test_f16_dequant_mode1_tensor_scales(w8a8, gpu):
    m, n, k = 256, 512, 256
    a, b, _, _ = inputs(m, n, k, 5)
    c = w8a8.gemm(dev(a, gpu), dev(b, gpu), tensor_scale_a=1 / 127, tensor_scale_b=1 / 127)
    assert_f16_bitexact(host(c), O.dequant_f16(O.gemm_i32(a, b), tsa=1 / 127, tsb=1 / 127))


def test_f16_one_vector_scale(w8a8, gpu):
    m, n, k = 128, 256, 128
    a, b, sa, _ = inputs(m, n, k, 6)
    c = w8a8.gemm(dev(a, gpu), dev(b, gpu), scale_a=dev(sa, gpu), tensor_scale_b=0.5)
    assert_f16_bitexact(host(c), O.dequant_f16(O.gemm_i32(a, b), sa=sa, tsb=0.5))


def test_config2_full_4096(w8a8, gpu):
    # A [4096,4096], B [4096(N),4096(K)], sa/sb U[1e-3,1e-2]
    import torch
    m = n = k = 4096
    seed = G.config_seed(2)
    a, b, sa, sb = inputs(m, n, k, seed)
    ad, bd = dev(a, gpu), dev(b, gpu)
    acc = O.gemm_i32(a, b)
    assert_i32_equal(host(w8a8.gemm(ad, bd, out_dtype=torch.int32)), acc)
    c = w8a8.gemm(ad, bd, dev(sa, gpu), dev(sb, gpu))
    assert_f16_bitexact(host(c), O.dequant_f16(acc, sa, sb))


def test_closed_forms_extremes(w8a8, gpu):
    import torch
    k = 28672  # largest K of the path: |acc| <= 16129*K must not overflow
    a = np.full((64, k), 127, np.int8)
    b = np.full((64, k), -127, np.int8)
    c = host(w8a8.gemm(dev(a, gpu), dev(b, gpu), out_dtype=torch.int32))
    assert (c == -16129 * k).all()


def test_generic_path_odd_k_and_strides(w8a8, gpu):
    import torch
    m, n, k = 70, 90, 17  # k % 16 != 0 -> generic kernel
    a, b, sa, sb = inputs(m, n, k, 9)
    c = w8a8.gemm(dev(a, gpu), dev(b, gpu), out_dtype=torch.int32)
    assert_i32_equal(host(c), O.gemm_i32(a, b))
    # row strides that are not multiples of 16 (lda = k + 3)
    m, n, k = 64, 80, 96
    a, b, sa, sb = inputs(m, n, k + 3, 10)
    ad = dev(a, gpu)[:, :k]
    bd = dev(b, gpu)[:, :k]
    c = w8a8.gemm(ad, bd, out_dtype=torch.int32)
    assert_i32_equal(host(c), O.gemm_i32(a[:, :k], b[:, :k]))


def test_sample_layout(w8a8, gpu):
    import torch
    # rocwmma_gemm_quantized.cpp:205: A col-major (lda = m), B row-major [K, N] (ldb = n)
    m, n, k = 384, 256, 320
    at = G.int8(31, G.TID_A, (k, m))  # col-major A == row-major [K, M]
    b = G.int8(31, G.TID_B, (k, n))
    exp = O.gemm_i32(at, b, layout=1)
    c = w8a8.gemm(dev(at, gpu), dev(b, gpu), layout=w8a8.LAYOUT_A_COL_B_KN,
                  out_dtype=torch.int32)
    assert_i32_equal(host(c), exp)
    # no workspace -> generic strided kernel
    empty = torch.empty(0, dtype=torch.uint8, device=gpu)
    c2 = w8a8.gemm(dev(at, gpu), dev(b, gpu), layout=w8a8.LAYOUT_A_COL_B_KN,
                   out_dtype=torch.int32, workspace=empty)
    assert_i32_equal(host(c2), exp)


@pytest.mark.parametrize("m,n,k", [(300, 200, 100), (1000, 520, 784)])
def test_sample_layout_ragged(w8a8, gpu, m, n, k):
    # the sample layout's repack: lda = m, ldb = n not multiples of 16 (byte
    # path) or ragged tile edges, K padded with zeros
    import torch
    at = G.int8(41 + m, G.TID_A, (k, m))
    b = G.int8(41 + m, G.TID_B, (k, n))
    c = w8a8.gemm(dev(at, gpu), dev(b, gpu), layout=w8a8.LAYOUT_A_COL_B_KN, out_dtype=torch.int32)
    assert_i32_equal(host(c), O.gemm_i32(at, b, layout=1))


def test_output_leading_dimension(w8a8, gpu):
    import torch
    m, n, k = 200, 300, 128
    a, b, sa, sb = inputs(m, n, k, 12)
    big = torch.full((m, n + 7), -1, dtype=torch.int32, device=gpu)
    w8a8.gemm(dev(a, gpu), dev(b, gpu), out=big[:, :n])
    got = host(big)
    assert_i32_equal(got[:, :n], O.gemm_i32(a, b))
    assert (got[:, n:] == -1).all()


def test_fused_sq_gemm(w8a8, gpu):
    m, n, k = 512, 1024, 4096
    seed = G.config_seed(3)
    x = G.activations(seed, m, k)
    s = G.uniform(seed, G.TID_S, (k,), 0.5, 2.0)
    w = G.int8(seed, G.TID_B, (n, k))
    sb = G.uniform(seed, G.TID_SB, (n,), 1e-3, 1e-2)
    c, q, r = w8a8.fused_sq_gemm(dev(x, gpu), dev(s, gpu), dev(w, gpu), dev(sb, gpu))
    qo, ro = O.smoothquant(x, s)
    assert np.array_equal(host(q), qo) and np.array_equal(host(r), ro)
    assert_f16_bitexact(host(c), O.dequant_f16(O.gemm_i32(qo, w), ro, sb))


# fused SmoothQuant + W8A8 GEMM on the Llama-3-8B
# projections at M in {512, 2048, 8192}.  These are the headline launches:
# at M = 8192 qkv / o_proj / gate_up (K = 4096, 32 k-tiles) run the persistent
# kernel and down (K = 14336) the one-tile-per-block kernel; at M = 512 the
# smaller tiles, down split along K (workspace allocated as the bench does).
# q and r are checked in full; c is checked bit-exact on the first and last
# tile rows (256 rows each) plus 256 seeded random rows.
CFG3_PROJECTIONS = [("qkv", 4096, 6144), ("o_proj", 4096, 4096), ("gate_up", 4096, 28672),
                    ("down", 14336, 4096)]
CFG3_M = [512, 2048, 8192]
_cfg3_cache: dict = {}


def cfg3_inputs(k, n):
    """Seeded cfg3 inputs at the largest M (smaller M take the first rows:
    every element is a function of its flat index)."""
    seed = G.config_seed(3)
    if ("x", k) not in _cfg3_cache:
        _cfg3_cache[("x", k)] = G.activations(seed, max(CFG3_M), k)
        _cfg3_cache[("s", k)] = G.uniform(seed, G.TID_S, (k,), 0.5, 2.0)
    if ("w", n, k) not in _cfg3_cache:
        _cfg3_cache[("w", n, k)] = G.int8(seed, G.TID_B, (n, k))
        _cfg3_cache[("sb", n, k)] = G.uniform(seed, G.TID_SB, (n,), 1e-3, 1e-2)
    return (_cfg3_cache[("x", k)], _cfg3_cache[("s", k)], _cfg3_cache[("w", n, k)],
            _cfg3_cache[("sb", n, k)])


def cfg3_rows(m, seed):
    tile = 256
    rng = np.random.default_rng(seed)
    return np.unique(np.concatenate([np.arange(min(tile, m)), np.arange(max(0, m - tile), m),
                                     rng.integers(0, m, 256)]))


@pytest.mark.parametrize("m", CFG3_M)
@pytest.mark.parametrize("name,k,n", CFG3_PROJECTIONS)
def test_config3_fused_projection(w8a8, gpu, name, k, n, m):
    import torch
    xf, s, w, sb = cfg3_inputs(k, n)
    x = xf[:m]
    wd, sbd = dev(w, gpu), dev(sb, gpu)
    c, q, r = w8a8.fused_sq_gemm(dev(x, gpu), dev(s, gpu), wd, sbd)
    qo, ro = O.smoothquant(x, s)
    assert np.array_equal(host(q), qo), f"{name} m={m}: quantized activations differ"
    assert np.array_equal(host(r).view(np.uint32), ro.view(np.uint32)), f"{name} m={m}: row scales"
    rows = cfg3_rows(m, m + k + n)
    rows_d = torch.from_numpy(rows).to(gpu)
    got = host(c.index_select(0, rows_d))
    acc = O.gemm_i32(np.ascontiguousarray(qo[rows]), w)
    assert_f16_bitexact(got, O.dequant_f16(acc, ro[rows], sb))
    if w8a8.gemm_workspace_size(m, n, k) > 0:
        # the K-split launch (workspace) equals the unsplit one everywhere
        none = torch.empty(0, dtype=torch.uint8, device=gpu)
        c2, _, _ = w8a8.fused_sq_gemm(dev(x, gpu), dev(s, gpu), wd, sbd, workspace=none)
        assert torch.equal(c.view(torch.int16), c2.view(torch.int16)), f"{name} m={m}: split"


# Seeded random shapes over every dispatch the library makes (decode-size m,
# the tile sizes and their K splits with the workspace, the persistent kernel
# at 2+ tiles per CU, ragged m / n / k), int32 and fp16, against the oracle on
# the first and last rows and a sample.
GEMM_FUZZ_SEEDS = [21, 22, 23, 24, 25, 26]


@pytest.mark.parametrize("seed", GEMM_FUZZ_SEEDS)
def test_random_shapes(w8a8, gpu, seed):
    import torch
    rng = np.random.default_rng(seed)
    m = int(rng.choice([1, 7, 64, 65, 300, 512, 1100, 2048, 4100, 8192]))
    n = int(rng.choice([8, 136, 1000, 2056, 4096, 6144, 9000]))
    k = int(rng.choice([16, 144, 1024, 2064, 4096, 8192]))
    a, b, sa, sb = inputs(m, n, k, seed)
    ws_bytes = w8a8.gemm_workspace_size(m, n, k)
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=gpu) if ws_bytes else None
    da, db = dev(a, gpu), dev(b, gpu)
    ci = host(w8a8.gemm(da, db, out_dtype=torch.int32, workspace=ws))
    cf = host(w8a8.gemm(da, db, dev(sa, gpu), dev(sb, gpu), workspace=ws))
    pick = np.unique(np.concatenate([np.arange(min(m, 4)), np.arange(max(0, m - 4), m),
                                     rng.integers(0, m, 24)]))
    acc = O.gemm_i32(a[pick], b)
    assert_i32_equal(ci[pick], acc)
    assert_f16_bitexact(cf[pick], O.dequant_f16(acc, sa[pick], sb))
