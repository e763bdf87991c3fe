"""GPU parity of the SmoothQuant quantizer against the CPU oracle (bit-exact on
q and on the bits of r) and, where oracle/_ref was built, against the
reference's own kernel_smoothquant / kernel_moe_smoothquant run on the same
device inputs."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from checks import plan
from optimized_rocwmma_samples_amd import _lib as L
from optimized_rocwmma_samples_amd import datagen as G

pytestmark = pytest.mark.gpu


def dev(a, device):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def host(t):
    return t.cpu().numpy()


def run_sq(w8a8, x_np, s_np, device, qmax=127.0):
    x = dev(x_np, device)
    s = dev(s_np, device)
    q, r = w8a8.smoothquant(x, s, qmax)
    return host(q), host(r)


def check_exact(qg, rg, qo, ro):
    assert np.array_equal(rg.view(np.uint32), ro.view(np.uint32)), "row scales differ"
    if not np.array_equal(qg, qo):
        bad = np.argwhere(qg != qo)
        raise AssertionError(f"{len(bad)} q mismatches, first at {bad[:5].tolist()}")


def test_config1_full(w8a8, gpu):
    # X fp16 [2048, 4096] N(0,1) with 0.5% outlier columns x20,
    # s fp32 [4096] U[0.5, 2].
    seed = G.config_seed(1)
    x = G.activations(seed, 2048, 4096)
    s = G.uniform(seed, G.TID_S, (4096,), 0.5, 2.0)
    qg, rg = run_sq(w8a8, x, s, gpu)
    qo, ro = O.smoothquant(x, s)
    check_exact(qg, rg, qo, ro)


@pytest.mark.parametrize("n", [1, 7, 8, 100, 512, 513, 1000, 1024, 2048, 3000, 4096, 4104, 8192,
                               8200, 14336, 16384, 20000, 28672, 32768, 40000])
def test_row_lengths(w8a8, gpu, n):
    m = 9  # not a multiple of the 4 rows per block
    seed = 100 + n
    x = G.activations(seed, m, n)
    s = G.uniform(seed, G.TID_S, (n,), 0.5, 2.0)
    qg, rg = run_sq(w8a8, x, s, gpu)
    check_exact(qg, rg, *O.smoothquant(x, s))


@pytest.mark.parametrize("m,n", [(8192, 4096), (8197, 1000), (12289, 8), (32767, 2056),
                                 (32768, 2056), (1023, 4096), (1024, 4096), (3328, 4096),
                                 (4095, 3000), (4096, 4000), (2048, 14336), (777, 16384)])
def test_many_rows(w8a8, gpu, m, n):
    # the row-count boundaries of the launch choice for 2049-4096 columns
    # (below 1024 rows: a row over two waves, two 256-thread blocks per CU;
    # 1024-4095 and from 32768: one wave per row; 4096-32767: four
    # 256-thread blocks per CU), rows not a multiple of the blocks' row
    # groups, and 8193-16384 columns (one 16-wave row group per block)
    seed = 400 + m + n
    x = G.activations(seed, m, n)
    s = G.uniform(seed, G.TID_S, (n,), 0.5, 2.0)
    qg, rg = run_sq(w8a8, x, s, gpu)
    check_exact(qg, rg, *O.smoothquant(x, s))


@pytest.mark.parametrize("m", [1, 64, 65])
@pytest.mark.parametrize("n", [8192, 12288, 16384, 28672])
def test_decode_row_counts(w8a8, gpu, m, n):
    # decode row counts take the one-block-per-row launch (rows <= 64)
    seed = 300 + m + n
    x = G.activations(seed, m, n)
    s = G.uniform(seed, G.TID_S, (n,), 0.5, 2.0)
    qg, rg = run_sq(w8a8, x, s, gpu)
    check_exact(qg, rg, *O.smoothquant(x, s))


def test_zero_rows_ties_and_qmax(w8a8, gpu):
    n = 1024
    x = np.zeros((4, n), np.float16)
    x[1, :10] = np.array([127, 2.5, 3.5, -2.5, 0.5, 1.5, -0.5, -1.5, 126.5, 4.25])
    x[2] = G.normal(5, G.TID_X, (n,))
    x[3, 500] = -1e-7  # fp16 subnormal
    s = np.ones(n, np.float32)
    for qmax in (127.0, 100.0, 1.0):
        qg, rg = run_sq(w8a8, x, s, gpu, qmax)
        check_exact(qg, rg, *O.smoothquant(x, s, qmax))
    qg, rg = run_sq(w8a8, x, s, gpu)
    assert rg[0] == 0 and (qg[0] == 0).all()
    assert qg[1, :10].tolist() == [127, 2, 4, -2, 0, 2, 0, -2, 126, 4]


@pytest.mark.parametrize("n", [1000, 4096, 14336])
def test_non_finite_inputs_and_fractional_qmax(w8a8, gpu, n):
    """Rows holding inf, -inf, NaN and the fp16 extremes, quantized with integer
    and fractional quant_max: q and r equal the oracle's restatement of the
    reference's float ops (a NaN element is ignored by the row max and lands on
    -quant_max through fmaxf / fminf; an infinite row max gives r = inf,
    inv = 0, so finite elements quantize to 0 and the infinite ones to
    +-quant_max)."""
    m = 12
    x = G.activations(900 + n, m, n)
    x[0, 3] = np.inf
    x[1, 5] = -np.inf
    x[2, 7] = np.nan
    x[3, :4] = [np.nan, np.inf, -np.inf, np.nan]
    x[4, 100] = np.float16(65504)
    x[4, 101] = np.float16(-65504)
    x[5, :] = np.nan
    x[6, n - 1] = np.inf
    x[7, ::97] = np.nan
    s = G.uniform(900 + n, G.TID_S, (n,), 0.5, 2.0)
    for qmax in (127.0, 100.6, 7.25, 0.5):
        qg, rg = run_sq(w8a8, x, s, gpu, qmax)
        check_exact(qg, rg, *O.smoothquant(x, s, qmax))


def test_reference_default_fill(w8a8, gpu):
    # rocwmma_smoothquant.cpp:140-141: x=0.5, s=1 -> q=127, r=0.5/127
    x = np.full((64, 4096), 0.5, np.float16)
    qg, rg = run_sq(w8a8, x, np.ones(4096, np.float32), gpu)
    assert (qg == 127).all() and (rg == np.float32(0.5) / np.float32(127)).all()


def test_strided_and_unaligned(w8a8, gpu):
    import torch
    m, n = 17, 1000
    seed = 77
    xfull = G.activations(seed, m, n + 13)
    s = G.uniform(seed, G.TID_S, (n,), 0.5, 2.0)
    xd = dev(xfull, gpu)
    sd = dev(s, gpu)
    # row stride n+13 (not a multiple of 8) and a base 1 element off 16-byte alignment
    for view in (xd[:, :n], xd[:, 1:n + 1]):
        q = torch.zeros((m, n + 5), dtype=torch.int8, device=gpu)
        qv, r = w8a8.smoothquant(view, sd, out=q[:, :n])
        qo, ro = O.smoothquant(host(view), s)
        check_exact(host(qv), host(r), qo, ro)
        assert (host(q)[:, n:] == 0).all()  # padding columns untouched


def test_matches_reference_kernel(w8a8, gpu):
    ref = O.ref()
    if ref is None:
        pytest.skip("oracle/_ref (reference kernels) not built")
    import torch
    for (m, n) in [(256, 4096), (33, 1024), (8, 8192)]:
        seed = 3000 + n
        x = G.activations(seed, m, n)
        s = G.uniform(seed, G.TID_S, (n,), 0.5, 2.0)
        xd, sd = dev(x, gpu), dev(s, gpu)
        yr = torch.zeros((m, n), dtype=torch.int8, device=gpu)
        rr = torch.zeros(m, dtype=torch.float32, device=gpu)
        torch.cuda.synchronize()
        assert ref.ref_kernel_smoothquant(xd.data_ptr(), sd.data_ptr(), yr.data_ptr(),
                                          rr.data_ptr(), m, n, 127.0) == 0
        qg, rg = w8a8.smoothquant(xd, sd)
        check_exact(host(qg), host(rg), host(yr), host(rr))
        check_exact(host(yr), host(rr), *O.smoothquant(x, s))


# ------------------------------------------------------------------ MoE
def moe_inputs(tokens, hidden, experts, topk, seed):
    x = G.activations(seed, tokens, hidden)
    s = G.uniform(seed, G.TID_EXPERT_S, (experts, hidden), 0.5, 2.0)
    h = G.hash64(seed, G.TID_LOGITS, 0, tokens * experts).reshape(tokens, experts)
    ids = np.argsort(h, axis=1, kind="stable")[:, :topk].astype(np.int32)  # distinct per token
    return x, s, ids


@pytest.mark.parametrize("tokens,hidden,experts,topk", [(64, 4096, 8, 2), (37, 1000, 4, 3),
                                                        (16, 14336, 8, 2), (5, 8, 2, 1)])
def test_moe_token_major(w8a8, gpu, tokens, hidden, experts, topk):
    import torch
    x, s, ids = moe_inputs(tokens, hidden, experts, topk, 11 + hidden)
    ids[1, 0] = -1
    ids[2, -1] = experts  # invalid ids: rows untouched (:86-87)
    rows = tokens * topk
    q = torch.full((rows, hidden), -99, dtype=torch.int8, device=gpu)
    r = torch.full((rows,), -99.0, dtype=torch.float32, device=gpu)
    w8a8.moe_smoothquant(dev(x, gpu), dev(s, gpu), dev(ids, gpu), out=q, row_scale=r)
    qo, ro = O.moe_smoothquant(x, s, ids, fill=-99)
    check_exact(host(q), host(r), qo, ro)


# Every kernel of moe_quant_plan (chunks per lane, waves per row, by tokens) at odd
# lengths (rows at odd addresses, a last chunk of 1-7 elements) and at the edges of
# its columns; ids outside the experts skipped.
@pytest.mark.parametrize("tokens,hidden,experts,topk,kernel", [
    (9, 512, 8, 6, (1, 1, 0)), (700, 257, 8, 6, (1, 1, 0)), (4510, 9, 64, 8, (1, 1, 1)),
    (9, 513, 8, 6, (1, 2, 0)), (255, 1024, 8, 6, (1, 2, 0)), (1300, 1001, 8, 6, (2, 1, 0)),
    (3080, 515, 64, 8, (2, 1, 1)), (37, 1025, 8, 6, (1, 4, 0)), (260, 2047, 8, 6, (4, 1, 0)),
    (85, 2049, 8, 6, (2, 4, 0)), (530, 2055, 8, 6, (4, 2, 0)), (1290, 2051, 64, 8, (8, 1, 0)),
    (40, 8191, 8, 6, (4, 4, 0)), (1800, 4097, 4, 2, (4, 4, 0)), (600, 4103, 16, 6, (4, 4, 1)),
    (3, 16001, 4, 3, (2, 16, 0)), (430, 8199, 4, 3, (2, 16, 1)), (3, 16399, 4, 2, (4, 16, 0)),
    (690, 16399, 4, 3, (4, 16, 1)), (3, 32769, 4, 2, (0, 0, 0))])
def test_moe_pairs_and_tokens(w8a8, gpu, tokens, hidden, experts, topk, kernel):
    assert plan(w8a8, L.PLAN_MOE_QUANT, tokens * topk, hidden, topk) == kernel
    test_moe_token_major(w8a8, gpu, tokens, hidden, experts, topk)


@pytest.mark.parametrize("m,n", [(37, 9), (37, 513), (700, 1337), (37, 2047), (33, 4095), (5, 8001),
                                 (3, 8201), (1030, 8201), (3, 16390), (3, 32767)])
def test_odd_rows_at_odd_addresses(w8a8, gpu, m, n):
    import torch
    x = G.activations(n, m, n)
    s = G.uniform(n, G.TID_S, (n + 1,), 0.5, 2.0)
    buf = torch.zeros(m * n + 1, dtype=torch.float16, device=gpu)
    xd = buf[1:].view(m, n).copy_(dev(x, gpu))
    qbuf = torch.full((m * (n + 3) + 1,), -99, dtype=torch.int8, device=gpu)
    q, r = w8a8.smoothquant(xd, dev(s, gpu)[1:], out=qbuf[1:].view(m, n + 3)[:, :n])
    check_exact(host(q), host(r), *O.smoothquant(x, s[1:]))
    got = host(qbuf)
    assert got[0] == -99 and (got[1:].reshape(m, n + 3)[:, n:] == -99).all()


def test_moe_sorted_destinations(w8a8, gpu):
    import torch
    tokens, hidden, experts, topk = 50, 4096, 8, 2
    x, s, ids = moe_inputs(tokens, hidden, experts, topk, 5)
    _, _, _, _, dst = O.moe_sort(ids, experts, 32)
    rows = int(dst.max()) + 1
    q = torch.zeros((rows, hidden), dtype=torch.int8, device=gpu)
    r = torch.zeros((rows,), dtype=torch.float32, device=gpu)
    w8a8.moe_smoothquant(dev(x, gpu), dev(s, gpu), dev(ids, gpu), dst_row=dev(dst, gpu),
                         rows=rows, out=q, row_scale=r)
    qo, ro = O.moe_smoothquant(x, s, ids, dst_row=dst, rows=rows)
    check_exact(host(q), host(r), qo, ro)


def test_moe_matches_reference_kernel(w8a8, gpu):
    ref = O.ref()
    if ref is None:
        pytest.skip("oracle/_ref (reference kernels) not built")
    import torch
    tokens, hidden, experts, topk = 128, 4096, 8, 2
    x, s, ids = moe_inputs(tokens, hidden, experts, topk, 21)
    xd, sd, idd = dev(x, gpu), dev(s, gpu), dev(ids, gpu)
    rows = tokens * topk
    qr = torch.zeros((rows, hidden), dtype=torch.int8, device=gpu)
    rr = torch.zeros(rows, dtype=torch.float32, device=gpu)
    torch.cuda.synchronize()
    assert ref.ref_kernel_moe_smoothquant(xd.data_ptr(), sd.data_ptr(), idd.data_ptr(),
                                          qr.data_ptr(), rr.data_ptr(), tokens, hidden, topk,
                                          experts, 127.0) == 0
    qg, rg = w8a8.moe_smoothquant(xd, sd, idd)
    check_exact(host(qg), host(rg), host(qr), host(rr))
