"""w8a8_gemm_noalloc: w8a8_gemm whose workspace is the library's own per-GPU
scratch array (no allocation in the call).  Through the C ABI it must equal
w8a8_gemm given a workspace, bit for bit, on consecutive calls (the second
smaller: the array keeps the first call's contents), on the K-split shapes
that actually use the scratch, on shapes that do not, and on the sample
layout's repack; shapes that would need more scratch than the library holds
are refused before any HIP call."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle_lib as O
from checks import assert_f16_bitexact, assert_i32_equal, dev, host, plan
from optimized_rocwmma_samples_amd import _lib as L
from optimized_rocwmma_samples_amd import datagen as G

SCRATCH = 32 << 20


def _noalloc(w8a8, a, b, c, sa=None, sb=None, layout=0, tsa=1.0, tsb=1.0, m=None, n=None, k=None):
    import torch
    lib = w8a8.library()
    if layout == 0:
        m, k = a.shape
        n = b.shape[0]
        lda, ldb = a.stride(0), b.stride(0)
    else:
        lda, ldb = m, n
    out = 0 if c.dtype == torch.int32 else 1
    stream = torch.cuda.current_stream(c.device).cuda_stream if c.is_cuda else None
    rc = lib.w8a8_gemm_noalloc(m, n, k, a.data_ptr(), b.data_ptr(), c.data_ptr(), lda, ldb,
                               c.stride(0), sa.data_ptr() if sa is not None else None,
                               sb.data_ptr() if sb is not None else None, tsa, tsb, out, layout,
                               stream)
    return rc, lib.w8a8_last_error().decode()


def _inputs(m, n, k, seed):
    return (G.int8(seed, G.TID_A, (m, k)), G.int8(seed, G.TID_B, (n, k)),
            G.uniform(seed, G.TID_SA, (m,), 1e-3, 1e-2), G.uniform(seed, G.TID_SB, (n,), 1e-3, 1e-2))


def test_noalloc_refuses_oversized_shapes_before_hip(w8a8):
    # sample layout m = n = k = 8192: the repack needs 128 MiB > 32 MiB; the
    # pointers are never touched (no HIP call happens on this path)
    lib = w8a8.library()
    fake = ctypes.c_void_p(0x1000)
    rc = lib.w8a8_gemm_noalloc(8192, 8192, 8192, fake, fake, fake, 8192, 8192, 8192, None, None,
                               1.0, 1.0, 0, 1, None)
    assert rc == 1 and "needs" in lib.w8a8_last_error().decode()
    rc = lib.w8a8_gemm_noalloc(0, 16, 16, fake, fake, fake, 16, 16, 16, None, None, 1.0, 1.0, 0,
                               0, None)
    assert rc == 1 and "w8a8_gemm_noalloc" in lib.w8a8_last_error().decode()


# (m, n, k), K pieces: two large and a smaller split (the scratch holds the partials),
# then two shapes with no split, one a decode kernel's, and split decode tiles
SHAPES = [(512, 4096, 14336, 2), (1200, 1067, 21200, 5), (300, 600, 8192, 5),
          (1000, 1000, 1008, 1), (512, 4096, 4096, 1), (8, 1000, 512, 1), (16, 4096, 4096, 4),
          (32, 4096, 16384, 8)]


@pytest.mark.gpu
def test_noalloc_equals_gemm_consecutive_calls(w8a8, gpu):
    import torch
    print("noalloc: consecutive calls", SHAPES, flush=True)
    for i, (m, n, k, pieces) in enumerate(SHAPES):
        assert plan(w8a8, L.PLAN_GEMM, m, n, k, SCRATCH)[2] == pieces
        a, b, sa, sb = _inputs(m, n, k, 0xA110C + i)
        ad, bd, sad, sbd = dev(a, gpu), dev(b, gpu), dev(sa, gpu), dev(sb, gpu)
        ref_i = w8a8.gemm(ad, bd, out_dtype=torch.int32)       # w8a8_gemm, workspace given
        ref_h = w8a8.gemm(ad, bd, sad, sbd)
        ci = torch.full((m, n), -7, dtype=torch.int32, device=gpu)
        ch = torch.full((m, n), -7, dtype=torch.float16, device=gpu)
        rc, msg = _noalloc(w8a8, ad, bd, ci)
        assert rc == 0, msg
        rc, msg = _noalloc(w8a8, ad, bd, ch, sad, sbd)
        assert rc == 0, msg
        assert torch.equal(ci, ref_i), (m, n, k)
        assert torch.equal(ch.view(torch.int16), ref_h.view(torch.int16)), (m, n, k)
        rows = np.unique(np.concatenate([np.arange(min(m, 8)), np.arange(max(0, m - 8), m)]))
        assert_i32_equal(host(ci)[rows], O.gemm_i32(np.ascontiguousarray(a[rows]), b))


@pytest.mark.gpu
def test_noalloc_second_call_smaller(w8a8, gpu):
    # the same entry point twice in a row, the second on a smaller split
    # shape: its partials overwrite only part of what the first left
    import torch
    outs = []
    for (m, n, k, seed) in [(512, 512, 16384, 1), (256, 1024, 4096, 2)]:
        assert plan(w8a8, L.PLAN_GEMM, m, n, k, SCRATCH)[2] > 1
        a, b, sa, sb = _inputs(m, n, k, 0xB0 + seed)
        ad, bd, sad, sbd = dev(a, gpu), dev(b, gpu), dev(sa, gpu), dev(sb, gpu)
        c = torch.empty((m, n), dtype=torch.float16, device=gpu)
        rc, msg = _noalloc(w8a8, ad, bd, c, sad, sbd)
        assert rc == 0, msg
        outs.append((a, b, sa, sb, c))
    for a, b, sa, sb, c in outs:
        assert_f16_bitexact(host(c), O.dequant_f16(O.gemm_i32(a, b), sa, sb))


@pytest.mark.gpu
def test_noalloc_sample_layout(w8a8, gpu):
    import torch
    m, n, k = 384, 256, 320
    at = G.int8(31, G.TID_A, (k, m))
    b = G.int8(31, G.TID_B, (k, n))
    c = torch.empty((m, n), dtype=torch.int32, device=gpu)
    rc, msg = _noalloc(w8a8, dev(at, gpu), dev(b, gpu), c, layout=1, m=m, n=n, k=k)
    assert rc == 0, msg
    assert_i32_equal(host(c), O.gemm_i32(at, b, layout=1))


# Run in a fresh process, so that the captured call is the first
# w8a8_gemm_noalloc call of the process on the device: its one-time lookup of
# the scratch array's device address then happens inside the capture.
_CAPTURE_FIRST = r"""
import ctypes
import sys
import numpy as np
import torch
sys.path.insert(0, sys.argv[1])
import optimized_rocwmma_samples_amd as w8a8
from optimized_rocwmma_samples_amd import datagen as G
dev = torch.device("cuda:0")
m, n, k = 512, 4096, 14336  # a K-split shape: the partials live in the scratch array
sizes, plan = (ctypes.c_uint32 * 4)(m, n, k, 32 << 20), (ctypes.c_uint32 * 3)()
assert w8a8.library().w8a8_debug_plan(1, sizes, plan) == 0 and list(plan) == [128, 128, 2]
a = torch.from_numpy(G.int8(7, G.TID_A, (m, k))).to(dev)
b = torch.from_numpy(G.int8(7, G.TID_B, (n, k))).to(dev)
sa = torch.from_numpy(G.uniform(7, G.TID_SA, (m,), 1e-3, 1e-2)).to(dev)
sb = torch.from_numpy(G.uniform(7, G.TID_SB, (n,), 1e-3, 1e-2)).to(dev)
c = torch.zeros((m, n), dtype=torch.float16, device=dev)
lib = w8a8.library()
torch.cuda.synchronize()
st = torch.cuda.Stream()
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g, stream=st):
    rc = lib.w8a8_gemm_noalloc(m, n, k, a.data_ptr(), b.data_ptr(), c.data_ptr(), k, k, n,
                               sa.data_ptr(), sb.data_ptr(), 1.0, 1.0, 1, 0,
                               torch.cuda.current_stream().cuda_stream)
assert rc == 0, lib.w8a8_last_error().decode()
ws = torch.empty(w8a8.gemm_workspace_size(m, n, k), dtype=torch.uint8, device=dev)
ref = w8a8.gemm(a, b, sa, sb, workspace=ws)
torch.cuda.synchronize()
for i in range(3):
    c.zero_()
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(c.view(torch.int16), ref.view(torch.int16)), f"replay {i} differs"
    # eager work between replays, over the same scratch (a smaller problem)
    c2 = torch.empty((256, 1024), dtype=torch.float16, device=dev)
    rc = lib.w8a8_gemm_noalloc(256, 1024, 4096, a.data_ptr(), b.data_ptr(), c2.data_ptr(), k, k,
                               1024, sa.data_ptr(), sb.data_ptr(), 1.0, 1.0, 1, 0,
                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.w8a8_last_error().decode()
    torch.cuda.synchronize()
print("CAPTURED-FIRST OK")
"""


@pytest.mark.gpu
def test_noalloc_first_call_under_graph_capture(w8a8, gpu, tmp_path):
    """The entry point's first call in a process, made under HIP graph capture
    (where a caller that cannot allocate would make it): the capture succeeds
    and every replay equals w8a8_gemm bit for bit, with eager calls over the
    same scratch between the replays."""
    import subprocess
    import sys
    from pathlib import Path
    root = Path(__file__).resolve().parents[1]
    script = tmp_path / "capture_first.py"
    script.write_text(_CAPTURE_FIRST)
    print("running noalloc capture-first subprocess", flush=True)
    r = subprocess.run([sys.executable, str(script), str(root)], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=110)
    assert r.returncode == 0 and "CAPTURED-FIRST OK" in r.stdout, r.stdout[-3000:]
