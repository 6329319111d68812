"""The add+RMSNorm (+ quantisation) with outputs apart from its inputs
(cek_add_rms_norm_out), and the fused norm+GEMV ops that use it beyond four
rows: bit for bit the in-place ops', inputs left alone, also where residual_out
shares memory with an input (the op then works on copies)."""

import pytest
import torch

from esimd_learning_amd import cabi, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,io", [(torch.float16, 0), (torch.bfloat16, 1)])
@pytest.mark.parametrize("T,H", [(1, 8), (5, 2056), (3, 1001), (1025, 512)])
def test_norm_out_equals_in_place(ops, dev, T, H, dtype, io):
    print(f"norm out T={T} H={H} {dtype}", flush=True)
    lib = cabi.load()
    h = synthetic.activations(T, H, seed=1, dtype=dtype).to(dev)
    r = synthetic.activations(T, H, seed=2, dtype=dtype).to(dev)
    w = synthetic.norm_weight(H, dtype=dtype).to(dev)
    h0, r0 = h.clone(), r.clone()
    ho, ro, rq = torch.empty_like(h), torch.empty_like(r), torch.empty_like(r)
    q = torch.empty(T, H, dtype=torch.float8_e4m3fn, device=dev)
    s = torch.empty(T, device=dev)
    st = cabi.stream_ptr()
    cabi.check(lib.cek_add_rms_norm_out(cabi.ptr(h), cabi.ptr(r), cabi.ptr(w), cabi.ptr(ro), cabi.ptr(ho), T, H, 1e-6,
                                        io, None, None, st))
    cabi.check(lib.cek_add_rms_norm_out(cabi.ptr(h), cabi.ptr(r), cabi.ptr(w), cabi.ptr(rq), None, T, H, 1e-6, io,
                                        cabi.ptr(q), cabi.ptr(s), st))
    assert torch.equal(h, h0) and torch.equal(r, r0)
    q2, s2, r2 = torch.empty_like(q), torch.empty_like(s), r.clone()
    ops.esimd_fused_add_rms_norm_quant_fp8(h, r2, w, 1e-6, q2, s2)
    assert torch.equal(rq, r2) and torch.equal(s, s2) and torch.equal(q.view(torch.uint8), q2.view(torch.uint8))
    ops.esimd_fused_add_rms_norm_batched(h, r, w, 1e-6)
    assert torch.equal(ho, h) and torch.equal(ro, r)


@pytest.mark.parametrize("H", [2048, 2056, 5120, 14336])
def test_norm_few_rows_equal_many(ops, dev, H):
    """512 rows and one more: the launches differ in when they load, not in values."""
    print(f"norm rows H={H}", flush=True)
    h, r = (synthetic.activations(513, H, seed=s).to(dev) for s in (1, 2))
    w = synthetic.norm_weight(H).to(dev)
    h1, r1 = h[:512].clone(), r[:512].clone()
    ops.esimd_fused_add_rms_norm_batched(h, r, w, 1e-6)
    ops.esimd_fused_add_rms_norm_batched(h1, r1, w, 1e-6)
    assert torch.equal(h[:512], h1) and torch.equal(r[:512], r1)


@pytest.mark.parametrize("alias", ["apart", "residual", "hidden", "half"])
@pytest.mark.parametrize("M,N,K", [(6, 272, 1024), (100, 300, 2048), (200, 256, 4096)])
def test_norm_gemv_beyond_four_rows(ops, dev, M, N, K, alias):
    print(f"norm gemv M={M} N={N} K={K} {alias}", flush=True)
    W8, sw = synthetic.weight_fp8(N, K, seed=3)
    W8, sw = W8.to(dev), sw.to(dev)
    buf = synthetic.activations(3 * M, K, seed=4).to(dev)
    w = synthetic.norm_weight(K).to(dev)
    h0, r0 = buf[:M].clone(), buf[M:2 * M].clone()
    x, rn = h0.clone(), r0.clone()
    ops.esimd_fused_add_rms_norm_batched(x, rn, w, 1e-6)
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    ops.esimd_gemv_fp8_pern(x, W8, sw, y, N, K)
    out = {"apart": slice(2 * M, 3 * M), "residual": slice(M, 2 * M), "hidden": slice(0, M),
           "half": slice(M + M // 2, 2 * M + M // 2)}[alias]
    y1 = torch.full_like(y, float("nan"))
    ops.esimd_fused_add_rms_norm_gemv_fp8(buf[:M], buf[M:2 * M], w, 1e-6, buf[out], W8, sw, y1)
    assert torch.equal(buf[out], rn) and torch.equal(y1, y)


@pytest.mark.parametrize("K,N", [(4096, 6144), (5120, 16384), (5120, 16386), (6144, 512)])
def test_quant_gemv_at_64_rows(ops, dev, K, N):
    """64 rows, where the a8w8 product is a streaming launch or split in K by its
    sizes: the fused op, its two ops and the entry point without a workspace of
    the caller's make the same choice, so they agree bit for bit."""
    M = 64
    print(f"norm quant gemv M={M} N={N} K={K}", flush=True)
    lib = cabi.load()
    W8, sw = synthetic.weight_fp8(N, K, seed=3)
    W8, sw = W8.view(torch.uint8).to(dev), sw.to(dev)
    h, r = (synthetic.activations(M, K, seed=s).to(dev) for s in (4, 5))
    w = synthetic.norm_weight(K).to(dev)
    q = torch.empty(M, K, dtype=torch.float8_e4m3fn, device=dev)
    s, ro, rn = torch.empty(M, device=dev), torch.empty_like(r), r.clone()
    ops.esimd_fused_add_rms_norm_quant_fp8(h, rn, w, 1e-6, q, s)
    a = q.view(torch.uint8)
    y, y1, y2, g, g1 = (torch.full((M, n), float("nan"), dtype=torch.float16, device=dev)
                        for n in (N, N, N, N // 2, N // 2))
    ops.esimd_gemm_fp8_a8w8(a, s, W8, sw, y)
    ops.esimd_gemm_fp8_a8w8_gelu_and_mul(a, s, W8, sw, g)
    cabi.check(lib.cek_gemm_fp8_a8w8_noalloc(cabi.ptr(a), cabi.ptr(s), cabi.ptr(W8), cabi.ptr(sw), cabi.ptr(y2), M, N,
                                             K, 0, cabi.stream_ptr()))
    assert torch.equal(y, y2)
    q1, s1 = torch.empty_like(q), torch.empty_like(s)
    ops.esimd_fused_add_rms_norm_quant_gemv_fp8(h, r, w, 1e-6, ro, q1, s1, W8, sw, y1)
    assert torch.equal(y, y1)
    ops.esimd_fused_add_rms_norm_quant_gemv_fp8(h, r, w, 1e-6, ro, q1, s1, W8, sw, g1, True)
    assert torch.equal(g, g1)
