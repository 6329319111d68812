"""a8w8 gate/up GEMM with gelu_and_mul in its epilogue (prefill), against the
plain GEMM without a workspace and gelu_and_mul: the K order of a sum does not
depend on the tile, so the outputs agree bit for bit.  One tile, ragged rows
and columns (tiles moved back inside the matrix, d not a multiple of 8), an odd
number of K steps, each tile shape of the plan, both types."""

import pytest
import torch

from esimd_learning_amd import cabi, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,io", [(torch.float16, 0), (torch.bfloat16, 1)])
@pytest.mark.parametrize("M,d,K", [
    (128, 128, 128), (129, 131, 128), (300, 1001, 256), (300, 2570, 384), (700, 4099, 640), (900, 8195, 384),
    (2048, 6912, 512), (1500, 8195, 1152), (261, 6620, 1152),
])
def test_glu_epilogue(ops, dev, M, d, K, dtype, io):
    print(f"a8w8 glu M={M} d={d} K={K} {dtype}", flush=True)
    lib = cabi.load()
    W8, sw = synthetic.weight_fp8(2 * d, K, seed=5)
    b, sb = W8.to(dev), sw.float().to(dev)
    x = synthetic.activations(M, K, seed=6, dtype=dtype).to(dev)
    a = torch.empty(M, K, dtype=torch.float8_e4m3fn, device=dev)
    sa = torch.empty(M, device=dev)
    ops.esimd_per_token_quant_fp8(x, a, sa)
    st = cabi.stream_ptr()
    gu = torch.empty(M, 2 * d, dtype=dtype, device=dev)
    cabi.check(lib.cek_gemm_fp8_a8w8(cabi.ptr(a), cabi.ptr(sa), cabi.ptr(b), cabi.ptr(sb), cabi.ptr(gu), M, 2 * d, K, io, st))
    want = torch.empty(M, d, dtype=dtype, device=dev)
    ops.esimd_gelu_and_mul(want, gu)
    buf = torch.full((M * d + 64,), float("nan"), dtype=dtype, device=dev)
    rc = lib.cek_gemm_fp8_a8w8_gelu_and_mul(cabi.ptr(a), cabi.ptr(sa), cabi.ptr(b), cabi.ptr(sb), cabi.ptr(buf[32:]),
                                            M, d, K, io, st)
    cabi.check(rc)
    got = buf[32:32 + M * d].view(M, d)
    assert torch.equal(got, want)
    assert buf[:32].isnan().all() and buf[32 + M * d:].isnan().all()


def test_glu_declines(dev):
    """Below a tile and for K % 128 nothing is launched; bad arguments are errors."""
    lib = cabi.load()
    z = torch.zeros(256 * 256, dtype=torch.uint8, device=dev)
    s, y = torch.zeros(512, device=dev), torch.zeros(256 * 256, dtype=torch.float16, device=dev)
    p, ps, py = cabi.ptr(z), cabi.ptr(s), cabi.ptr(y)

    def call(M, d, K, a=p):
        return lib.cek_gemm_fp8_a8w8_gelu_and_mul(a, ps, p, ps, py, M, d, K, 0, cabi.stream_ptr())

    unsupported, invalid = call(128, 128, 144), call(128, 128, 8)
    assert call(127, 128, 128) == unsupported and call(128, 127, 128) == unsupported and unsupported != 0
    assert call(128, 128, 128, a=None) == invalid and call(-1, 128, 128) == invalid and invalid not in (0, unsupported)
    assert call(0, 128, 128) == 0


def test_glu_declines_faster_pair(ops, dev):
    """Where the GEMM (256 x 192 tiles fit) and gelu_and_mul are faster, nothing is launched."""
    lib = cabi.load()
    M, d, K = 640, 6912, 5120
    y = torch.full((M, d), float("nan"), dtype=torch.float16, device=dev)
    z, s = torch.zeros(2 * d * K, dtype=torch.uint8, device=dev), torch.zeros(2 * d, device=dev)
    rc = lib.cek_gemm_fp8_a8w8_gelu_and_mul(cabi.ptr(z), cabi.ptr(s), cabi.ptr(z), cabi.ptr(s), cabi.ptr(y), M, d, K, 0,
                                            cabi.stream_ptr())
    assert rc == cabi.CEK_ERR_UNSUPPORTED and y.isnan().all()


@pytest.mark.parametrize("shared", ["a", "b", "a_scale"])
def test_glu_output_over_operand(ops, dev, shared):
    """An output that shares memory with an operand: the op keeps the two
    launches, whose first has read the operands before the second writes."""
    M, d, K = 700, 4099, 640
    print(f"a8w8 glu output over {shared}", flush=True)
    W8, sw = synthetic.weight_fp8(2 * d, K, seed=5)
    a, sa = synthetic.quantize_rows(synthetic.activations(M, K, seed=6).float())
    t = {"a": a.view(torch.uint8), "b": W8.view(torch.uint8), "a_scale": sa, "b_scale": sw.float()}
    t = {k: v.to(dev) for k, v in t.items()}
    want = torch.empty(M, d, dtype=torch.float16, device=dev)
    ops.esimd_gemm_fp8_a8w8_gelu_and_mul(t["a"], t["a_scale"], t["b"], t["b_scale"], want)
    nbytes = t[shared].numel() * t[shared].element_size()
    buf = torch.empty(max(M * d * 2, nbytes), dtype=torch.uint8, device=dev)
    t[shared] = buf[:nbytes].view(t[shared].dtype).view(t[shared].shape).copy_(t[shared])
    got = buf[:M * d * 2].view(torch.float16).view(M, d)
    ops.esimd_gemm_fp8_a8w8_gelu_and_mul(t["a"], t["a_scale"], t["b"], t["b_scale"], got)
    assert torch.equal(got, want)
