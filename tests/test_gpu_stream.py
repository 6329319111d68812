"""GPU parity of the weight-streaming kernel (csrc/cek_stream.hip).

It serves 3 .. 64 rows at K outside the LDS-staged GEMV's set (any multiple of
64), 9 .. 16 rows of wide matrices, and 17 .. 64 rows at any K, for fp16 / bf16
activations with e4m3 / e5m2 weights and for e4m3 activations.  The sizes here
are the edges of its activation blocks (4, 8, 16, 32, 48, 64 rows), K of less
than a stage, of whole stages and with a remainder in the last one, fewer
stages than ring slots, and row counts that leave a workgroup's last rows (or
all but one) outside the matrix.

Reference: the product in float64 on the CPU.  Bound per output: half a unit
in the last place of the output type, 2^-11 (fp16) or 2^-8 (bf16) of the
value (2^-25 below fp16's normal range), plus the fp32 sum's (K + 16) 2^-24 sum
|x w| s.
"""

import ctypes

import pytest
import torch

from conftest import assert_close_fp
from esimd_learning_amd import synthetic

pytestmark = pytest.mark.gpu


def _check(y, x64, w64, s64, K, what):
    ref = (x64 @ w64.t()) * s64
    mag = (x64.abs() @ w64.abs().t()) * s64
    half_ulp = (2.0 ** -11 if y.dtype == torch.float16 else 2.0 ** -8) * ref.abs() + 2.0 ** -25
    bound = half_ulp * 1.001 + (K + 16) * 2.0 ** -24 * mag
    err = (y.cpu().double() - ref).abs()
    assert bool((err <= bound).all()), f"{what}: {float((err / bound).max()):.3g} of the bound"


@pytest.mark.parametrize("io,fmt,per_channel", [(torch.float16, torch.float8_e4m3fn, True),
                                                (torch.bfloat16, torch.float8_e5m2, False)])
@pytest.mark.parametrize("K,N", [(64, 7), (320, 250), (2112, 1025), (2560, 8200), (10240, 1), (6144, 136), (8192, 2048),
                                 (8192, 2049)])
@pytest.mark.parametrize("M", [3, 4, 5, 8, 9, 16])
def test_stream_gemv(ops, dev, M, K, N, io, fmt, per_channel):
    print(f"stream gemv M={M} K={K} N={N} {io} {fmt}", flush=True)
    W8, s = synthetic.weight_fp8(N, K, seed=K + N, fmt=fmt)
    x = synthetic.activations(M, K, seed=M, dtype=io)
    y = torch.full((M, N), float("nan"), dtype=io, device=dev)
    if per_channel:
        ops.esimd_gemv_fp8_pern(x.to(dev), W8.to(dev), s.to(dev), y, N, K)
    else:
        s = s[:1].contiguous()
        ops.esimd_gemv_fp8_pert(x.to(dev), W8.to(dev), s.to(dev), y)
    _check(y, x.double(), W8.float().double(), s.double(), K, f"M={M} K={K} N={N}")


@pytest.mark.parametrize("io,fmt", [(torch.float16, torch.float8_e4m3fn), (torch.bfloat16, torch.float8_e5m2)])
@pytest.mark.parametrize("M,K,N", [(17, 64, 33), (32, 448, 2050), (33, 4096, 1000), (48, 2112, 6145), (49, 1024, 17),
                                   (64, 320, 16400), (64, 5120, 300)])
def test_stream_gemm(ops, dev, M, K, N, io, fmt):
    print(f"stream gemm M={M} K={K} N={N} {io} {fmt}", flush=True)
    W8, s = synthetic.weight_fp8(N, K, seed=K + N, fmt=fmt)
    x = synthetic.activations(M, K, seed=M, dtype=io)
    y = torch.full((M, N), float("nan"), dtype=io, device=dev)
    ops.esimd_gemm_fp8_pert(x.to(dev), W8.to(dev), s[:1].to(dev), y)
    _check(y, x.double(), W8.float().double(), s[:1].double(), K, f"M={M} K={K} N={N}")


@pytest.mark.parametrize("M,K,N", [(3, 2560, 1000), (8, 576, 40), (16, 10240, 700), (17, 64, 33), (32, 4096, 6144),
                                   (33, 1088, 16390), (48, 5120, 129), (63, 2112, 4100), (24, 2048, 16500)])
def test_stream_a8w8(ops, dev, M, K, N):
    print(f"stream a8w8 M={M} K={K} N={N}", flush=True)
    W8, s = synthetic.weight_fp8(N, K, seed=K + N)
    a8, sa = synthetic.quantize_rows(synthetic.activations(M, K, seed=M).float())
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
    ops.esimd_gemm_fp8_a8w8(a8.to(dev), sa.to(dev), W8.to(dev), s.to(dev), y)
    # the two scales are multiplied in fp32 (2^-24), one more rounding of the product
    _check(y, a8.float().double() * sa.double()[:, None], W8.float().double(), s.double(), K + 2,
           f"M={M} K={K} N={N}")


@pytest.mark.parametrize("act,M,K,N", [("fp16", 17, 192, 16385), ("fp16", 17, 256, 16385), ("fp16", 64, 576, 16390),
                                       ("fp16", 64, 640, 16390), ("fp16", 33, 64, 32769), ("e4m3", 20, 768, 16400),
                                       ("e4m3", 20, 832, 16400), ("e4m3", 32, 1024, 32800), ("e4m3", 40, 128, 10240),
                                       ("e4m3", 40, 192, 10241), ("e4m3", 64, 256, 10250), ("e4m3", 64, 320, 10250),
                                       ("e4m3", 4, 16384, 4096), ("e4m3", 4, 16384, 4097), ("fp16", 4, 16384, 4097)])
def test_stream_or_tiles(ops, dev, act, M, K, N):
    """Wide matrices of short K on both sides of the line to the tiled GEMMs
    (whose fp8 MFMA sums 128 products in one step, hence the op pack's
    tolerance for e4m3 activations)."""
    print(f"stream or tiles {act} M={M} K={K} N={N}", flush=True)
    W8, s = synthetic.weight_fp8(N, K, seed=K)
    x = synthetic.activations(M, K, seed=M)
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
    if act == "e4m3":
        x, sa = synthetic.quantize_rows(x.float())
        ops.esimd_gemm_fp8_a8w8(x.to(dev), sa.to(dev), W8.to(dev), s.to(dev), y)
        ref = (x.float().double() * sa.double()[:, None]) @ (W8.float().double() * s.double()[:, None]).t()
        assert_close_fp(y.cpu(), ref, f"a8w8 M={M} K={K} N={N}")
    else:
        ops.esimd_gemv_fp8_pern(x.to(dev), W8.to(dev), s.to(dev), y, N, K)
        _check(y, x.double(), W8.float().double(), s.double(), K, "w8a16")


@pytest.mark.parametrize("M", [3, 5, 16])
@pytest.mark.parametrize("K", [320, 2560, 10240])
def test_stream_a8w8_fp32_sums(ops, dev, M, K):
    """Up to 16 rows of e4m3 activations are summed in fp32: an error of about
    1e-7 of the result moves some 2 1e-7 / 2^-11 = 0.05% of the fp16 outputs to the
    other side of a rounding boundary (the fp8 MFMA's sums move 6.7%)."""
    N = 2050
    print(f"stream a8w8 sums M={M} K={K}", flush=True)
    W8, s = synthetic.weight_fp8(N, K, seed=K)
    a8, sa = synthetic.quantize_rows(synthetic.activations(M, K, seed=M).float())
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    ops.esimd_gemm_fp8_a8w8(a8.to(dev), sa.to(dev), W8.to(dev), s.to(dev), y)
    ref = (a8.float().double() @ W8.float().double().t()) * (sa[:, None] * s[None]).double()
    assert float((y.cpu() != ref.half()).double().mean()) < 5e-3


# Columns at which a workgroup has 8, 12, 16, 24, 32, 40, 48, 56 and 64 weight rows
FORM_N = [1001, 2500, 3500, 5000, 6201, 8201, 11000, 12700, 16001]


@pytest.mark.parametrize("act,out,fmt", [("fp16", torch.float16, torch.float8_e4m3fn),
                                         ("bf16", torch.bfloat16, torch.float8_e5m2),
                                         ("e4m3", torch.float16, torch.float8_e4m3fn),
                                         ("e4m3", torch.bfloat16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("M", [3, 6, 13, 20, 30, 40, 60])
def test_stream_every_form(ops, dev, M, act, out, fmt):
    """Every activation block (4 .. 64 rows) with every count of weight rows, K of a
    whole stage and a part."""
    K = 320
    Wall, sall = synthetic.weight_fp8(max(FORM_N), K, seed=31, fmt=fmt)
    x = synthetic.activations(M, K, seed=M, dtype=torch.float16 if act == "e4m3" else out)
    if act == "e4m3":
        x, sa = synthetic.quantize_rows(x.float())
    for N in FORM_N:
        print(f"stream form M={M} N={N} {act} {out} {fmt}", flush=True)
        W8, s = Wall[:N], sall[:N]
        y = torch.full((M, N), float("nan"), dtype=out, device=dev)
        if act == "e4m3":
            ops.esimd_gemm_fp8_a8w8(x.to(dev), sa.to(dev), W8.to(dev), s.to(dev), y)
            _check(y, x.float().double() * sa.double()[:, None], W8.float().double(), s.double(), K + 2, f"N={N}")
        elif M <= 16:
            ops.esimd_gemv_fp8_pern(x.to(dev), W8.to(dev), s.to(dev), y, N, K)
            _check(y, x.double(), W8.float().double(), s.double(), K, f"N={N}")
        else:
            s = s[:1].contiguous()
            ops.esimd_gemm_fp8_pert(x.to(dev), W8.to(dev), s.to(dev), y)
            _check(y, x.double(), W8.float().double(), s.double(), K, f"N={N}")


@pytest.mark.parametrize("M,K,Ns", [(4, 2560, (4096, 512, 512)), (8, 2112, (9000, 1000, 8200)),
                                    (16, 4096, (14336, 4096, 9000)), (3, 6144, (1000, 3000))])
def test_stream_fused_equals_single(ops, dev, M, K, Ns):
    """A multi-matrix call gives each matrix what it gets alone, bit for bit
    (rotated K order for matrices of 8192 rows or more, and rows that other
    kernels serve, among them)."""
    print(f"stream fused M={M} K={K} N={Ns}", flush=True)
    x = synthetic.activations(M, K, seed=5).to(dev)
    ws, ss, ys = [], [], []
    for i, n in enumerate(Ns):
        W8, s = synthetic.weight_fp8(n, K, seed=20 + i)
        ws.append(W8.to(dev))
        ss.append(s.to(dev))
        ys.append(torch.full((M, n), float("nan"), dtype=torch.float16, device=dev))
    ops.esimd_gemv_fp8_pern_fused(x, ws, ss, ys)
    for n, w, s, y in zip(Ns, ws, ss, ys):
        one = torch.empty(M, n, dtype=torch.float16, device=dev)
        ops.esimd_gemv_fp8_pern(x, w, s, one, n, K)
        assert torch.equal(one, y), f"N={n}"


def _launches(fn):
    """Kernels that fn launches: the nodes of a graph captured from it."""
    with open("/proc/self/maps") as f:  # the HIP runtime that this process runs on
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        fn()
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("M,K,Ns,launches", [
    (4, 2560, (9000, 9000, 9000), 1), (5, 2560, (5120, 1024, 1024), 1), (8, 1088, (8191, 17), 1),
    (9, 4096, (8192, 1024, 1024), 1), (12, 6144, (8192, 1024, 1024), 1), (16, 2560, (1000, 9000, 14336, 9001), 2),
    (3, 1088, (9000, 1000, 8200), 2), (12, 4096, (14336, 4096), 2)])
def test_stream_fused_launches(ops, dev, M, K, Ns, launches):
    """Matrices of a multi-matrix call share a launch unless their sums differ in
    order (narrow ones and ones that start at rotated K stages, or whose rotation
    differs; the streaming and the staged kernel), and get what they get alone."""
    print(f"stream launches M={M} K={K} N={Ns}", flush=True)
    x = synthetic.activations(M, K, seed=5).to(dev)
    ws, ss = zip(*[[t.to(dev) for t in synthetic.weight_fp8(n, K, seed=20 + i)] for i, n in enumerate(Ns)])
    ys = [torch.full((M, n), float("nan"), dtype=torch.float16, device=dev) for n in Ns]
    ops.esimd_gemv_fp8_pern_fused(x, ws, ss, ys)
    for n, w, s, y in zip(Ns, ws, ss, ys):
        one = torch.empty(M, n, dtype=torch.float16, device=dev)
        ops.esimd_gemv_fp8_pern(x, w, s, one, n, K)
        assert torch.equal(one, y), f"N={n}"
    assert _launches(lambda: ops.esimd_gemv_fp8_pern_fused(x, ws, ss, ys)) == launches
