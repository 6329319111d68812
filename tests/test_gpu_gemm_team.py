"""GPU parity of the w8a16 GEMM's 128 x 128 tile in two K teams.

It serves 65 and more rows where its tiles make one round of at most 256
workgroups, unsplit or, with a workspace, in 2 or 4 parts of K.  Sizes: rows
and columns of less than a tile and of a tile and a few, K of one 64-deep
step (the second team has none), of an odd count of them (a last stage of half
its values), and parts whose own count is odd.

Reference: the product in float64.  Bound per output: half a unit in the last
place of the output type plus the fp32 sum's (K + 16) 2^-24 sum |x w| s.
"""

import pytest
import torch

from esimd_learning_amd import cabi, synthetic

pytestmark = pytest.mark.gpu

TEAM = 6  # its index in the list of w8a16 tiles


@pytest.mark.parametrize("io,fmt", [(torch.float16, torch.float8_e4m3fn), (torch.bfloat16, torch.float8_e5m2)])
@pytest.mark.parametrize("M,K,N,parts", [(65, 64, 128, 1), (100, 320, 300, 1), (129, 1088, 131, 1), (333, 128, 2050, 1),
                                         (127, 2176, 136, 2), (200, 4288, 260, 1), (65, 4160, 4096, 1),
                                         (133, 2048, 132, 2), (65, 28672, 8100, 4)])
def test_gemm_team(ops, dev, M, K, N, parts, io, fmt):
    """Without a workspace (the bare C ABI) and with the one the plan asks for (the op)."""
    print(f"gemm team M={M} K={K} N={N} {io} parts={parts}", flush=True)
    lib = cabi.load()
    assert lib.cek_gemm_fp8_pert_plan(M, N, K, 0) == 16 * TEAM + 1
    assert lib.cek_gemm_fp8_pert_plan(M, N, K, lib.cek_gemm_fp8_pert_workspace_size(M, N, K)) == 16 * TEAM + parts
    W8, s = synthetic.weight_fp8(N, K, seed=K + N, fmt=fmt)
    x = synthetic.activations(M, K, seed=M, dtype=io)
    xd, Wd, sd = x.to(dev), W8.to(dev), s.to(dev)
    y, y1 = (torch.full((M, N), float("nan"), dtype=io, device=dev) for _ in range(2))
    ops.esimd_gemv_fp8_pern(xd, Wd, sd, y, N, K)
    cabi.check(lib.cek_gemv_fp8_pern(cabi.ptr(xd), cabi.ptr(Wd), cabi.ptr(sd), cabi.ptr(y1), M, N, K,
                                     cabi.CEK_F16 if io == torch.float16 else cabi.CEK_BF16,
                                     cabi.CEK_E4M3 if fmt == torch.float8_e4m3fn else cabi.CEK_E5M2, cabi.CEK_F32,
                                     cabi.stream_ptr()))
    x64, w64, s64 = x.double(), W8.float().double(), s.double()
    ref = (x64 @ w64.t()) * s64
    half_ulp = (2.0 ** -11 if io == torch.float16 else 2.0 ** -8) * ref.abs() + 2.0 ** -25
    bound = half_ulp * 1.001 + (K + 16) * 2.0 ** -24 * ((x64.abs() @ w64.abs().t()) * s64)
    for out in (y, y1):
        err = (out.cpu().double() - ref).abs()
        assert bool((err <= bound).all()), f"{float((err / bound).max()):.3g} of the bound"
