"""GPU parity of the w8a16 GEMM's 128 x 128 tile in two K teams.

It serves 65 and more rows where its tiles make one round of at most 256
workgroups, unsplit (any caller) and, with a workspace, in parts of K.  Sizes:
rows and columns of less than a tile and of a tile and a few, K of one 64-deep
step (the second team has none), of an odd count of them (a last stage of half
its values), and parts whose own count is odd.

Reference: the product in float64.  Bound per output: half a unit in the last
place of the output type plus the fp32 sum's (K + 16) 2^-24 sum |x w| s.
"""

import pytest
import torch

from esimd_learning_amd import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("io,fmt", [(torch.float16, torch.float8_e4m3fn), (torch.bfloat16, torch.float8_e5m2)])
@pytest.mark.parametrize("M,K,N", [(65, 64, 128), (100, 320, 300), (129, 1088, 131), (333, 128, 2050), (127, 2176, 136),
                                   (200, 4288, 260), (65, 4160, 4096)])
@pytest.mark.parametrize("split", [False, True])
def test_gemm_team(ops, dev, M, K, N, io, fmt, split):
    print(f"gemm team M={M} K={K} N={N} {io} split={split}", flush=True)
    W8, s = synthetic.weight_fp8(N, K, seed=K + N, fmt=fmt)
    x = synthetic.activations(M, K, seed=M, dtype=io)
    y = torch.full((M, N), float("nan"), dtype=io, device=dev)
    if split:  # the op with a per-tensor scale takes the workspace the plan asks for
        s = s[:1].contiguous()
        ops.esimd_gemm_fp8_pert(x.to(dev), W8.to(dev), s.to(dev), y)
    else:
        ops.esimd_gemv_fp8_pern(x.to(dev), W8.to(dev), s.to(dev), y, N, K)
    x64, w64, s64 = x.double(), W8.float().double(), s.double()
    ref = (x64 @ w64.t()) * s64
    half_ulp = (2.0 ** -11 if io == torch.float16 else 2.0 ** -8) * ref.abs() + 2.0 ** -25
    bound = half_ulp * 1.001 + (K + 16) * 2.0 ** -24 * ((x64.abs() @ w64.abs().t()) * s64)
    err = (y.cpu().double() - ref).abs()
    assert bool((err <= bound).all()), f"{float((err / bound).max()):.3g} of the bound"
