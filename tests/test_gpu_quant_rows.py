"""Per-token quantisation, bit for bit, over the row lengths at which its launch
changes form: 256, 512 and 1024 threads of 1 .. 8 units (8 elements each), few
and many rows, the loop for longer and unaligned rows.

The codes are those of the IEEE quotient x / scale, which the kernel forms
from one reciprocal per row: the rows hold every sign of zero, values from the
type's smallest to amax, a zero row, and (fp16, bf16) rows of tiny and huge
values, where the scale's floor and its largest values are reached.  A row that
holds an infinity keeps an infinite scale and signed zero codes for its finite
elements.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _codes(x, s):
    return (x.float() / s[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,H", [(5, 8), (5, 2048), (5, 2056), (5, 4096), (5, 4104), (5, 8200), (3, 16384), (3, 16392),
                                 (2, 32768), (2, 32776), (3, 1001), (513, 2056), (513, 8192), (512, 8200),
                                 (512, 16400)])
def test_quant_rows(ops, dev, T, H, dtype):
    print(f"quant rows T={T} H={H} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g) * torch.exp2(torch.randint(-20, 1, (T, H), generator=g).float())
    x[0, ::3] = -0.0
    x[0, 1::3] = 0.0
    x[1] = -0.0
    if T > 2:
        x[2] *= 2.0 ** -18                       # the floor of the scale
    if T > 3:
        x[3] *= 6e4 if dtype == torch.float16 else 1e38
    x = x.clamp(-6e4, 6e4).to(dtype) if dtype == torch.float16 else x.to(dtype)
    if T > 4:
        x[4, H // 2] = float("inf")
    q = torch.full((T, H), 0x55, dtype=torch.uint8, device=dev)
    s = torch.full((T,), float("nan"), device=dev)
    ops.esimd_per_token_quant_fp8(x.to(dev), q, s)
    ref_s = torch.clamp_min(x.float().abs().amax(1) / 448.0, 1.0 / (448.0 * 512.0))
    assert torch.equal(s.cpu(), ref_s)
    fin = torch.isfinite(x.float())
    assert torch.equal(q.cpu()[fin], _codes(x, ref_s)[fin])
