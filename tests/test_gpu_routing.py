"""Which kernel (by its mangled name) a call runs, at the lines that the launchers' rules draw, and its result on both sides of them."""
from __future__ import annotations

import pytest
import torch

import elsa_amd
from gpu_util import TORCH_DT, kernel_names

pytestmark = pytest.mark.gpu


def _inputs(shape, dtype, count=4):
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    return [torch.randn(shape, generator=g, device="cuda").to(TORCH_DT[dtype]) for _ in range(count)]


def _exact_rows(q, k, v, rows, causal):
    """The forward of some rows of every head in 64 bits."""
    s = torch.matmul(q[:, :, rows].double(), k.double().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    if causal:
        s = s.masked_fill(torch.arange(q.shape[2], device=q.device) > rows.view(-1, 1), float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v.double())


# causal 16-bit forwards: 128-row blocks (one 32-row tile a wave) up to 1024 of them and 6K keys per slot of the chip,
# else 256-row ones
@pytest.mark.parametrize("shape,tiles", [((1, 8, 4096, 64), 1), ((1, 32, 4096, 64), 1), ((1, 33, 4096, 48), 2), ((1, 12, 8192, 64), 1), ((1, 13, 8192, 64), 2),
                                         ((1, 32, 8192, 64), 2), ((1, 24, 8574, 48), 2), ((1, 8, 16383, 64), 2),
                                         ((1, 32, 8192, 32), 1)])
def test_causal_forward_blocks(shape, tiles):
    q, k, v = _inputs(shape, "bf16", 3)
    names = kernel_names(lambda: elsa_amd.twopass_attention(q, k, v, is_causal=True))
    dp = 32 if shape[3] <= 32 else 64
    assert any(f"phase1_half_kernelIDF16bLi{dp}ELi{tiles}ELi4E" in n for n in names), names
    out = elsa_amd.twopass_attention(q, k, v, is_causal=True)
    n = shape[2]
    rows = torch.tensor([0, 1, 127, 128, 255, 256, 511, 512, n // 2, n - 129, n - 2, n - 1], device="cuda")
    ex = _exact_rows(q, k, v, rows, True)
    assert ((out[:, :, rows].double() - ex).norm() / ex.norm()).item() <= 1.2e-2
