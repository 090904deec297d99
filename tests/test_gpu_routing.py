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


# head dims above 64: dk/dv in two wave groups from 65 rows, dq (its kernel's last template argument) from 129
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("shape,causal,groups,dq_groups", [
    ((2, 3, 64, 128), False, False, 1), ((2, 3, 20, 72), True, False, 1), ((1, 2, 64, 80), True, False, 1),
    ((2, 3, 65, 128), False, True, 1), ((1, 2, 65, 72), True, True, 1), ((1, 2, 128, 128), True, True, 1),
    ((2, 3, 128, 80), False, True, 1), ((2, 3, 129, 128), False, True, 2), ((1, 2, 129, 96), True, True, 2)])
def test_head_dim_128_backward(dtype, shape, causal, groups, dq_groups):
    q, k, v, do = _inputs(shape, dtype)
    for t in (q, k, v):
        t.requires_grad_(True)
    out = elsa_amd.twopass_attention_train(q, k, v, is_causal=causal)
    names = kernel_names(lambda: torch.autograd.grad(out, (q, k, v), do, retain_graph=True))
    assert any("bwd_dkdv_d128_kernel" in x for x in names) == groups, names
    assert any("bwd_dkdv_half_kernel" in x for x in names) != groups, names
    assert any("bwd_dq_half_kernel" in x and f"Lb0ELi{dq_groups}EE" in x for x in names), names
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), do)
    c, (q64, k64, v64, do64) = shape[3] ** -0.5, (t.detach().double() for t in (q, k, v, do))
    s = torch.matmul(q64, k64.transpose(-1, -2).contiguous()) * c
    if causal:
        s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    dsum = p * (do64 * torch.matmul(p, v64)).sum(-1, keepdim=True)
    ds = p * torch.matmul(do64, v64.transpose(-1, -2).contiguous()) - dsum
    want_k, want_v = (torch.matmul(a.transpose(-1, -2).contiguous(), b) for a, b in ((ds, q64 * c), (p, do64)))
    want_q, other_q = torch.matmul(ds, k64 * c), torch.matmul(dsum, k64 * c)
    other = torch.matmul(dsum.transpose(-1, -2).contiguous(), q64 * c)
    bound = {"fp16": 2.0 ** -10, "bf16": 2.0 ** -7}[dtype]  # 2 u, dq and dk against the size of both terms of dS
    assert ((dq.double() - want_q).norm() / (want_q.norm() + other_q.norm())).item() <= bound
    assert ((dk.double() - want_k).norm() / (want_k.norm() + other.norm())).item() <= bound
    assert ((dv.double() - want_v).norm() / want_v.norm()).item() <= bound
