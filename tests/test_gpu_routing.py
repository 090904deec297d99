"""Which kernel a call runs, at the lines that the launchers' rules draw, and its result on both sides of them."""
from __future__ import annotations

import pytest
import torch

import elsa_amd
from gpu_util import TORCH_DT, kernels_run

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
    run = kernels_run(lambda: elsa_amd.twopass_attention(q, k, v, is_causal=True))
    want = ["bf16", 32 if shape[3] <= 32 else 64, tiles, 4]
    assert any(name == "phase1_half_kernel" and args[:4] == want for name, args in run), run
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
    run = dict(kernels_run(lambda: torch.autograd.grad(out, (q, k, v), do, retain_graph=True)))
    assert ("bwd_dkdv_d128_kernel" in run) == groups and ("bwd_dkdv_half_kernel" in run) != groups, run
    assert run["bwd_dq_half_kernel"][1] == 128 and run["bwd_dq_half_kernel"][-1] == dq_groups, run
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


# fp32 forwards: 4 or 8 waves by the rounds of the chip (partitions by the planner)
@pytest.mark.parametrize("shape,waves", [((1, 96, 100, 64), 4), ((1, 48, 300, 64), 4), ((1, 24, 513, 64), 4),
                                         ((8, 3, 1025, 64), 8), ((1, 8, 4096, 64), 8), ((1, 16, 257, 128), 4),
                                         ((1, 48, 257, 128), 4), ((1, 200, 197, 128), 8), ((1, 8, 2048, 128), 8)])
def test_fp32_forward_waves(shape, waves):
    q, k, v = _inputs(shape, "fp32", 3)
    run = dict(kernels_run(lambda: elsa_amd.twopass_attention(q, k, v)))
    assert run["phase1_x3_kernel"][:2] == [shape[3], waves], run
    out = elsa_amd.twopass_attention(q, k, v)
    rows = torch.unique(torch.tensor([0, 31, 32, 99, shape[2] // 2, shape[2] - 1], device="cuda"))
    ex = _exact_rows(q, k, v, rows, False)
    assert ((out[:, :, rows].double() - ex).norm() / ex.norm()).item() <= 6e-7
