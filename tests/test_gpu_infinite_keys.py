"""Backward of a call in which one key holds -inf: its score is -inf for every row (q > 0 there), so it drops out
and its dk and dv are 0, whatever the sequence's remainder in a tile.  One test per kernel family of the backward."""
from __future__ import annotations

import pytest
import torch

import elsa_amd
from gpu_util import TORCH_DT

pytestmark = pytest.mark.gpu


# short kernel; 32- and 64-row stages with every kind of remainder; 8-wave, split and paired grids; d128 with wave groups
@pytest.mark.parametrize("dtype", ["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("shape", [(2, 2, 40, 64), (1, 3, 49, 32), (1, 2, 64, 64), (1, 2, 65, 64), (1, 8, 300, 64),
                                   (2, 2, 200, 40), (8, 3, 577, 64), (1, 2, 300, 128), (1, 2, 40, 128), (2, 2, 129, 80),
                                   (1, 8, 1030, 64), (4, 64, 300, 64), (1, 4, 512, 128), (1, 2, 333, 32)])
@pytest.mark.parametrize("causal", [False, True])
def test_key_at_minus_infinity_gets_no_gradient(dtype, shape, causal):
    print(f"infinite key {dtype} {shape} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    q, k, v, do = (torch.randn(shape, generator=g, device="cuda").to(TORCH_DT[dtype]) for _ in range(4))
    n, j = shape[2], shape[2] // 4
    q[..., 3] = q[..., 3].abs() + 0.1
    k[:, :, j, 3] = float("-inf")
    ins = [t.detach().requires_grad_(True) for t in (q, k, v)]
    out = elsa_amd.twopass_attention_train(*ins, is_causal=causal)
    dq, dk, dv = torch.autograd.grad(out, ins, do)
    assert out.isfinite().all()
    for name, t in (("dk", dk), ("dv", dv)):
        assert t.isfinite().all(), (name, sorted({int(i) for i in (~t.isfinite()).nonzero()[:, 2]})[:8])
        assert (t[:, :, j] == 0).all(), name
    cols = [c for c in range(shape[3]) if c != 3]  # dq[..., 3] is a sum with 0 x inf
    assert dq[..., cols].isfinite().all()
    # the other keys' gradients are those of the call without that key
    if not causal:
        rest = [i for i in range(n) if i != j]
        q64, k64, v64, do64 = q.double(), k[:, :, rest].double(), v[:, :, rest].double(), do.double()
        s = torch.matmul(q64, k64.transpose(-1, -2).contiguous()) * shape[3] ** -0.5
        want = torch.matmul(torch.softmax(s, -1).transpose(-1, -2).contiguous(), do64)
        bound = {"fp16": 2.0 ** -10, "bf16": 2.0 ** -7, "fp32": 2.0 ** -20}[dtype]  # 2 u, as in test_gpu_short
        assert ((dv[:, :, rest].double() - want).norm() / want.norm()).item() <= bound
