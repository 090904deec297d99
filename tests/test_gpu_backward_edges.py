"""Rows without a key, rows whose keys are all pushed down alike, and operands past 2 GiB at head dim 128, through the
backward's kernels, against the fp64 closed form.

Bounds as in test_gpu_short: 2 u (u = 2^-11 fp16, 2^-8 bf16; 2^-20 for fp32), dq, dk and dbias against the size of both
terms of dS."""
from __future__ import annotations

import pytest
import torch

import elsa_amd
from gpu_util import TORCH_DT, kernels_run

pytestmark = pytest.mark.gpu
BOUND = {"fp16": 2.0 ** -10, "bf16": 2.0 ** -7, "fp32": 2.0 ** -20}


def _closed_form(q, k, v, do, bias, causal):
    """out, dq, dk, dv, dS and the size of dS's second term; rows without a key give zeros."""
    q, k, v, do = (t.detach().double() for t in (q, k, v, do))
    c = q.shape[-1] ** -0.5
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * c + bias.detach().double()
    if causal:
        n = q.shape[-2]
        s = s.masked_fill(torch.ones((n, n), dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    p = torch.softmax(s, -1).nan_to_num(0.0)
    out = torch.matmul(p, v)
    dsum = p * (do * out).sum(-1, keepdim=True)
    ds = p * torch.matmul(do, v.transpose(-1, -2).contiguous()) - dsum
    t, u = (x.transpose(-1, -2).contiguous() for x in (ds, dsum))
    grads = [torch.matmul(ds, k) * c, torch.matmul(t, q) * c, torch.matmul(p.transpose(-1, -2).contiguous(), do)]
    other = [(torch.matmul(dsum, k) * c).norm(), (torch.matmul(u, q) * c).norm(), 0.0]
    return out, grads, ds, other, dsum


# the short kernel with each destination of dS; 4- and 8-wave 16-bit kernels; fp32 4-wave ones; head dims to 128
@pytest.mark.parametrize("dtype", ["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("shape,bias_bh", [((5, 3, 49, 32), (1, 3)), ((3, 2, 64, 64), (3, 2)), ((2, 2, 33, 40), (1, 1)),
                                           ((2, 3, 100, 64), (1, 3)), ((1, 2, 300, 64), (1, 2)), ((1, 2, 130, 128), (1, 2)),
                                           ((2, 2, 40, 128), (2, 2)), ((48, 8, 256, 64), (1, 8)), ((2, 2, 200, 32), (2, 2))])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_without_a_key(dtype, shape, bias_bh, causal):
    print(f"masked rows {dtype} {shape} {bias_bh} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    q, k, v, do = (torch.randn(shape, generator=g, device="cuda").to(TORCH_DT[dtype]) for _ in range(4))
    n = shape[2]
    bias = torch.randn((*bias_bh, n, n), generator=g, device="cuda").to(TORCH_DT[dtype])
    rows = sorted({0, 7, 31, 32, n // 2, n - 1} & set(range(n)))
    bias[:, :, rows] = float("-inf")          # no key at all
    bias[:, :, 5, : n - 1] = float("-inf")    # only the last key, which a causal mask takes too
    if dtype == "fp16":
        bias[:, :, 6] = torch.finfo(torch.float16).min  # every key alike: the plain softmax
    bias[:, :, :, 11] = float("-inf")         # a key that no row has
    ins = [t.requires_grad_(True) for t in (q, k, v, bias)]
    out = elsa_amd.twopass_attention_train(q, k, v, bias=bias, is_causal=causal)
    grads = torch.autograd.grad(out, ins, do)
    ex, want, ds, other, dsum = _closed_form(q, k, v, do, bias, causal)
    for dim in (0, 1):
        if bias_bh[dim] == 1:
            ds, dsum = ds.sum(dim, keepdim=True), dsum.sum(dim, keepdim=True)
    assert ((out.double() - ex).norm() / ex.norm()).item() <= BOUND[dtype]
    for name, got, w, ot in zip(("dq", "dk", "dv", "dbias"), grads, [*want, ds], [*other, dsum.norm()]):
        assert got.isfinite().all(), name
        rel = ((got.double() - w).norm() / (w.norm() + ot)).item()
        assert rel <= BOUND[dtype], (name, rel)
    dq, dk, dv, db = grads
    assert (out[:, :, rows] == 0).all() and (dq[:, :, rows] == 0).all() and (db[:, :, rows] == 0).all()
    assert (dk[:, :, 11] == 0).all() and (dv[:, :, 11] == 0).all() and (db[..., 11] == 0).all()


@pytest.mark.parametrize("dtype,causal", [("fp16", False), ("bf16", True)])
def test_head_dim_128_over_rows_past_2_gib(dtype, causal):
    """Rows that span 2^31 bytes or more: dk/dv on the kernel that loads through registers, since a buffer range holds
    less; the call on dense copies takes the one with wave groups.  The two agree to the rounding of their outputs."""
    n, d = 1100, 128
    row = -(-(1 << 31) // (2 * n) // 64) * 64 + 64
    assert n * row * 2 >= 1 << 31
    g = torch.Generator(device="cuda").manual_seed(5)
    print(f"head dim 128 past 2 GiB {dtype} causal={causal}", flush=True)

    def wide():
        t = torch.empty((n, row), dtype=TORCH_DT[dtype], device="cuda").as_strided((1, 2, n, d), (n * row, d, row, 1))
        return t.copy_(torch.randn((1, 2, n, d), generator=g, device="cuda"))

    q, k, v, do = wide(), wide(), wide(), torch.randn((1, 2, n, d), generator=g, device="cuda").to(TORCH_DT[dtype])
    res = []
    for dense in (False, True):
        ins = [(t.contiguous() if dense else t).detach().requires_grad_(True) for t in (q, k, v)]
        out = elsa_amd.twopass_attention_train(*ins, is_causal=causal)
        run = dict(kernels_run(lambda: torch.autograd.grad(out, ins, do, retain_graph=True)))
        assert ("bwd_dkdv_d128_kernel" in run) == dense and ("bwd_dkdv_half_kernel" in run) != dense, run
        res.append(torch.autograd.grad(out, ins, do))
    for name, a, b in zip(("dq", "dk", "dv"), *res):
        assert b.isfinite().all()
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() <= 2 * BOUND[dtype], name
