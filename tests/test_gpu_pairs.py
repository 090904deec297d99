"""fp16 / bf16 backward on work-groups of two wave groups (alternate stages, sums added in LDS) and on ragged
grids whose splits take their stages in turn, against the fp64 closed form.

Bound: as in test_gpu_short (2 u against the size of both terms of dS); every extra fp32 add is 2^-24.
"""
from __future__ import annotations

import pytest
import torch

import elsa_amd

pytestmark = pytest.mark.gpu
BOUND = {"fp16": 2.0 ** -10, "bf16": 2.0 ** -7}
DT = {"fp16": torch.float16, "bf16": torch.bfloat16}

# pairs with no partials left (one and several 64-key stages per group, an odd stage count, a ragged end), with
# two ranges left, at D = 32, at D = 128 (dq only; one stage for the second group to skip), causal
# D = 128; then split grids in a ragged round and causal grids in both column layouts
SHAPES = [((2, 8, 1024, 64), False), ((8, 3, 577, 64), False), ((5, 8, 513, 64), False), ((4, 3, 1025, 64), False),
          ((9, 4, 640, 32), False), ((1, 2, 60, 128), False), ((1, 4, 1000, 128), True), ((2, 3, 129, 80), False),
          ((2, 8, 2200, 64), False), ((3, 3, 1200, 64), True), ((2, 8, 1100, 64), True),
          # head dims that pad to 64 (staged through registers): pairs with no partials left and with two, a causal
          # split, one range, 8-wave work-groups
          ((8, 3, 577, 40), False), ((4, 3, 1025, 48), False), ((1, 8, 1100, 56), False), ((1, 8, 1100, 56), True),
          ((4, 4, 197, 40), True), ((16, 8, 600, 48), False)]


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("shape,causal", SHAPES)
def test_backward_against_fp64(dt, shape, causal):
    print(f"pairs {dt} {shape} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    q, k, v, do = (torch.randn(shape, generator=g, device="cuda").to(DT[dt]) for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_(True)
    out = elsa_amd.twopass_attention_train(q, k, v, is_causal=causal)
    grads = torch.autograd.grad(out, (q, k, v), do)
    n, c = shape[2], shape[3] ** -0.5
    err, size = [0.0] * 3, [0.0] * 3
    for b in range(shape[0]):  # one batch entry at a time: [H, N, N] in 64 bits
        q64, k64, v64, do64 = (t[b].detach().double() for t in (q, k, v, do))
        s = torch.matmul(q64, k64.transpose(-1, -2).contiguous()) * c
        if causal:
            s = s.masked_fill(torch.ones((n, n), dtype=torch.bool, device="cuda").triu(1), float("-inf"))
        p = torch.softmax(s, -1)
        dsum = p * (do64 * torch.matmul(p, v64)).sum(-1, keepdim=True)
        ds = p * torch.matmul(do64, v64.transpose(-1, -2).contiguous()) - dsum
        dst, dsumt = ds.transpose(-1, -2).contiguous(), dsum.transpose(-1, -2).contiguous()
        want = (torch.matmul(ds, k64) * c, torch.matmul(dst, q64) * c,
                torch.matmul(p.transpose(-1, -2).contiguous(), do64))
        other = ((torch.matmul(dsum, k64) * c).norm(), (torch.matmul(dsumt, q64) * c).norm(), 0.0)
        for i in range(3):
            err[i] += (grads[i][b].double() - want[i]).norm().item() ** 2
            size[i] += (want[i].norm() + other[i]).item() ** 2
    for name, e, sz in zip(("dq", "dk", "dv"), err, size):
        assert (e / sz) ** 0.5 <= BOUND[dt], (name, (e / sz) ** 0.5)


@pytest.mark.parametrize("shape,partials", [((8, 3, 1025, 64), 0), ((2, 8, 1024, 32), 2), ((4, 8, 1024, 32), 0),
                                            ((4, 3, 1025, 64), 2), ((1, 8, 1024, 64), 4)])
def test_backward_allocates_no_partials_that_pairs_do_not_write(shape, partials):
    q, k, v, do = (torch.randn(shape, device="cuda").half() for _ in range(4))
    for t in (q, k, v):
        t.requires_grad_(True)
    for _ in range(2):  # the first pass also loads code and starts the engine
        out = elsa_amd.twopass_attention_train(q, k, v)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        grads = torch.autograd.grad(out, (q, k, v), do)
        peak = torch.cuda.max_memory_allocated() - before
    rows = shape[0] * shape[1] * shape[2]
    # three gradients, three floats per row, the partials; each allocation rounded up to at most 2 MiB
    expect = 3 * q.numel() * 2 + 3 * rows * 4 + 3 * partials * q.numel() * 4
    assert expect <= peak <= expect + (8 << 20), (peak, expect)
    assert all(g.isfinite().all() for g in grads)


@pytest.mark.parametrize("dt", ["fp16", "bf16"])
@pytest.mark.parametrize("shape,bias_bh,causal", [((2, 3, 100, 128), (1, 3), False), ((1, 2, 129, 128), (1, 2), True),
                                                  ((2, 2, 200, 72), (2, 2), False), ((2, 2, 257, 64), (1, 2), True),
                                                  ((3, 2, 130, 40), (1, 1), False), ((1, 4, 520, 128), (1, 4), False),
                                                  ((70, 8, 256, 64), (1, 8), False)])
def test_biased_backward_against_fp64(dt, shape, bias_bh, causal):
    print(f"biased {dt} {shape} {bias_bh} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    q, k, v, do = (torch.randn(shape, generator=g, device="cuda").to(DT[dt]) for _ in range(4))
    n, c = shape[2], shape[3] ** -0.5
    bias = torch.randn((*bias_bh, n, n), generator=g, device="cuda").to(DT[dt])
    ins = [t.requires_grad_(True) for t in (q, k, v, bias)]
    out = elsa_amd.twopass_attention_train(q, k, v, bias=bias, is_causal=causal)
    grads = torch.autograd.grad(out, ins, do)
    q64, k64, v64, do64 = (t.detach().double() for t in (q, k, v, do))
    s = torch.matmul(q64, k64.transpose(-1, -2).contiguous()) * c + bias.detach().double()
    if causal:
        s = s.masked_fill(torch.ones((n, n), dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    dsum = p * (do64 * torch.matmul(p, v64)).sum(-1, keepdim=True)
    ds = p * torch.matmul(do64, v64.transpose(-1, -2).contiguous()) - dsum
    dst, dsumt = ds.transpose(-1, -2).contiguous(), dsum.transpose(-1, -2).contiguous()
    want = [torch.matmul(ds, k64) * c, torch.matmul(dst, q64) * c, torch.matmul(p.transpose(-1, -2).contiguous(), do64)]
    other = [(torch.matmul(dsum, k64) * c).norm(), (torch.matmul(dsumt, q64) * c).norm(), 0.0]
    for dim in (0, 1):
        if bias_bh[dim] == 1:
            ds, dsum = ds.sum(dim, keepdim=True), dsum.sum(dim, keepdim=True)
    for name, got, ex, ot in zip(("dq", "dk", "dv", "dbias"), grads, [*want, ds], [*other, dsum.norm()]):
        rel = ((got.double() - ex).norm() / (ex.norm() + ot)).item()
        assert rel <= BOUND[dt], (name, rel)
