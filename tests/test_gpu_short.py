"""The one-launch backward of sequences of at most 64 rows against the fp64 closed form and against the staged
kernels (elsa_bwd_stage), over its edges: one and two 32-row tiles, padded head dims, each dS destination.

Bounds: an output rounded to the type is within u / sqrt(3) of it (rms); P and dS are rounded once more each
before their product.  2 u (u = 2^-11 fp16, 2^-8 bf16, and 2^-21 for the fp32 sums) holds all of them; the two
routes differ by at most twice that.  dS = p (dP - D) is a difference whose terms carry those roundings (D that of
the stored output), so dq, dk and dbias are measured against the size of both terms' products: at two rows the
terms nearly cancel and the difference alone would say nothing.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

import elsa_amd
from elsa_amd import _lib
from elsa_amd.attention import _canonical_bias
from elsa_amd.attention_bwd import _bwd_args

pytestmark = pytest.mark.gpu
BOUND = {"fp16": 2.0 ** -10, "bf16": 2.0 ** -7, "fp32": 2.0 ** -20}
DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

CASES = [((1, 1, 2, 8), None, False), ((2, 3, 31, 32), None, True), ((3, 2, 32, 64), (1, 2), False),
         ((2, 2, 33, 40), (2, 2), True), ((5, 3, 49, 32), (5, 3), False), ((400, 3, 49, 32), (1, 3), False),
         ((300, 4, 64, 64), (1, 4), True), ((4, 6, 64, 32), (1, 1), False), ((3, 2, 63, 64), (3, 1), False),
         ((6, 2, 64, 64), None, False), ((2, 3, 16, 16), (1, 3), True)]


def _rel(a, b, other=0.0):
    return ((a.double() - b.double()).norm() / (b.double().norm() + other)).item()


@pytest.mark.parametrize("dt", ["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("shape,bias_bh,causal", CASES)
def test_short_backward(dt, shape, bias_bh, causal):
    print(f"short backward {dt} {shape} bias={bias_bh} causal={causal}", flush=True)
    b, h, n, d = shape
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    q, k, v, do = (torch.randn(shape, generator=g, device="cuda").to(DT[dt]) for _ in range(4))
    bias = None if bias_bh is None else torch.randn((*bias_bh, n, n), generator=g, device="cuda").to(DT[dt])
    ins = [t.requires_grad_(True) for t in (q, k, v)] + ([] if bias is None else [bias.requires_grad_(True)])
    out = elsa_amd.twopass_attention_train(q, k, v, bias=bias, is_causal=causal)
    grads = torch.autograd.grad(out, ins, do)

    q64, k64, v64, do64 = (t.detach().double() for t in (q, k, v, do))
    c = d ** -0.5
    s = torch.matmul(q64, k64.transpose(-1, -2).contiguous()) * c
    if bias is not None:
        s = s + bias.detach().double()
    if causal:
        s = s.masked_fill(torch.ones((n, n), dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    o64 = torch.matmul(p, v64)
    dsum = p * (do64 * o64).sum(-1, keepdim=True)
    ds = p * torch.matmul(do64, v64.transpose(-1, -2).contiguous()) - dsum
    dst = ds.transpose(-1, -2).contiguous()
    other = {"dq": (torch.matmul(dsum, k64) * c).norm(), "dv": 0.0,
             "dk": (torch.matmul(dsum.transpose(-1, -2).contiguous(), q64) * c).norm()}
    want = [torch.matmul(ds, k64) * c, torch.matmul(dst, q64) * c,
            torch.matmul(p.transpose(-1, -2).contiguous(), do64)]
    if bias is not None:
        for dim, size in ((0, bias_bh[0]), (1, bias_bh[1])):
            if size == 1:
                ds, dsum = ds.sum(dim, keepdim=True), dsum.sum(dim, keepdim=True)
        want.append(ds)
        other["dbias"] = dsum.norm()
    for name, got, ex in zip(("dq", "dk", "dv", "dbias"), grads, want):
        assert _rel(got, ex, other[name]) <= BOUND[dt], (name, _rel(got, ex, other[name]))

    # the staged kernels on the same call
    lib = _lib.load()
    qd, kd, vd = (t.detach() for t in (q, k, v))
    o, rm, rz = elsa_amd.twopass_attention_with_state(qd, kd, vd, bias=None if bias is None else bias.detach(),
                                                      is_causal=causal)
    meta = _canonical_bias(None if bias is None else bias.detach(), batch=b, heads=h, seq_len=n, device=q.device)
    outs = [torch.full_like(qd, float("nan")) for _ in range(3)]
    args = _bwd_args(qd, kd, vd, o, do, rm, rz, *outs, meta, is_causal=causal, scale=c)
    ws = torch.empty(int(lib.elsa_bwd_workspace_bytes(ctypes.byref(args))), dtype=torch.uint8, device="cuda")
    args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
    for stage in (0, 1, 2):
        _lib.check(lib.elsa_bwd_stage(ctypes.byref(args), stage, _lib.stream_handle(q.device)), "elsa_bwd_stage")
    torch.cuda.synchronize()
    for name, got, ex in zip(("dq", "dk", "dv"), grads, outs):
        assert _rel(got, ex, other[name]) <= 2 * BOUND[dt], (name, _rel(got, ex, other[name]))


def test_short_backward_is_the_same_from_run_to_run():
    q, k, v, do = (torch.randn((300, 3, 49, 32), device="cuda", dtype=torch.float16) for _ in range(4))
    bias = torch.randn((1, 3, 49, 49), device="cuda", dtype=torch.float16, requires_grad=True)
    for t in (q, k, v):
        t.requires_grad_(True)
    runs = []
    for _ in range(3):
        out = elsa_amd.twopass_attention_train(q, k, v, bias=bias)
        runs.append(torch.autograd.grad(out, (q, k, v, bias), do))
    for r in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], r))


def test_default_calls_match_calls_with_a_knob():
    """A call with default options skips the Python checks where its operands are plain; the same call with a
    knob that changes nothing (phase1_warps) goes through them: the same bits, and what they refuse stays refused."""
    g = torch.Generator(device="cuda").manual_seed(4)
    base = torch.randn((2, 50, 3, 3, 32), generator=g, device="cuda").half()
    views = {"dense": lambda t: t.contiguous(), "strided": lambda t: t, "odd": lambda t: t[..., :20],
             "misaligned": lambda t: t.contiguous().reshape(-1)[4:4 + 2 * 3 * 48 * 32].view(2, 3, 48, 32)}
    for name, view in views.items():
        q, k, v = (view(t) for t in base.permute(2, 0, 3, 1, 4).unbind(0))
        n = q.shape[2]
        for bias in (None, torch.randn((1, 3, n, n), generator=g, device="cuda").half(),
                     torch.randn((3, n, n), generator=g, device="cuda"),
                     torch.randn((1, 3, n, n), generator=g, device="cuda").double(),
                     torch.randn((2, 1, 1, n), generator=g, device="cuda").half().expand(2, 1, n, n)):
            for causal in (False, True):
                a = elsa_amd.twopass_attention(q, k, v, bias=bias, is_causal=causal)
                b = elsa_amd.twopass_attention(q, k, v, bias=bias, is_causal=causal, phase1_warps=4)
                assert torch.equal(a, b), name
                ins = [t.detach().clone(memory_format=torch.preserve_format).requires_grad_(True) for t in (q, k, v)]
                x = elsa_amd.twopass_attention_train(*ins, bias=bias, is_causal=causal)
                y = elsa_amd.twopass_attention_train(*ins, bias=bias, is_causal=causal, phase1_warps=4)
                gx, gy = (torch.autograd.grad(o, ins, torch.ones_like(o)) for o in (x, y))
                assert torch.equal(x, y) and all(torch.equal(s, t) for s, t in zip(gx, gy)), name
    q = base.permute(2, 0, 3, 1, 4)[0]
    for bad, err in (((q, q[:, :, :20], q), "identical shapes"), ((q, q.float(), q), "one dtype"),
                     ((q.double(),) * 3, "supported dtypes"), ((q, q.cpu(), q), "one device"), ((q[0],) * 3, "B,H,N,D")):
        for call in (elsa_amd.twopass_attention, elsa_amd.twopass_attention_train):
            with pytest.raises(ValueError, match=err):
                call(*bad)
    with pytest.raises(ValueError, match="bias"):
        elsa_amd.twopass_attention(q, q, q, bias=torch.zeros((2, 3, 49, 50), device="cuda"))
