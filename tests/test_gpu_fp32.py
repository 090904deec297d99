"""fp32 forward and backward on the bf16 matrix cores (three parts per operand) against the fp64 closed form,
at the edges of their tiles, stages, work-groups and splits.

Bound: a product keeps 2^-24 (rms) of |x y|; S over d and the stage sums are short fp32 chains added over
N / 32 stages, so the relative 2-norm error stays near 2^-24 sqrt(N / 32 + d / 8): below 6e-7 here, where
one fp32 chain over N / 2 steps showed up to 2e-6.
"""
from __future__ import annotations

import pytest
import torch

import elsa_amd

pytestmark = pytest.mark.gpu
BOUND = 6e-7


def _exact(q, k, v, do, bias, causal):
    q, k, v, do = (t.detach().double() for t in (q, k, v, do))
    c = q.shape[-1] ** -0.5
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * c
    if bias is not None:
        s = s + bias.detach().double()
    if causal:
        n = q.shape[-2]
        s = s.masked_fill(torch.ones((n, n), dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    out = torch.matmul(p, v)
    ds = p * (torch.matmul(do, v.transpose(-1, -2).contiguous()) - (do * out).sum(-1, keepdim=True))
    t = ds.transpose(-1, -2).contiguous()
    return [out, torch.matmul(ds, k) * c, torch.matmul(t, q) * c, torch.matmul(p.transpose(-1, -2).contiguous(), do)], ds


def _inputs(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(shape, generator=g, device="cuda") for _ in range(4)]


def _check(q, k, v, do, bias, causal, what):
    print(what, flush=True)
    ins = [t.requires_grad_(True) for t in (q, k, v)] + ([bias.requires_grad_(True)] if bias is not None else [])
    out = elsa_amd.twopass_attention_train(q, k, v, bias=bias, is_causal=causal)
    grads = torch.autograd.grad(out, ins, do)
    want, ds = _exact(q, k, v, do, bias, causal)
    if bias is not None:
        if bias.shape[0] == 1:
            ds = ds.sum(0, keepdim=True)
        if bias.shape[1] == 1:
            ds = ds.sum(1, keepdim=True)
        want.append(ds)
    for name, got, ex in zip(("out", "dq", "dk", "dv", "dbias"), (out, *grads), want):
        rel = ((got.double() - ex).norm() / ex.norm()).item()
        assert rel <= BOUND, (what, name, rel)


# two rows; the edges of a 32-row tile and stage; of the short kernel (64), of 128- and 256-row work-groups;
# few heads (splits) and grids that fill the chip with 8-wave work-groups; head dims below and at each width
SHAPES = [((1, 1, 2, 64), False), ((1, 2, 31, 8), False), ((2, 1, 32, 32), True), ((1, 3, 33, 64), False),
          ((2, 2, 63, 40), True), ((3, 2, 64, 64), False), ((1, 2, 65, 64), True), ((2, 2, 65, 32), False),
          ((1, 1, 64, 128), False), ((1, 2, 127, 72), False), ((1, 2, 129, 128), True), ((2, 3, 255, 64), False),
          ((1, 2, 257, 64), True), ((1, 2, 257, 128), False), ((48, 4, 300, 64), False), ((32, 8, 256, 64), False),
          ((4, 12, 513, 64), True), ((3, 8, 1500, 64), False), ((1, 4, 1025, 64), True), ((2, 4, 600, 80), False)]


@pytest.mark.parametrize("shape,causal", SHAPES, ids=[f"{s}-{'causal' if c else 'full'}" for s, c in SHAPES])
def test_fp32_forward_and_backward_against_fp64(shape, causal):
    q, k, v, do = _inputs(shape, sum(shape))
    _check(q, k, v, do, None, causal, f"fp32 {shape} causal={causal}")


@pytest.mark.parametrize("shape,bias_bh", [((5, 3, 49, 32), (5, 3)), ((700, 2, 49, 32), (1, 2)), ((3, 2, 64, 64), (1, 2)),
                                           ((4, 2, 33, 64), (1, 1)), ((2, 3, 100, 32), (1, 3)), ((2, 2, 200, 64), (2, 2)),
                                           ((1, 2, 40, 128), (1, 2)), ((1, 1, 17, 16), (1, 1))])
@pytest.mark.parametrize("causal", [False, True])
def test_fp32_bias_gradients_against_fp64(shape, bias_bh, causal):
    q, k, v, do = _inputs(shape, sum(shape) + 1)
    n = shape[2]
    bias = torch.randn((*bias_bh, n, n), generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
    _check(q, k, v, do, bias, causal, f"fp32 bias {shape} {bias_bh} causal={causal}")


def test_fp32_operands_of_any_scale():
    # parts are bf16 (exact from 2^-110 on); the logits stay of order one
    for n in (50, 300):
        q, k, v, do = _inputs((1, 2, n, 64), n)
        _check(q * 2.0 ** 60, k * 2.0 ** -60, v * 2.0 ** -40, do * 2.0 ** 30, None, False, f"fp32 scaled N{n}")


def test_fp32_infinite_value_stays_in_its_column():
    for n in (40, 300):
        q, k, v, _ = _inputs((1, 1, n, 64), n)
        ref = elsa_amd.twopass_attention(q, k, v)
        v = v.clone()
        v[0, 0, 7, 5] = float("inf")
        out = elsa_amd.twopass_attention(q, k, v)
        assert (out[..., 5] == float("inf")).all()
        keep = [d for d in range(64) if d != 5]
        assert torch.equal(out[..., keep], ref[..., keep])


def test_fp32_key_at_minus_infinity_drops_out():
    # q > 0 where one key is -inf: its score is -inf, so the others' softmax
    for n in (40, 300):
        q, k, v, do = _inputs((1, 1, n, 64), n)
        q[..., 3] = q[..., 3].abs() + 0.1
        k[0, 0, 9, 3] = float("-inf")
        out = elsa_amd.twopass_attention(q, k, v)
        rest = [i for i in range(n) if i != 9]
        want = torch.softmax(q.double() @ k[:, :, rest].double().transpose(-1, -2).contiguous() / 8, -1) @ v[:, :, rest].double()
        rel = ((out.double() - want).norm() / want.norm()).item()
        assert rel <= BOUND, (n, rel)


@pytest.mark.parametrize("n,d", [(49, 64), (64, 32), (100, 64), (100, 32), (128, 128)])
def test_fp32_values_near_the_largest_do_not_overflow(n, d):
    # a key a little above the maximum of the stages before it must not scale the sums past the fp32 range (64 keys
    # of equal weight, the most in a partition here, stay inside it)
    q = torch.zeros((1, 1, n, d), device="cuda")
    k, v = torch.zeros_like(q), torch.full_like(q, 3.0e36)
    q[..., 0] = d ** 0.5
    k[0, 0, n - 3, 0] = 5.0
    out = elsa_amd.twopass_attention(q, k, v)
    assert ((out.double() / 3.0e36 - 1).abs() <= 1e-6).all()


def test_fp32_infinity_beside_a_large_partner():
    # a product of an infinity and a value past 2^16, whose parts are large too: still the infinity
    for n, d in ((40, 64), (64, 64), (49, 32), (300, 64), (300, 128), (600, 32)):
        q, k, v, do = _inputs((1, 2, n, d), n)
        q[..., 3] = (q[..., 3].abs() + 1) * 2.0 ** 18
        k[..., 3] = k[..., 3] * 2.0 ** -18
        k[:, :, 9, 3] = float("-inf")
        out = elsa_amd.twopass_attention(q, k, v)
        rest = [i for i in range(n) if i != 9]
        ks, vs = k[:, :, rest].double(), v[:, :, rest].double()
        want = torch.softmax(q.double() @ ks.transpose(-1, -2).contiguous() * d ** -0.5, -1) @ vs
        assert ((out.double() - want).norm() / want.norm()).item() <= BOUND, (n, d)
        # the gradient of v: a row of dO that is infinite in one column
        ins = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = elsa_amd.twopass_attention_train(*ins)
        do = do.clone()
        do[:, :, 5, 1] = float("inf")
        dv = torch.autograd.grad(o, ins[2], do)[0]
        cols = [c for c in range(d) if c != 1]
        p = torch.softmax(q.double() @ k.double().nan_to_num(neginf=-1e300).transpose(-1, -2).contiguous() * d ** -0.5, -1)
        want = p.transpose(-1, -2).contiguous() @ do.double()[..., cols]
        assert ((dv[..., cols].double() - want).norm() / want.norm()).item() <= BOUND, (n, d)
        assert (dv[:, :, rest, 1] == float("inf")).all() and not dv[:, :, 9, 1].isfinite().any()


def test_fp32_strided_operands_match_dense_ones():
    qkv = torch.randn((2, 197, 3, 3, 64), device="cuda", generator=torch.Generator(device="cuda").manual_seed(9))
    do = torch.randn((2, 3, 197, 64), device="cuda", generator=torch.Generator(device="cuda").manual_seed(10))
    res = []
    for dense in (False, True):
        q, k, v = (t.contiguous() if dense else t for t in qkv.permute(2, 0, 3, 1, 4).unbind(0))
        q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
        out = elsa_amd.twopass_attention_train(q, k, v)
        res.append((out.detach(), *torch.autograd.grad(out, (q, k, v), do)))
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [1, 9, 31, 32, 33, 49, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_fp32_short_windows_against_fp64(n, causal):
    # one 32-key stage, two, and a ragged second one; more windows than run at once
    q, k, v, do = _inputs((1100, 1, n, 64), n)
    out = elsa_amd.twopass_attention(q, k, v, is_causal=causal)
    ex = _exact(q, k, v, do, None, causal)[0][0]
    assert ((out.double() - ex).norm() / ex.norm()).item() <= BOUND
    bias = torch.randn((1, 1, n, n), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    out = elsa_amd.twopass_attention(q, k, v, bias=bias, is_causal=causal)
    ex = _exact(q, k, v, do, bias, causal)[0][0]
    assert ((out.double() - ex).norm() / ex.norm()).item() <= BOUND
