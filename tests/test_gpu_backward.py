"""GPU parity of the recompute backward (preprocess + dq kernel + dk/dv kernel), the
row-stats recompute and dbias, through the C ABI, against the oracle and the fp64
closed form.  Shapes follow the reference's tests/test_attention_bwd.py:15-46 and
benchmarks/bwd_grad_correctness.py:11-34 (ViT odd lengths)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import elsa_amd
from elsa_amd.attention_bwd import _dense_bias_backward
from oracle import elsa_oracle as O
from tests.gpu_util import GRAD_TOL, TORCH_DT, assert_parity, describe, dev, host, max_abs, ulp

pytestmark = pytest.mark.gpu


def _run_train(q, k, v, do, dt, **kw):
    qt, kt, vt = (dev(x, dt).requires_grad_(True) for x in (q, k, v))
    out = elsa_amd.twopass_attention_train(qt, kt, vt, **kw)
    out.backward(dev(do, dt))
    torch.cuda.synchronize()
    return out, qt.grad, kt.grad, vt.grad


CASES = [
    ((1, 2, 64, 32), "fp32", False),
    ((1, 2, 64, 32), "fp32", True),
    ((1, 2, 64, 32), "fp16", False),
    ((1, 2, 64, 32), "fp16", True),
    ((2, 3, 1025, 64), "fp32", False),
    ((2, 3, 1025, 64), "fp16", False),
    ((1, 2, 1025, 64), "fp16", True),
    ((1, 2, 197, 64), "fp16", True),
    ((1, 2, 4096, 64), "fp16", False),
    ((1, 2, 4097, 64), "fp16", True),
    ((1, 2, 2049, 64), "fp16", True),   # split into 8 ranges of every eighth stage
    ((1, 4, 2049, 64), "fp16", False),  # 4 ranges of every fourth stage, 33 stages
    ((1, 2, 300, 128), "fp16", False),
    ((1, 2, 300, 128), "fp32", True),
    ((1, 8, 1025, 64), "fp32", True),   # 8 ranges of every eighth stage
    ((1, 3, 197, 64), "bf16", False),
    ((1, 2, 90, 40), "fp32", False),
    ((2, 3, 49, 32), "bf16", True),     # 2-wave work-groups: at most 64 rows, head dims up to 32
    ((4, 3, 49, 24), "fp32", False),
    ((2, 2, 33, 32), "fp16", False),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-{c[1]}-{'causal' if c[2] else 'full'}" for c in CASES])
def test_backward_matches_oracle_and_closed_form(case):
    shape, dt, causal = case
    describe(f"backward {case}")
    q, k, v, do = O.make_inputs(shape, seed=2026 + shape[2], dtype=dt, with_dout=True, dout_scale=1.0)
    out, dq, dk, dv = _run_train(q, k, v, do, dt, is_causal=causal)
    qf, kf, vf, dof = (np.asarray(x, np.float32) for x in (q, k, v, do))
    eq, ek, ev, _ = O.exact_backward(qf, kf, vf, dof, is_causal=causal)
    fo, fm, fz = O.forward(q, k, v, is_causal=causal, dtype=dt, mode="ref")
    rq, rk, rv = O.backward(q, k, v, fo, do, fm, fz, is_causal=causal, dtype=dt, mode="ref")
    for name, got, exp, ref in (("dq", dq, eq, rq), ("dk", dk, ek, rk), ("dv", dv, ev, rv)):
        describe(f"{name} {assert_parity(host(got), exp, ref, GRAD_TOL[dt], name, dt)}")


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("causal", [False, True])
def test_reference_train_test_against_sdpa(dt, causal):
    # tests/test_attention_bwd.py:15-46 (seed 11, q,k x0.5, dO x0.25, atol=rtol 2.5e-3 / 8e-2)
    torch.manual_seed(11)
    shape = (1, 2, 64, 32)
    dtype = torch.float32 if dt == "fp32" else torch.float16
    q = (torch.randn(shape, device="cuda", dtype=dtype) * 0.5).requires_grad_(True)
    k = (torch.randn(shape, device="cuda", dtype=dtype) * 0.5).requires_grad_(True)
    v = torch.randn(shape, device="cuda", dtype=dtype).requires_grad_(True)
    dout = torch.randn(shape, device="cuda", dtype=dtype) * 0.25
    q_ref, k_ref, v_ref = (t.detach().float().cpu().requires_grad_(True) for t in (q, k, v))
    ref = torch.nn.functional.scaled_dot_product_attention(q_ref, k_ref, v_ref, is_causal=causal,
                                                           scale=1.0 / shape[-1] ** 0.5)
    ref.backward(dout.float().cpu())
    out = elsa_amd.twopass_attention_train(q, k, v, is_causal=causal)
    out.backward(dout)
    tol = 2.5e-3 if dt == "fp32" else 8e-2
    torch.testing.assert_close(out.float().cpu(), ref, atol=tol, rtol=tol)
    for a, b in ((q.grad, q_ref.grad), (k.grad, k_ref.grad), (v.grad, v_ref.grad)):
        torch.testing.assert_close(a.float().cpu(), b, atol=tol, rtol=tol)


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
def test_backward_without_saved_state_uses_row_stats(dt):
    describe(f"backward row-stats {dt}")
    q, k, v, do = O.make_inputs((1, 2, 333, 64), seed=4, dtype=dt, with_dout=True, dout_scale=1.0)
    qd, kd, vd, dod = (dev(x, dt) for x in (q, k, v, do))
    out, rm, rz = elsa_amd.twopass_attention_with_state(qd, kd, vd, is_causal=True)
    g_state = elsa_amd.twopass_attention_backward(qd, kd, vd, out, dod, is_causal=True, row_m=rm, row_z=rz)
    g_none = elsa_amd.twopass_attention_backward(qd, kd, vd, out, dod, is_causal=True)
    for a, b in zip(g_state, g_none):  # both fp16/fp32 outputs: one ulp of slack
        ha, hb = host(a), host(b)
        assert (np.abs(ha - hb) - ulp(hb, dt)).max() <= GRAD_TOL[dt]
    from elsa_amd.attention_bwd import _row_stats
    from elsa_amd.attention import _canonical_bias
    m2, z2 = _row_stats(qd, kd, _canonical_bias(None, batch=1, heads=2, seq_len=333, device=qd.device),
                        is_causal=True, scale=1 / 8)
    _, em, ez = O.exact_forward(np.float32(q), np.float32(k), np.float32(v), is_causal=True)
    assert np.abs(host(m2) - em).max() <= 1e-4 * np.abs(em).max()
    np.testing.assert_allclose(host(z2), ez, rtol=1e-4 if dt == "fp32" else 2e-3)


@pytest.mark.parametrize("dt", ["fp32", "fp16"])
@pytest.mark.parametrize("bias_shape", [(1, 3, 49, 49), (4, 3, 49, 49), (49, 49), (3, 49, 49), (4, 1, 49, 49)])
def test_bias_gradients(dt, bias_shape):
    describe(f"backward bias {bias_shape} {dt}")
    shape = (4, 3, 49, 32)
    q, k, v, do = O.make_inputs(shape, seed=9, dtype=dt, with_dout=True, dout_scale=1.0)
    bias = (np.random.default_rng(9).standard_normal(bias_shape) * 0.5).astype(np.float32)
    qt, kt, vt = (dev(x, dt).requires_grad_(True) for x in (q, k, v))
    bt = dev(bias, "fp32").requires_grad_(True)
    out = elsa_amd.twopass_attention_train(qt, kt, vt, bias=bt)
    out.backward(dev(do, dt))
    torch.cuda.synchronize()
    qf, kf, vf, dof = (np.asarray(x, np.float32) for x in (q, k, v, do))
    eq, ek, ev, _ = O.exact_backward(qf, kf, vf, dof, bias=bias)
    eo, em, ez = O.exact_forward(qf, kf, vf, bias=bias)
    edb = O.dbias(qf, kf, vf, eo, dof, em, ez, bias=bias)
    tol = GRAD_TOL[dt]
    fo, fm, fz = O.forward(q, k, v, bias=bias, dtype=dt, mode="ref")
    rq, rk, rv = O.backward(q, k, v, fo, do, fm, fz, bias=bias, dtype=dt, mode="ref")
    for name, got, exp, ref in (("dq", qt.grad, eq, rq), ("dk", kt.grad, ek, rk), ("dv", vt.grad, ev, rv)):
        assert_parity(host(got), exp, ref, tol, name, dt)
    assert bt.grad.shape == bias.shape
    summed = (shape[0] * shape[1]) // int(np.prod(bias_shape[:-2]))  # (b, h) pairs folded into each entry
    rdb = O.dbias(qf, kf, vf, fo, dof, fm, fz, bias=bias, mode="ref")
    assert_parity(host(bt.grad), edb, rdb, tol * summed, "dbias", "fp32")


def test_dbias_causal_matches_closed_form():
    describe("dbias causal")
    q, k, v, do = O.make_inputs((2, 2, 70, 32), seed=12, dtype="fp32", with_dout=True, dout_scale=1.0)
    bias = (np.random.default_rng(12).standard_normal((2, 2, 70, 70)) * 0.3).astype(np.float32)
    qd, kd, vd, dod, bd = (dev(x, "fp32") for x in (q, k, v, do, bias))
    out, rm, rz = elsa_amd.twopass_attention_with_state(qd, kd, vd, bias=bd, is_causal=True)
    db = _dense_bias_backward(qd, kd, vd, out, dod, bias=bd, is_causal=True, row_m=rm, row_z=rz)
    eo, em, ez = O.exact_forward(q, k, v, bias=bias, is_causal=True)
    edb = O.dbias(q, k, v, eo, do, em, ez, bias=bias, is_causal=True)
    fo, fm, fz = O.forward(q, k, v, bias=bias, is_causal=True, dtype="fp32", mode="ref")
    rdb = O.dbias(q, k, v, fo, do, fm, fz, bias=bias, is_causal=True, mode="ref")
    describe(str(assert_parity(host(db), edb, rdb, GRAD_TOL["fp32"], "dbias", "fp32")))


@pytest.mark.parametrize("causal", [False, True])
def test_dbias_beyond_the_reference_dense_limit(causal):
    """B*H*N^2 above the 64M elements where the reference's dense fallback raises
    NotImplementedError (attention_bwd.py:923-924): both dbias routes (the training call's
    dS store and the separate recompute kernel) against the closed form on sampled rows, and
    the sum of every full row against its closed form."""
    b, h, n, d = 1, 2, 5800, 64
    assert b * h * n * n > 64 * 1024 * 1024
    describe(f"dbias beyond 64M elements causal={causal}")
    q, k, v, do = O.make_inputs((b, h, n, d), seed=33, dtype="fp16", with_dout=True, dout_scale=1.0)
    bias = (np.random.default_rng(33).standard_normal((h, n, n)) * 0.3).astype(np.float32)
    qt, kt, vt = (dev(x, "fp16").requires_grad_(True) for x in (q, k, v))
    bt = dev(bias, "fp32").requires_grad_(True)
    out = elsa_amd.twopass_attention_train(qt, kt, vt, bias=bt, is_causal=causal)
    out.backward(dev(do, "fp16"))
    with torch.no_grad():
        o2, rm, rz = elsa_amd.twopass_attention_with_state(qt.detach(), kt.detach(), vt.detach(), bias=bt.detach(),
                                                           is_causal=causal)
        db2 = _dense_bias_backward(qt.detach(), kt.detach(), vt.detach(), o2, dev(do, "fp16"), bias=bt.detach(),
                                   is_causal=causal, row_m=rm, row_z=rz)
    torch.cuda.synchronize()
    rows = np.sort(np.random.default_rng(1).choice(n, 12, replace=False))
    qf, kf, vf, dof = (np.asarray(x, np.float64) for x in (q, k, v, do))
    # D = rowsum(dO * out) with the stored fp16 output, as the reference's preprocess forms it
    # (attention_bwd.py:188-224).  Each full row of dS then sums to
    # sum_j p_ij dp_ij - D_i = dO_i . (out_exact_i - out_i): the closed form on every row.
    o16 = host(o2)
    dd = (dof * o16).sum(-1)
    o_exact = np.empty_like(o16)
    for hi in range(h):
        for r0 in range(0, n, 512):
            r = np.arange(r0, min(n, r0 + 512))
            s = qf[0, hi, r] @ kf[0, hi].T / np.sqrt(d) + bias[hi, r].astype(np.float64)
            if causal:
                s = np.where(np.arange(n)[None, :] <= r[:, None], s, -np.inf)
            p = np.exp(s - s.max(-1, keepdims=True))
            o_exact[0, hi, r] = (p / p.sum(-1, keepdims=True)) @ vf[0, hi]
    row_sum = (dof * (o_exact - o16)).sum(-1)[0]
    for name, got in (("train", bt.grad), ("dense", db2)):
        g = host(got)
        assert g.shape == (h, n, n)
        assert (np.abs(g.sum(-1) - row_sum) <= 1e-3 * np.abs(g).sum(-1) + 1e-6).all(), name
        for hi in range(h):
            s = qf[0, hi, rows] @ kf[0, hi].T / np.sqrt(d) + bias[hi, rows].astype(np.float64)
            if causal:
                s = np.where(np.arange(n)[None, :] <= rows[:, None], s, -np.inf)
            p = np.exp(s - s.max(-1, keepdims=True))
            p /= p.sum(-1, keepdims=True)
            dp = dof[0, hi, rows] @ vf[0, hi].T
            ds = p * (dp - dd[0, hi, rows][:, None])
            # the same fp16 inputs and D: what remains is fp32 arithmetic, far below 0.1% of
            # the largest entry
            assert np.abs(g[hi, rows] - ds).max() <= 1e-3 * np.abs(ds).max(), (name, hi)


@pytest.mark.parametrize("bias_shape", [(1, 3, 49, 49), (49, 49)])
def test_dbias_split_reduction_matches_unsplit_and_closed_form(bias_shape):
    """Swin-like shape (many windows folded into each bias entry): the reduction over the
    broadcast (b, h) pairs is split across work-groups and summed in order."""
    import ctypes

    from elsa_amd import _lib
    from elsa_amd.attention import _canonical_bias
    from elsa_amd.attention_bwd import _bwd_args

    describe(f"dbias split {bias_shape}")
    shape = (64, 3, 49, 32)
    q, k, v, do = O.make_inputs(shape, seed=21, dtype="fp32", with_dout=True, dout_scale=1.0)
    bias = (np.random.default_rng(21).standard_normal(bias_shape) * 0.5).astype(np.float32)
    qd, kd, vd, dod, bd = (dev(x, "fp32") for x in (q, k, v, do, bias))
    out, rm, rz = elsa_amd.twopass_attention_with_state(qd, kd, vd, bias=bd)
    split = _dense_bias_backward(qd, kd, vd, out, dod, bias=bd, is_causal=False, row_m=rm, row_z=rz)
    eo, em, ez = O.exact_forward(q, k, v, bias=bias)
    edb = O.dbias(q, k, v, eo, do, em, ez, bias=bias)
    assert max_abs(host(split), edb) <= 1e-6 * (shape[0] * shape[1]) ** 0.5

    # the same call with only the backward workspace runs unsplit
    lib = _lib.load()
    meta = _canonical_bias(bd, batch=shape[0], heads=shape[1], seq_len=shape[2], device=qd.device)
    bias_b = 1 if meta.stride_b == 0 else shape[0]
    bias_h = 1 if meta.stride_h == 0 else shape[1]
    args = _bwd_args(qd, kd, vd, out, dod, rm, rz, None, None, None, meta, is_causal=False, scale=1 / np.sqrt(32))
    small = int(lib.elsa_bwd_workspace_bytes(ctypes.byref(args)))
    assert int(lib.elsa_dbias_workspace_bytes(ctypes.byref(args), bias_b, bias_h)) > small
    ws = torch.empty(small, dtype=torch.uint8, device=qd.device)
    args.workspace, args.workspace_bytes = ws.data_ptr(), small
    unsplit = torch.empty((bias_b, bias_h, 49, 49), dtype=torch.float32, device=qd.device)
    _lib.check(lib.elsa_dbias(ctypes.byref(args), unsplit.data_ptr(), bias_b, bias_h, _lib.stream_handle(qd.device)),
               "elsa_dbias")
    torch.cuda.synchronize()
    # the same fp32 sums in two orders over the 192 broadcast pairs
    np.testing.assert_allclose(host(split).reshape(-1), host(unsplit).reshape(-1), rtol=1e-5,
                               atol=1e-6 * (shape[0] * shape[1]) ** 0.5)


@pytest.mark.parametrize("dt,n,causal,d,bh", [("fp16", 197, False, 64, (2, 3)), ("bf16", 1025, True, 64, (2, 3)),
                                              ("fp32", 300, False, 64, (2, 3)), ("fp16", 4097, True, 64, (2, 3)),
                                              ("fp16", 49, False, 32, (2, 3)), ("fp16", 300, False, 128, (2, 3)),
                                              # the 8-wave dq and dK/dV kernels, which load Q/dO and K/V
                                              # straight into LDS through the strided rows
                                              ("fp16", 16384, False, 64, (1, 8)), ("bf16", 16384, True, 64, (1, 8))])
def test_strided_backward_is_bitwise_the_dense_one(dt, n, causal, d, bh):
    """q, k, v as views of a fused [B,N,3,H,D] projection, out and dO as [B,N,H,D] memory,
    and dq, dk, dv written into one fused [B,N,3,H,D] gradient: the same bits as the
    backward on dense copies.  The kernels read and write through the layouts, no copy."""
    from elsa_amd.attention import _BiasMeta
    from elsa_amd.attention_bwd import _backward, _with_state

    b, h = bh
    describe(f"strided backward {dt} n={n} causal={causal} d={d}")
    g = torch.Generator().manual_seed(4242 + n)
    qkv = (torch.randn((b, n, 3, h, d), generator=g) * 0.5).to(TORCH_DT[dt]).cuda()
    do_bnhd = torch.randn((b, n, h, d), generator=g).to(qkv.dtype).cuda()
    q, k, v = qkv.permute(2, 0, 3, 1, 4).unbind(0)
    do = do_bnhd.permute(0, 2, 1, 3)
    out, rm, rz = _with_state(q, k, v, is_causal=causal, out_bnhd=True)
    assert out.stride()[1] == d and not out.is_contiguous()
    meta = _BiasMeta(None, 0, 0, 0, 0, False)
    dense = _backward(*(t.contiguous() for t in (q, k, v, out, do)), meta, is_causal=causal, row_m=rm, row_z=rz)
    dqkv = torch.full_like(qkv, float("nan"))
    grads = dqkv.permute(2, 0, 3, 1, 4).unbind(0)
    ret = _backward(q, k, v, out, do, meta, is_causal=causal, row_m=rm, row_z=rz, grads=grads)
    torch.cuda.synchronize()
    assert all(r.data_ptr() == gr.data_ptr() for r, gr in zip(ret, grads))
    for name, a, ref in zip("qkv", grads, dense):
        assert torch.equal(a, ref), f"d{name} differs from the dense backward"
    # the public entry point on the same views (dense outputs)
    pub = elsa_amd.twopass_attention_backward(q, k, v, out, do, is_causal=causal, row_m=rm, row_z=rz)
    for a, ref in zip(pub, dense):
        assert torch.equal(a, ref)


@pytest.mark.parametrize("dt,n,h,causal", [("fp16", 16384, 8, False), ("bf16", 16384, 8, True), ("fp16", 1100, 1, False)])
def test_backward_over_row_ranges_past_2gib_is_bitwise_the_dense_one(dt, n, h, causal):
    """q, k and v as views of [N, S] buffers (heads 64 elements apart within a row) whose N rows span
    2^31 bytes or more: the LDS-direct loads address a 32-bit buffer range, so the backward stages
    K/V and Q/dO through registers there (the 8-wave two-tile dq, the 8-wave one-tile dq and dK/dV
    at 16K, the split 4-wave kernels at N1100).  Both stagings move the same tiles into the same
    LDS layout: the same bits as the backward on dense copies, which runs the LDS-direct kernels."""
    from elsa_amd.attention import _BiasMeta
    from elsa_amd.attention_bwd import _backward, _with_state

    d = 64
    need = -(-(1 << 31) // (2 * n))
    row = max(65536, (need + 63) // 64 * 64)  # n * row * 2 bytes >= 2^31
    assert n * row * 2 >= 1 << 31
    describe(f"backward over {n} rows of stride {row} elements ({n * row * 2 / 2**30:.2f} GiB), {dt} h={h} causal={causal}")
    g = torch.Generator(device="cuda").manual_seed(n + h)
    views = []
    for _ in range(3):
        buf = torch.empty((n, row), dtype=TORCH_DT[dt], device="cuda")
        v = buf.as_strided((1, h, n, d), (n * row, d, row, 1))
        v.copy_(torch.randn((1, h, n, d), generator=g, device="cuda"))
        views.append(v)
    q, k, v = views
    do = torch.randn((1, h, n, d), generator=g, device="cuda").to(TORCH_DT[dt])
    out, rm, rz = _with_state(q, k, v, is_causal=causal)
    meta = _BiasMeta(None, 0, 0, 0, 0, False)
    strided = _backward(q, k, v, out, do, meta, is_causal=causal, row_m=rm, row_z=rz)
    dense = _backward(q.contiguous(), k.contiguous(), v.contiguous(), out, do, meta, is_causal=causal, row_m=rm,
                      row_z=rz)
    torch.cuda.synchronize()
    for name, a, ref in zip("qkv", strided, dense):
        assert torch.isfinite(ref).all()
        assert torch.equal(a, ref), f"d{name} differs from the dense backward"
    del views, q, k, v


def test_strided_backward_with_head_broadcast_inputs():
    """k and v broadcast over heads (zero head stride) are read in place; the gradients
    per head match those of the materialised copies."""
    from elsa_amd.attention import _BiasMeta
    from elsa_amd.attention_bwd import _backward, _with_state

    describe("strided backward, head-broadcast k/v")
    g = torch.Generator().manual_seed(77)
    b, h, n, d = 1, 4, 333, 64
    q = torch.randn((b, h, n, d), generator=g).half().cuda()
    k1 = torch.randn((b, 1, n, d), generator=g).half().cuda()
    v1 = torch.randn((b, 1, n, d), generator=g).half().cuda()
    do = torch.randn((b, h, n, d), generator=g).half().cuda()
    k, v = k1.expand(b, h, n, d), v1.expand(b, h, n, d)
    out, rm, rz = _with_state(q, k, v)
    meta = _BiasMeta(None, 0, 0, 0, 0, False)
    strided = _backward(q, k, v, out, do, meta, is_causal=False, row_m=rm, row_z=rz)
    dense = _backward(q, k.contiguous(), v.contiguous(), out, do, meta, is_causal=False, row_m=rm, row_z=rz)
    torch.cuda.synchronize()
    for a, ref in zip(strided, dense):
        assert torch.equal(a, ref)


@pytest.mark.parametrize("dt,n,bias", [("fp16", 197, False), ("bf16", 49, True), ("fp32", 130, True)])
def test_qkv_attention_train_matches_twopass_attention_train(dt, n, bias):
    """The fused-qkv autograd path (the drop-ins' training path) gives the same output and
    the same q/k/v (and bias) gradients, bit for bit, as twopass_attention_train on the
    unbound views."""
    from elsa_amd.attention_bwd import qkv_attention_train

    b, h, d = 2, 3, 32 if n == 49 else 64
    describe(f"qkv_attention_train {dt} n={n} bias={bias}")
    g = torch.Generator().manual_seed(900 + n)
    tdt = TORCH_DT[dt]
    base = torch.randn((b, n, 3, h, d), generator=g).to(tdt).cuda()
    do = torch.randn((b, h, n, d), generator=g).to(tdt).cuda()
    bias_t = (torch.randn((1, h, n, n), generator=g) * 0.3).to(tdt).cuda() if bias else None

    qkv1 = base.clone().requires_grad_(True)
    bias1 = bias_t.clone().requires_grad_(True) if bias else None
    out1 = qkv_attention_train(qkv1, bias=bias1)
    out1.backward(do)
    qkv2 = base.clone().requires_grad_(True)
    bias2 = bias_t.clone().requires_grad_(True) if bias else None
    q, k, v = qkv2.permute(2, 0, 3, 1, 4).unbind(0)
    out2 = elsa_amd.twopass_attention_train(q, k, v, bias=bias2)
    out2.backward(do)
    torch.cuda.synchronize()
    assert torch.equal(out1, out2)
    assert qkv1.grad.is_contiguous() and torch.equal(qkv1.grad, qkv2.grad)
    if bias:
        assert torch.equal(bias1.grad, bias2.grad)


def test_torch_module_launches_on_the_current_stream():
    """The C++ autograd module enqueues on the stream torch considers current, also inside
    a side-stream context."""
    from elsa_amd import _lib

    mod = _lib.torch_module()
    assert mod.current_stream() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert mod.current_stream() == side.cuda_stream


@pytest.mark.parametrize("dt,bias", [("fp16", False), ("bf16", True)])
def test_cpp_and_python_fused_qkv_paths_agree(dt, bias):
    """qkv_attention_train's C++ autograd function and its Python twin give the same bits."""
    from elsa_amd.attention_bwd import _TwopassQkvAutograd, qkv_attention_train

    describe(f"C++ vs Python fused-qkv autograd {dt} bias={bias}")
    g = torch.Generator().manual_seed(31)
    b, n, h, d = 2, 197, 3, 64
    base = torch.randn((b, n, 3, h, d), generator=g).to(TORCH_DT[dt]).cuda()
    do = torch.randn((b, h, n, d), generator=g).to(TORCH_DT[dt]).cuda()
    bias_t = (torch.randn((1, h, n, n), generator=g) * 0.3).to(TORCH_DT[dt]).cuda() if bias else None
    res = []
    for use_cpp in (True, False):
        qkv = base.clone().requires_grad_(True)
        bt = bias_t.clone().requires_grad_(True) if bias else None
        if use_cpp:
            out = qkv_attention_train(qkv, bias=bt)
        else:
            out = _TwopassQkvAutograd.apply(qkv, bt, False, {}, {})
        out.backward(do)
        res.append((out.detach(), qkv.grad, bt.grad if bias else None))
    torch.cuda.synchronize()
    (o1, g1, b1), (o2, g2, b2) = res
    assert o1.stride() == o2.stride() and torch.equal(o1, o2)
    assert torch.equal(g1, g2)
    if bias:
        assert torch.equal(b1, b2)


@pytest.mark.parametrize("dt,causal,bias", [("fp16", True, False), ("bf16", False, True), ("fp32", False, False)])
def test_cpp_and_python_training_paths_agree(dt, causal, bias):
    """twopass_attention_train's C++ autograd function and its Python twin give the same bits."""
    from elsa_amd.attention_bwd import _TwopassAttentionAutograd

    describe(f"C++ vs Python training autograd {dt} causal={causal} bias={bias}")
    g = torch.Generator().manual_seed(57)
    b, h, n, d = 2, 3, 300, 64
    base = [torch.randn((b, h, n, d), generator=g).to(TORCH_DT[dt]).cuda() for _ in range(3)]
    do = torch.randn((b, h, n, d), generator=g).to(TORCH_DT[dt]).cuda()
    bias_t = (torch.randn((h, n, n), generator=g) * 0.3).to(TORCH_DT[dt]).cuda() if bias else None
    res = []
    for use_cpp in (True, False):
        q, k, v = (t.clone().requires_grad_(True) for t in base)
        bt = bias_t.clone().requires_grad_(True) if bias else None
        if use_cpp:
            out = elsa_amd.twopass_attention_train(q, k, v, bias=bt, is_causal=causal)
        else:
            out = _TwopassAttentionAutograd.apply(q, k, v, bt, causal, {}, {})
        out.backward(do)
        res.append((out.detach(), q.grad, k.grad, v.grad, bt.grad if bias else None))
    torch.cuda.synchronize()
    for a, ref in zip(res[0], res[1]):
        if ref is not None:
            assert torch.equal(a, ref)


@pytest.mark.parametrize("dt,shape,bias_shape,causal", [
    ("fp16", (2, 3, 197, 64), (2, 3, 197, 197), False),   # dbias is dS itself
    ("bf16", (2, 3, 130, 64), (1, 3, 130, 130), True),    # summed over the batch, causal zeros
    ("fp32", (4, 2, 49, 32), (49, 49), False),            # summed over batch and heads
    ("fp16", (8, 3, 49, 32), (8, 1, 49, 49), True),       # summed over heads
    ("fp32", (1, 2, 300, 128), (1, 2, 300, 300), True),   # D = 128
])
def test_bwd_dbias_matches_bwd_then_dbias(dt, shape, bias_shape, causal):
    """elsa_bwd_dbias (dS stored by the dk/dv kernel, summed over the broadcast dims) against
    elsa_bwd followed by elsa_dbias (which recomputes S and dP): the same dq, dk, dv bits and
    the same dbias up to the fp32 summation order."""
    import ctypes

    from elsa_amd import _lib
    from elsa_amd.attention import _canonical_bias
    from elsa_amd.attention_bwd import _bwd_args

    describe(f"elsa_bwd_dbias {dt} {shape} bias {bias_shape} causal={causal}")
    b, h, n, d = shape
    q, k, v, do = O.make_inputs(shape, seed=n + d, dtype=dt, with_dout=True, dout_scale=1.0)
    bias = (np.random.default_rng(n).standard_normal(bias_shape) * 0.5).astype(np.float32)
    qd, kd, vd, dod = (dev(x, dt) for x in (q, k, v, do))
    bd = dev(bias, dt)
    out, rm, rz = elsa_amd.twopass_attention_with_state(qd, kd, vd, bias=bd, is_causal=causal)
    lib = _lib.load()
    meta = _canonical_bias(bd, batch=b, heads=h, seq_len=n, device=qd.device)
    bias_b = 1 if meta.stride_b == 0 else b
    bias_h = 1 if meta.stride_h == 0 else h
    sh = _lib.stream_handle(qd.device)

    def call(fused):
        grads = tuple(torch.full_like(qd, float("nan")) for _ in range(3))
        db = torch.full((bias_b, bias_h, n, n), float("nan"), dtype=torch.float32, device=qd.device)
        args = _bwd_args(qd, kd, vd, out, dod, rm, rz, *grads, meta, is_causal=causal, scale=1 / np.sqrt(d))
        if fused:
            nbytes = int(lib.elsa_bwd_dbias_workspace_bytes(ctypes.byref(args), bias_b, bias_h))
        else:
            nbytes = int(lib.elsa_dbias_workspace_bytes(ctypes.byref(args), bias_b, bias_h))
        ws = torch.empty(nbytes, dtype=torch.uint8, device=qd.device)
        args.workspace, args.workspace_bytes = ws.data_ptr(), nbytes
        if fused:
            _lib.check(lib.elsa_bwd_dbias(ctypes.byref(args), db.data_ptr(), bias_b, bias_h, sh), "elsa_bwd_dbias")
        else:
            _lib.check(lib.elsa_bwd(ctypes.byref(args), sh), "elsa_bwd")
            _lib.check(lib.elsa_dbias(ctypes.byref(args), db.data_ptr(), bias_b, bias_h, sh), "elsa_dbias")
        torch.cuda.synchronize()
        return grads, db

    (g1, db1), (g2, db2) = call(True), call(False)
    for name, a, ref in zip("qkv", g1, g2):
        assert torch.equal(a, ref), f"d{name} differs"
    x, y = host(db1), host(db2)
    assert np.isfinite(x).all()
    pairs = (b * h) // (bias_b * bias_h)
    # two fp32 evaluations of dS: the dk/dv kernel's dP runs over the head dim in one MFMA
    # chain of D/2 steps, the dbias kernel's in four; their rounding grows with sqrt(D / 32)
    chain = max(1.0, d / 32) ** 0.5
    assert np.abs(x - y).max() <= 1e-6 * max(1.0, np.abs(y).max()) * pairs ** 0.5 * chain + 1e-7


# elsa_bwd_stage 0 / 1 / 2 launched one by one (what bench.py times) against elsa_bwd in one call,
# which sums the split backward's dq, dK and dV partials in a single combine launch and, at d = 64,
# runs the preprocess inside the dq kernels: the same bits.
@pytest.mark.parametrize("shape,dt,causal", [((1, 8, 1024, 64), "fp16", False), ((8, 3, 1025, 64), "bf16", False),
                                             ((1, 4, 2048, 64), "fp16", True), ((2, 32, 1024, 64), "fp16", False),
                                             ((1, 8, 16384, 64), "fp16", False), ((1, 8, 8192, 64), "bf16", True),
                                             ((1, 4, 1000, 32), "fp16", False)])
def test_backward_stages_one_by_one_are_the_whole_backward(shape, dt, causal):
    import ctypes
    import math

    from elsa_amd import _lib
    from elsa_amd.attention import _BiasMeta
    from elsa_amd.attention_bwd import _attach_workspace, _bwd_args

    describe(f"backward stages one by one {shape} {dt} causal={causal}")
    lib = _lib.load()
    g = torch.Generator().manual_seed(31)
    q, k, v, do = (torch.randn(shape, generator=g).to(TORCH_DT[dt]).cuda() for _ in range(4))
    out, rm, rz = elsa_amd.twopass_attention_with_state(q, k, v, is_causal=causal)
    grads = []
    for stages in ((-1,), (0, 1, 2)):
        dq, dk, dv = torch.full_like(q, float("nan")), torch.full_like(k, float("nan")), torch.full_like(v, float("nan"))
        ba = _bwd_args(q, k, v, out, do, rm, rz, dq, dk, dv, _BiasMeta(None, 0, 0, 0, 0, False), is_causal=causal,
                       scale=1.0 / math.sqrt(shape[-1]))
        ws = _attach_workspace(lib, ba, q.device)
        for st in stages:
            _lib.check(lib.elsa_bwd_stage(ctypes.byref(ba), st, _lib.stream_handle(q.device)), "elsa_bwd_stage")
        torch.cuda.synchronize()
        grads.append((dq, dk, dv))
        del ws
    for name, a, b in zip(("dq", "dk", "dv"), *grads):
        assert not torch.isnan(a).any() and torch.equal(a, b), name


# The split backward's causal work-groups whose range holds nothing write no partials, and the
# combine skips those ranges and any range that starts past N.  With the workspace filled with NaN
# first, a partial read that no work-group wrote shows up in the gradients, and so does a row's D or
# LSE2 that the dq kernels (the preprocess at d = 64) left unwritten for the dK/dV kernel.
@pytest.mark.parametrize("shape,causal,dt", [((1, 2, 2049, 64), True, "fp16"), ((1, 2, 2049, 64), False, "fp16"),
                                             ((1, 4, 2049, 64), True, "fp16"),
                                             ((1, 8, 2048, 64), True, "fp16"), ((8, 3, 1025, 64), True, "fp16"),
                                             ((1, 2, 4097, 64), True, "fp16"), ((1, 8, 16385, 64), False, "fp16"),
                                             ((1, 8, 8192, 64), True, "fp16"),
                                             # fp32: ranges down to 64 rows, and causal splits that count
                                             # only the work-groups holding work
                                             ((1, 8, 1025, 64), True, "fp32"), ((2, 8, 2049, 64), True, "fp32"),
                                             ((1, 8, 4097, 64), True, "fp32"), ((8, 3, 197, 64), False, "fp32")])
def test_split_backward_reads_only_written_partials(shape, causal, dt):
    import ctypes
    import math

    from elsa_amd import _lib
    from elsa_amd.attention import _BiasMeta
    from elsa_amd.attention_bwd import _attach_workspace, _bwd_args

    describe(f"split backward over a NaN workspace {shape} causal={causal} {dt}")
    lib = _lib.load()
    g = torch.Generator().manual_seed(32)
    q, k, v, do = (torch.randn(shape, generator=g).to(TORCH_DT[dt]).cuda() for _ in range(4))
    out, rm, rz = elsa_amd.twopass_attention_with_state(q, k, v, is_causal=causal)
    want = elsa_amd.twopass_attention_backward(q, k, v, out, do, is_causal=causal, row_m=rm, row_z=rz)
    dq, dk, dv = (torch.full_like(x, float("nan")) for x in (q, k, v))
    ba = _bwd_args(q, k, v, out, do, rm, rz, dq, dk, dv, _BiasMeta(None, 0, 0, 0, 0, False), is_causal=causal,
                   scale=1.0 / math.sqrt(shape[-1]))
    ws = _attach_workspace(lib, ba, q.device)
    ws[: ws.numel() // 4 * 4].view(torch.float32).fill_(float("nan"))
    _lib.check(lib.elsa_bwd_stage(ctypes.byref(ba), -1, _lib.stream_handle(q.device)), "elsa_bwd_stage")
    torch.cuda.synchronize()
    for name, a, b in zip(("dq", "dk", "dv"), (dq, dk, dv), want):
        assert not torch.isnan(a).any(), name
        assert torch.equal(a, b), name


def test_two_tile_dq_with_large_row_sums():
    """D = rowsum(O * dO) far past fp16's range (|D| ~ 5e5: dO ~ 8000 N(0,1), v ~ 8 + N(0,1)) in the
    two-tile dq (B2 H64 N1024 fills its 512-row work-groups), where -D enters dP through an MFMA
    operand in fp16 parts: finite gradients within fp16 rounding of the reference restatement."""
    from oracle import torch_scan as T

    shape = (2, 64, 1024, 64)
    describe(f"two-tile dq with |D| past fp16 range {shape}")
    g = torch.Generator().manual_seed(41)
    q = (torch.randn(shape, generator=g) * 0.5).half()
    k = (torch.randn(shape, generator=g) * 0.5).half()
    v = (8.0 + torch.randn(shape, generator=g)).half()
    do = (torch.randn(shape, generator=g) * 8000.0).half()
    qd, kd, vd, dod = (x.cuda() for x in (q, k, v, do))
    out, rm, rz = elsa_amd.twopass_attention_with_state(qd, kd, vd)
    dq, dk, dv = elsa_amd.twopass_attention_backward(qd, kd, vd, out, dod, row_m=rm, row_z=rz)
    torch.cuda.synchronize()
    dd = (out.float() * dod.float()).sum(-1)
    assert dd.abs().max().item() > 1e5  # the case this test is for
    heads = [0, 127]
    flat = lambda x: x.reshape(1, 128, 1024, 64)[:, heads]  # noqa: E731
    rq, rk, rv = T.backward(flat(q), flat(k), flat(v), flat(out.cpu()).float(), flat(do), rm.cpu()[heads],
                            rz.cpu()[heads], dtype="fp16", row_chunk=512)
    for name, got, ref in (("dq", dq, rq), ("dk", dk, rk), ("dv", dv, rv)):
        gg = flat(got.float().cpu()).double()
        rr = ref.double()
        assert torch.isfinite(gg).all(), name
        err = ((gg - rr).abs().max() / rr.abs().max()).item()
        describe(f"  {name} max |got - ref| / max |ref| = {err:.2e}")
        assert err <= 2e-3, (name, err)
