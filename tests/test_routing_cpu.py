"""The planner's and the workspace rules of the C ABI, over shapes where a rule could cost a call its speed, its
memory or its being accepted.  No kernel is launched."""
from __future__ import annotations

import ctypes

import pytest

from elsa_amd import _lib


def _fwd_args(dtype, b, h, n, d, causal=False, summary=None):
    a = _lib.FwdArgs()
    a.q = a.k = a.v = a.out = 16
    a.batch, a.heads, a.seq_len, a.head_dim = b, h, n, d
    a.dtype = dtype
    a.summary_dtype = dtype if summary is None else summary
    a.is_causal = int(causal)
    return a


def _plan(a):
    lib, plan = _lib.load(), _lib.FwdPlan()
    assert lib.elsa_fwd_plan_get(ctypes.byref(a), ctypes.byref(plan)) == _lib.ELSA_OK, lib.elsa_last_error()
    return plan


# B1 d128 bf16 with n / 4 keys per partition against 4096: H1 8K 0.053 against 0.091 ms, H2 0.060 against 0.092, H4 0.101
# against 0.106, H1 12K 0.074 against 0.094; H16 8K 0.335 against 0.315
@pytest.mark.parametrize("h", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n,parts", [(8192, 4), (12288, 4), (16384, 4)])
def test_long_causal_calls_are_cut_in_four_at_every_head_dim(h, n, parts):
    for d in (32, 64, 128):
        plan = _plan(_fwd_args(_lib.ELSA_BF16, 1, h, n, d, causal=True))
        assert (plan.partitions, plan.partition_len) == (parts, n // parts), (d, plan.partitions)


def _accepted(a):
    """Whether elsa_fwd takes the call: elsa_phase1 runs the same checks before that of its row range."""
    lib = _lib.load()
    a.workspace, a.workspace_bytes = 256, 1 << 62
    rc = lib.elsa_phase1(ctypes.byref(a), -1, 1, None)
    msg = lib.elsa_last_error()
    assert rc in (_lib.ELSA_ERR_INVALID, _lib.ELSA_ERR_UNSUPPORTED), msg
    assert (rc == _lib.ELSA_ERR_INVALID) == (b"row range" in msg), msg
    return rc == _lib.ELSA_ERR_INVALID


# rows so far apart that only the shorter partitions of the work-group target span less than 2 GiB
@pytest.mark.parametrize("dtype,b,h,n,d,row", [
    (_lib.ELSA_F32, 1, 3, 4139, 64, 907352), (_lib.ELSA_BF16, 16, 1, 2448, 8, 1661696),
    (_lib.ELSA_F16, 4, 3, 3654, 128, 801496), (_lib.ELSA_F16, 1, 16, 5474, 80, 349656),
    (_lib.ELSA_F32, 2, 8, 2048, 64, 1 << 19), (_lib.ELSA_BF16, 4, 8, 1024, 64, 1 << 20)])
def test_wide_rows_are_cut_into_partitions_below_2_gib(dtype, b, h, n, d, row):
    a = _fwd_args(dtype, b, h, n, d)
    a.q_layout = a.k_layout = a.v_layout = a.out_layout = _lib.Layout(8, 8, row)
    assert _accepted(a)
    size = 4 if dtype == _lib.ELSA_F32 else 2
    assert _plan(a).partition_len * row * size < 1 << 31
    # dense operands of the same shape are not affected, and one partition that spans 2 GiB stays refused
    assert _accepted(_fwd_args(dtype, b, h, n, d))
    a.partition_len = -(-(1 << 31) // (row * size))
    assert a.partition_len > n or not _accepted(a)


def _bwd_workspace(dtype, b, h, n, d, causal=False):
    """(bytes asked for, bytes of D and the two parts of LSE2 alone)"""
    a = _lib.BwdArgs()
    a.batch, a.heads, a.seq_len, a.head_dim = b, h, n, d
    a.dtype, a.is_causal = dtype, int(causal)
    return int(_lib.load().elsa_bwd_workspace_bytes(ctypes.byref(a))), 3 * (-(-b * h * n * 4 // 256) * 256)


@pytest.mark.parametrize("b,h,n,d", [(8, 8, 16385, 128), (8, 16, 16385, 64), (7, 15, 40000, 128), (8, 16, 8193, 128),
                                     (4, 16, 65537, 64)])
def test_large_fp32_backwards_need_no_partials(b, h, n, d):
    # up to 12 GiB of partials for a modelled half percent
    need, rows = _bwd_workspace(_lib.ELSA_F32, b, h, n, d)
    assert need == rows


@pytest.mark.parametrize("b,h,n,d,split", [(2, 8, 4097, 64, 5), (1, 8, 2048, 128, 2), (4, 2, 300, 128, 4)])
def test_ragged_fp32_backwards_keep_their_ranges(b, h, n, d, split):
    need, rows = _bwd_workspace(_lib.ELSA_F32, b, h, n, d)
    assert need == rows + 3 * split * b * h * n * d * 4


def test_fp32_partials_stay_below_512_mib():
    for d in (64, 128):
        for bh in (1, 3, 8, 16, 24, 48, 96, 200, 1000):
            for n in (300, 513, 1025, 2049, 4097, 8193, 16385, 32769):
                for causal in (False, True):
                    need, rows = _bwd_workspace(_lib.ELSA_F32, 1, bh, n, d, causal)
                    assert need - rows <= 512 << 20, (d, bh, n, causal, need)


# fp16 forwards above head dim 64: partitions where they pay for their merge (ms with the count before and after)
@pytest.mark.parametrize("h,n,d,parts", [
    (24, 700, 128, 1),   # 0.0244 with 2, 0.0218
    (24, 513, 128, 2),   # 0.0207 with 3, 0.0181
    (32, 513, 128, 1),   # 0.0222 with 2, 0.0193
    (6, 2048, 80, 4),    # 0.0288 with 2, 0.0270
    (16, 1500, 80, 2),   # 0.0367 with 1, 0.0348
    (8, 1000, 128, 4),   # 0.0287 with 1, 0.0192
    (16, 2048, 128, 1)]) # 0.0577 with 4, 0.0498
def test_wide_head_forward_partitions(h, n, d, parts):
    assert _plan(_fwd_args(_lib.ELSA_F16, 1, h, n, d)).partitions == parts


def test_wide_head_forwards_keep_one_work_group_per_cu_or_partitions_of_512_keys():
    for h in (1, 2, 3, 6, 8, 12, 16, 24, 48):
        for n in (512, 600, 1025, 2048, 4095, 8192):
            for d in (72, 80, 128):
                plan = _plan(_fwd_args(_lib.ELSA_BF16, 1, h, n, d))
                wgs = h * -(-n // plan.block_m) * plan.partitions
                assert plan.partitions == 1 or plan.partition_len >= 512 or (wgs <= 256 and plan.partition_len >= 128)


# causal fp32 backwards above head dim 64, ranges by their own cost (ms with the count before and after)
@pytest.mark.parametrize("h,n,split", [
    (8, 2048, 4),    # 0.363 with 2, 0.249
    (24, 1025, 2),   # 0.348 with 1, 0.242
    (16, 2049, 2),   # 0.600 with 3, 0.472
    (16, 1024, 3),   # 0.205 with 2
    (4, 3000, 5),
    (1, 8192, 8),    # 0.672 with 5, 0.431
    (16, 4097, 1),   # 1.816 with 5, 1.484
    (100, 300, 1), (32, 2048, 1)])
def test_causal_fp32_ranges_above_head_dim_64(h, n, split):
    need, rows = _bwd_workspace(_lib.ELSA_F32, 1, h, n, 128, causal=True)
    assert need == rows + (3 * -(-split * h * n * 128 * 4 // 256) * 256 if split > 1 else 0)
