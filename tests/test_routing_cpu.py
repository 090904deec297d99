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
