"""CPU model of the fp32 kernels' products: x = h + m + l in bf16 parts and the six partial products of
order 2^-16 and above (split3_any, split3_reg and mma3_small in elsa_mfma.h)."""
from __future__ import annotations

import numpy as np
import pytest


def _bf16_rne(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32)


def _bf16_trunc(x):
    return (np.asarray(x, np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)


def _split(x, truncate_h):
    f = np.where(np.isinf(x), np.sign(x), x).astype(np.float32)  # an infinity goes to the last part, beside +-1
    h = _bf16_trunc(f) if truncate_h else _bf16_rne(f)
    m = _bf16_rne(f - h)
    r = (x - h) - m
    return h, m, np.where(np.isfinite(x), _bf16_rne(r), r)


@pytest.mark.parametrize("truncate_h", [True, False])
def test_three_parts_hold_every_bit(truncate_h):
    rng = np.random.default_rng(5)
    x = (rng.standard_normal(200_000) * 2.0 ** rng.integers(-100, 100, 200_000)).astype(np.float32)
    h, m, l = _split(x, truncate_h)
    assert np.array_equal(h.astype(np.float64) + m + l, x.astype(np.float64))


@pytest.mark.parametrize("truncate_h", [True, False])
def test_parts_of_small_values_end_at_bf16s_smallest_subnormal(truncate_h):
    rng = np.random.default_rng(9)
    x = (rng.standard_normal(100_000) * 2.0 ** rng.integers(-126, -90, 100_000)).astype(np.float32)
    h, m, l = _split(x, truncate_h)
    err = np.abs(h.astype(np.float64) + m + l - x)
    assert err.max() <= 2.0 ** -134
    assert err[np.abs(x) >= 2.0 ** -110].max() == 0 and err.max() > 0


def test_infinities_stay_in_the_last_part_and_the_largest_values_finite():
    x = np.array([np.inf, -np.inf, np.finfo(np.float32).max, -np.finfo(np.float32).max, 0.0], np.float32)
    h, m, l = _split(x, True)
    assert np.isfinite(h).all() and np.isfinite(m).all()
    assert np.array_equal(np.isinf(l), np.isinf(x))
    fin = np.isfinite(x)
    assert np.array_equal(h[fin].astype(np.float64) + m[fin] + l[fin], x[fin].astype(np.float64))


def test_products_with_an_infinity_are_the_fp32_ones():
    rng = np.random.default_rng(7)
    b = (rng.standard_normal(1000) * 2.0 ** rng.integers(-20, 14, 1000)).astype(np.float32)
    for a in (np.inf, -np.inf):
        ah, am, al = _split(np.full(1000, a, np.float32), True)
        for truncate_b, y in ((True, b), (False, np.clip(np.abs(b), 0, 256).astype(np.float32))):
            # operands are truncated; probabilities, at most 2^8, are rounded
            bh, bm, bl = _split(y, truncate_b)
            with np.errstate(over="ignore"):
                got = al * bh + ah * bl + am * bm + am * bh + ah * bm + ah * bh
            assert np.array_equal(got, np.float32(a) * y)


def test_products_with_an_infinity_hold_for_every_partner():
    rng = np.random.default_rng(8)
    y = (rng.standard_normal(4000) * 2.0 ** rng.integers(-120, 127, 4000)).astype(np.float32)
    y = np.concatenate([y, np.array([np.inf, -np.inf, np.finfo(np.float32).max], np.float32)])
    bh, bm, bl = _split(y, True)
    for a in (np.inf, -np.inf):
        ah, am, al = _split(np.full(len(y), a, np.float32), True)
        got = al * bh + ah * bl + am * bm + am * bh + ah * bm + ah * bh
        assert np.array_equal(got, np.float32(a) * y)


@pytest.mark.parametrize("truncate_a,truncate_b", [(True, True), (True, False), (False, False)])
def test_dropped_products_are_below_an_fp32_rounding(truncate_a, truncate_b):
    rng = np.random.default_rng(6)
    a, b = (rng.standard_normal(400_000).astype(np.float32) for _ in range(2))
    ah, am, al = (t.astype(np.float64) for t in _split(a, truncate_a))
    bh, bm, bl = (t.astype(np.float64) for t in _split(b, truncate_b))
    kept = al * bh + ah * bl + am * bm + am * bh + ah * bm + ah * bh
    err = np.abs(kept - a.astype(np.float64) * b) / np.abs(a.astype(np.float64) * b)
    # |m| < 2^-7 |x| and |l| <= 2^-16 |x| (h truncated): m l' + l m' + l l' < 2 * 2^-23 + 2^-32
    assert err.max() < 2.0 ** -22
    assert np.sqrt((err ** 2).mean()) < 2.0 ** -24
