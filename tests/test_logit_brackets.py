"""The logit brackets of the whole-row passes (x_floor and x_ceil of
csrc/ls_sampling.hip, restated): no logit outside them has a p on the other
side of the value, subnormal p included. p is monotone in the logit, so the
neighbours of the two brackets decide."""

import math

import numpy as np
import pytest

from oracle import sampling as osmp

H = 2.0 ** -150       # half of the smallest subnormal
SLACK = 2.0 ** -10    # octaves, for the relative roundings


def x_floor(soft, cd, v):
    e = float(soft.s) * (v - H) - H
    if not e > 0.0:
        return np.float32(-np.inf)
    return np.nextafter(np.float32((math.log2(e) - SLACK + float(soft.mcmax)) / cd), np.float32(-np.inf))


def x_ceil(soft, cd, v):
    e = float(soft.s) * (v - H) + H
    return np.nextafter(np.float32((math.log2(e) + SLACK + float(soft.mcmax)) / cd), np.float32(np.inf))


@pytest.mark.parametrize("n,x0,temperature", [(1, 0.0, 1.0), (1, 11.3, 0.31), (3, -2.7, 1.0), (7, 300.0, 2.0),
                                              (2048, 0.5, 0.7), (9000, 4.0, 1.3)])
def test_brackets_over_subnormal_and_normal_p(n, x0, temperature):
    """n equal largest logits (S = n) at several temperatures."""
    pr = osmp.process_logits(np.full(n, x0, dtype=np.float32), temperature)
    soft = osmp.softmax_row(pr)
    ulps = [1, 2, 3, 5, 255, 256, 257, 511, 512, 768, 1024, 1536, 2048, 3 << 8, 7 << 10, 1 << 19, 5 << 19, 1 << 20]
    values = [u * 2.0 ** -149 for u in ulps] + [2.0 ** -126, 1.5 * 2.0 ** -120, 2.0 ** -60, 1e-6, 1e-3, 0.99 / n]
    below, above = [], []
    for v in values:
        lo, hi = x_floor(soft, pr.cd, v), x_ceil(soft, pr.cd, v)
        assert lo <= hi, v
        below.append(np.nextafter(lo, np.float32(-np.inf)))
        above.append(np.nextafter(hi, np.float32(np.inf)))
    values = np.array(values)
    assert np.all(osmp.p_of(soft, np.array(below, dtype=np.float32)).astype(np.float64) < values)
    assert np.all(osmp.p_of(soft, np.array(above, dtype=np.float32)).astype(np.float64) >= values)


def test_half_a_subnormal_ulp_below_the_value():
    """p = 256 * 2^-149 at the logits whose power of two is 255.5 .. 256 of it:
    a relative slack of 1e-3 octaves would leave most of them out."""
    pr = osmp.process_logits(np.zeros(1, dtype=np.float32), 1.0)
    soft = osmp.softmax_row(pr)
    x = np.float32(math.log(255.6 * 2.0 ** -149))
    assert osmp.p_of(soft, np.array([x]))[0] == np.float32(256 * 2.0 ** -149)
    assert x >= x_floor(soft, pr.cd, 256 * 2.0 ** -149)
    assert float(x) < (math.log2(256 * 2.0 ** -149) - 1e-3) / pr.cd
