"""CPU model of the fp16 filter of the feature-space `nearest` search
(pytorch_cluster_amd/csrc/nearest_feat_impl.hpp): a row at distance D -- as the
reference's scalar loop computes it (csrc/cuda/nearest_cuda.cu:36-43) -- must
have a filter value s that is not above the cut for D, whatever constants the
rows and the workgroup's queries give the bound.

The model rounds as the kernels do (numpy float16, the same flush, the scales'
powers of two) and adds the products up in float64, i.e. without the matrix
cores' own accumulation error; the test therefore demands that the share of the
bound reserved for that, d + 16 terms of 2^-22 of |kappa| |a|^2 + 1.01 |a| |2 b|,
is left over.
"""
import math

import numpy as np
import pytest

from helpers import stable_seed
from test_filter_bounds import h, inv_sigma

LARGE_ROW = 4096.0
LARGE_EXPONENTS = 12


def distances(x, y):
    """[rows, queries], one fused multiply-add per component."""
    acc = np.zeros((len(x), len(y)), dtype=np.float32)
    with np.errstate(over="ignore", invalid="ignore"):
        for c in range(x.shape[1]):
            t = (x[:, None, c] - y[None, :, c]).astype(np.float32)
            acc = (t.astype(np.float64) ** 2 + acc).astype(np.float32)
    return acc


def squares(v):
    return (v.astype(np.float64) ** 2).sum(1)


def rows_of_x(x):
    """nf_rows: typical norm, limit and scale of the operands."""
    sq = squares(x)
    some = sq[sq > 0]
    if len(some) == 0:
        return 1.0, 1e36, 16.0 * inv_sigma(0)
    mean = 2.0 ** (0.5 * np.log2(some).mean())
    limit = min(mean * LARGE_ROW, 1e18)
    top = np.abs(x[sq > 0]).max()
    return (min(math.sqrt(some.mean()), 2.0 * mean), limit ** 2,
            16.0 * inv_sigma(min(top, limit)))


def exponent(v):
    return int((np.float32(v).view(np.uint32) >> 23) & 0xff)


def check(x, y):
    """One workgroup with the queries y against the rows x; returns the largest
    margin of a pair, as a share of |a|^2 + |b|^2."""
    x = np.ascontiguousarray(x, dtype=np.float32)
    y = np.ascontiguousarray(y, dtype=np.float32)
    d = x.shape[1]
    typical, limit_sq, s_c = rows_of_x(x)
    tops = np.abs(y).max(1)
    exps = [exponent(t) for t in tops if t != 0]
    mean = int(sum(exps) / len(exps)) if exps else 127
    ours = np.array([exponent(t) <= mean + LARGE_EXPONENTS for t in tops])
    assert ours.any()
    y = y[ours]  # (the others are searched exactly)
    s_q = 8.0 * inv_sigma(np.abs(y).max())
    a = x.astype(np.float64) * s_c
    b = y.astype(np.float64) * s_q
    large = squares(x) > limit_sq
    ha = h(np.where(large[:, None], 0.0, a))
    hb = h(-2.0 * b)
    ysq = squares(b)
    top_sq = ysq.max()
    r = s_q / s_c
    A = typical * s_c
    if not 2.0 ** -10 < A < 1e7:
        A = 1.0
    largest = math.sqrt(top_sq) + 1e-3
    ordinary = 2.0 * math.sqrt(d) * 2.0 ** (max(mean, 1) - 127) * s_q
    if largest > ordinary:
        largest = math.sqrt(largest * ordinary)
    largest = max(largest, 1e-3)
    lam = largest / A
    eps = 2.0 ** -10 + (d + 20) * 2.0 ** -21
    delta = (d + 20) * 2.0 ** -21
    root_d = math.sqrt(d) * 1.01
    kappa = r * (1.0 - delta) - eps * lam - root_d / (32768.0 * A)
    asq = squares(a)
    start = asq * kappa
    # a large row
    gain, loss = 0.24 * r * asq, 1.01 * top_sq / r
    start[large] = (np.where(gain >= loss, gain, 0.0) - loss)[large]
    start = np.minimum(start, 1e37)
    s = start[:, None] + ha @ hb.T
    dist = distances(x, y).astype(np.float64)
    per_sq = (eps / lam - 1.0 / r +
              (d + 6) * (1.0 / r + eps / lam) * 2.0 ** -24)
    cut = (s_c * s_q * (dist + d * 5.7e-45) * (1.0 + (d + 6) * 2.0 ** -24) +
           ysq * per_sq + root_d * np.sqrt(ysq) / 8192.0 +
           root_d * A / 32768.0 + d * 2.0 ** -27)
    norm_a, norm_b = np.sqrt(asq), np.sqrt(ysq)
    spare = (d + 16) * 2.0 ** -22 * (
        abs(kappa) * asq[:, None] + 1.01 * norm_a[:, None] * 2.0 * norm_b)
    spare[large] = 0.0
    finite = np.isfinite(dist) & (dist < 1e38)
    slack = cut - (s + spare)
    assert (slack[finite] >= 0).all(), slack[finite].min()
    scale = r * asq[:, None] + ysq / r + 1e-30
    return float((slack / scale)[finite].max())


@pytest.mark.parametrize("d", [9, 17, 64, 96, 128])
def test_random_rows(d):
    rng = np.random.default_rng(stable_seed("nearest", d))
    x = rng.standard_normal((700, d))
    y = x[rng.integers(0, 700, 200)] + 0.5 * rng.standard_normal((200, d))
    # (and the cut is not far above what it has to be)
    assert check(x, y) < 0.02
    check(np.maximum(x, 0), np.maximum(y, 0))
    check(x + 10, y + 10)
    check(x, x[:200])  # distances of zero


@pytest.mark.parametrize("d", [16, 128])
def test_rounding_midpoints_with_one_sign(d):
    # every component half a unit above an fp16 number, rows and queries alike,
    # so that the roundings of a product add up
    rng = np.random.default_rng(stable_seed("midpoints", d))
    steps = rng.integers(0, 1024, (300, d))
    for shift in (0.5, -0.5 + 2.0 ** -12):
        v = (1.0 + (steps + shift) / 1024.0) * 2.0 ** rng.integers(
            -3, 1, (300, d))
        check(v, v[:100])
        check(v, -v[:100])
        check(v, v[:100] * np.float32(0.5))


@pytest.mark.parametrize("scale_x,scale_y", [
    (1.0, 1e-4), (1e-4, 1.0), (1e-15, 1e-15), (1e12, 1e12), (1e9, 1.0),
    (1.0, 1e9)])
def test_scales(scale_x, scale_y):
    rng = np.random.default_rng(stable_seed("scales", scale_x, scale_y))
    check(scale_x * rng.standard_normal((400, 24)),
          scale_y * rng.standard_normal((150, 24)))


@pytest.mark.parametrize("factor", [30.0, 1e3, 1e5, 1e8])
@pytest.mark.parametrize("d", [12, 64])
def test_rows_and_queries_far_larger_than_the_others(d, factor):
    rng = np.random.default_rng(stable_seed("large", d, factor))
    x = rng.standard_normal((600, d))
    y = x[rng.integers(0, 600, 200)] + 0.5 * rng.standard_normal((200, d))
    few = x.copy()
    few[::150] *= factor
    check(few, y)
    check(few, few[rng.integers(0, 600, 200)] + rng.standard_normal((200, d)))
    loud = y.copy()
    loud[::50] *= factor
    check(x, loud)
    check(few, loud)
    many = y.copy()
    many[::3] *= factor
    check(x, many)
    spread = np.exp(rng.standard_normal((600, 1)) * math.log(factor) / 3)
    check(x * spread, y * spread[:200])


def test_zeros_and_the_flush_limit():
    rng = np.random.default_rng(stable_seed("zeros"))
    x = rng.standard_normal((300, 20))
    x[::3] = 0
    y = rng.standard_normal((100, 20))
    y[::4] = 0
    check(x, y)
    check(np.zeros((10, 20)), y)
    check(x, np.zeros((10, 20)))
    # components around 2^-14 after scaling, beside one of full size
    x = rng.standard_normal((300, 20)) * 2.0 ** -24
    x[:, 0] = rng.standard_normal(300)
    check(x, x[:100] + 2.0 ** -25)
