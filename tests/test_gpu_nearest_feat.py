"""The feature-space `nearest` search through one fp16 product per pair
(csrc/nearest_feat_impl.hpp) against the oracle's play-through of the reference
kernel: the edges of its tiles and of its scans of 4,096 rows, and inputs on
which its bound says little, so that rows are gone through again."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from pytorch_cluster_amd import capi  # noqa: E402
from gpu_common import dev, ragged_ptrs  # noqa: E402


@pytest.fixture(autouse=True)
def always(monkeypatch):
    monkeypatch.setenv("PCA_NEAREST_FEAT", "1")


def check(oracle, x, y, ptr_x=None, ptr_y=None):
    got = capi.nearest_rows(dev(x), dev(y), dev(ptr_x, torch.long),
                            dev(ptr_y, torch.long))
    torch.cuda.synchronize()
    want = oracle.nearest_op(
        x, y, [0, len(x)] if ptr_x is None else ptr_x,
        [0, len(y)] if ptr_y is None else ptr_y)
    assert (got.cpu().numpy() == want).all()


@pytest.mark.parametrize("m", [1, 3, 31, 33, 127, 129, 4095, 4097, 8223])
@pytest.mark.parametrize("n,d", [(1, 17), (127, 9), (129, 40), (400, 64)])
def test_edges_of_tiles_and_scans(oracle, n, m, d):
    rng = np.random.default_rng(n + m)
    check(oracle, rng.standard_normal((n, d)).astype(np.float32),
          rng.standard_normal((m, d)).astype(np.float32))


@pytest.mark.parametrize("d", [9, 16, 17, 32, 47, 64, 65, 96, 100, 112, 127,
                               128])
def test_every_number_of_blocks(oracle, d):
    # (enough rows for the kernel with all sets of queries per wave: the
    # 256 workgroups of the launcher's rule take 512 rows each at most)
    rng = np.random.default_rng(d)
    n, segments = 132000, 40
    x = rng.standard_normal((n, d)).astype(np.float32)
    y = rng.standard_normal((segments * 9, d)).astype(np.float32)
    ptr_x = ragged_ptrs(rng, n, segments)
    check(oracle, x, y, ptr_x, np.arange(segments + 1, dtype=np.int64) * 9)


@pytest.mark.parametrize("d", [12, 64, 128])
def test_duplicates_and_ties(oracle, d):
    # more equal rows than the scan keeps minima
    rng = np.random.default_rng(d)
    pool = rng.integers(-2, 3, (40, d)).astype(np.float32)
    y = pool[rng.integers(0, 40, 6000)]
    x = pool[rng.integers(0, 40, 700)]
    x[::3] += 1
    check(oracle, x, y)


@pytest.mark.parametrize("scale_x,scale_y", [
    (1.0, 2e-4),      # a code book at its start, far smaller than the rows
    (2e-4, 1.0), (1e-15, 1e-15), (1e-22, 1e-22), (1e12, 1e12),
    (1e18, 1.0), (3.0, 1e-30)])
def test_scales(oracle, scale_x, scale_y):
    rng = np.random.default_rng(5)
    x = (scale_x * rng.standard_normal((500, 24))).astype(np.float32)
    y = (scale_y * rng.standard_normal((900, 24))).astype(np.float32)
    check(oracle, x, y)


def test_rows_the_filter_cannot_represent(oracle):
    rng = np.random.default_rng(6)
    x = rng.standard_normal((600, 20)).astype(np.float32)
    y = rng.standard_normal((5000, 20)).astype(np.float32)
    x[3, 4] = np.nan
    x[70, 0] = np.inf
    x[71] = 3e18
    x[200] = 2e19
    y[17, 3] = np.nan
    y[18, 19] = -np.inf
    y[4100] = 3e18
    y[4101] = 2e19
    y[1000] *= 1e6
    check(oracle, x, y)
    check(oracle, x, np.full((40, 20), np.inf, np.float32))
    check(oracle, x, np.zeros((40, 20), np.float32))


# one scan of 4,096 rows and several; a handful of large ones and a third
@pytest.mark.parametrize("factor", [50.0, 3e3, 1e5, 1e9])
@pytest.mark.parametrize("n,m,d", [(700, 4096, 24), (300, 9000, 64),
                                   (135000, 500, 20)])
def test_rows_and_queries_far_larger_than_the_others(oracle, n, m, d, factor):
    rng = np.random.default_rng(m)
    y = rng.standard_normal((m, d)).astype(np.float32)
    x = y[rng.integers(0, m, n)] + 0.5 * rng.standard_normal((n, d))
    x = x.astype(np.float32)
    few_x, few_y, many_x = x.copy(), y.copy(), x.copy()
    few_x[::101] *= np.float32(factor)
    few_y[::333] *= np.float32(factor)
    many_x[::3] *= np.float32(factor)
    if n > 1000:  # (all sets of queries per wave)
        check(oracle, few_x, few_y)
        return
    check(oracle, few_x, y)
    check(oracle, x, few_y)
    check(oracle, few_x, few_y)
    check(oracle, many_x, few_y)
    near = few_y[rng.integers(0, m, n)] + rng.standard_normal((n, d))
    check(oracle, near.astype(np.float32), few_y)
    spread = np.exp(rng.standard_normal((m, 1)) * np.log(factor) / 3)
    wide = (y * spread).astype(np.float32)
    check(oracle, wide[rng.integers(0, m, n)] + x, wide)
    every = (x * factor * 1e9).astype(np.float32)  # (|x|^2 beyond 1e30, too)
    check(oracle, every, y)


@pytest.mark.parametrize("m,d", [(4096, 24), (9000, 64), (4500, 128)])
def test_norms_over_many_magnitudes(oracle, m, d):
    # large rows that a large query of the workgroup could have for its nearest
    # one are left out of the first pass; in the third example every row is one
    rng = np.random.default_rng(m)

    def norms(rows):
        return np.exp(3 * rng.standard_normal((rows, 1)))

    y = rng.standard_normal((m, d)) * norms(m)
    x = rng.standard_normal((700, d)) * norms(700)
    check(oracle, x.astype(np.float32), y.astype(np.float32))
    near = y[rng.integers(0, m, 700)] * (1 + 0.1 * rng.standard_normal((700, d)))
    check(oracle, near.astype(np.float32), y.astype(np.float32))
    y[-40:] = 1e4 * rng.standard_normal((40, d))
    near[-300:] = 1e3 * rng.standard_normal((300, d)) * norms(300)
    check(oracle, near.astype(np.float32), y.astype(np.float32),
          [0, 300, 400, 700], [0, 50, m - 40, m])


@pytest.mark.parametrize("d", [16, 70, 128])
def test_candidates_that_were_not_kept_in_several_scans(oracle, d):
    # dozens of rows within the margin of the nearest one, in the first, the
    # last and the middle 4,096 rows
    rng = np.random.default_rng(d)
    y = (30 + rng.standard_normal((13000, d))).astype(np.float32)
    for at in (100, 5000, 12500):
        y[at:at + 60] = y[at] + (1e-3 * rng.standard_normal((60, d)))
    x = np.concatenate([y[[100, 130, 5001, 5055, 12500, 12530]],
                        30 + rng.standard_normal((200, d))])
    check(oracle, x.astype(np.float32), y)
    check(oracle, np.repeat(x[:3], 70, 0).astype(np.float32), y)


def test_time_with_a_large_row_and_large_queries():
    """One row of a code book a million times the others took 130 times as
    long, a thousandth of the queries ten thousand times the others 35."""
    g = torch.Generator(device="cuda").manual_seed(1)
    y = torch.randn(4096, 64, generator=g, device="cuda")
    x = y[torch.randint(0, 4096, (50000,), generator=g, device="cuda")]
    x = x + 0.5 * torch.randn(50000, 64, generator=g, device="cuda")

    def least(x, y):
        times = []
        for _ in range(6):
            begin, end = (torch.cuda.Event(enable_timing=True)
                          for _ in range(2))
            begin.record()
            capi.nearest_rows(x, y)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    usual = least(x, y)
    large_y, large_x = y.clone(), x.clone()
    large_y[77] *= 1e6
    large_x[::1000] *= 1e4
    assert least(x, large_y) < 5 * usual
    assert least(large_x, y) < 5 * usual


def test_rows_far_from_the_origin(oracle):
    # |x - y|^2 far below the rounding margin of |x|^2 + |y|^2
    rng = np.random.default_rng(7)
    x = (100 + 0.01 * rng.standard_normal((300, 33))).astype(np.float32)
    y = (100 + 0.01 * rng.standard_normal((4500, 33))).astype(np.float32)
    check(oracle, x, y)


def test_rows_at_odd_addresses(oracle):
    rng = np.random.default_rng(8)
    flat = rng.standard_normal(200 * 30 + 1).astype(np.float32)
    x = torch.from_numpy(flat).cuda()[1:].view(200, 30)
    y = rng.standard_normal((333, 30)).astype(np.float32)
    got = capi.nearest_rows(x, dev(y))
    torch.cuda.synchronize()
    want = oracle.nearest_op(flat[1:].reshape(200, 30), y, [0, 200], [0, 333])
    assert (got.cpu().numpy() == want).all()
