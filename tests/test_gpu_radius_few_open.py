"""The matrix-core radius search where most queries of a workgroup are full
early and the others go on by a wave each (csrc/radius_mc_impl.hpp), against
the oracle: numbers of open queries around the switch and the waves' shares,
rows around a tile and a wave, every compiled dimension."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from gpu_common import gpu_radius  # noqa: E402


@pytest.fixture(autouse=True)
def always(monkeypatch):
    monkeypatch.setenv("PCA_RADIUS_MATRIX_CORES", "1")
    monkeypatch.setenv("PCA_RADIUS_SHORT", "0")


def check(oracle, x, y, ptr_x, ptr_y, r, limit, ignore_same=False):
    want = oracle.radius_op(x, y, ptr_x, ptr_y, r, limit,
                            ignore_same_index=ignore_same)
    got = gpu_radius(x, y, ptr_x, ptr_y, r, limit, ignore_same)
    assert got.shape == want.shape and (got == want).all()


@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("open_queries", [1, 3, 4, 5, 31, 32, 33, 60])
def test_open_queries(oracle, d, open_queries):
    rng = np.random.default_rng(d * 100 + open_queries)
    n = 3 * 1024 + 65
    # rows near the origin, some near (3, ...): few and late, some nowhere
    x = (0.1 * rng.random((n, d))).astype(np.float32)
    x[1500::97] += 3
    y = (0.1 * rng.random((140, d))).astype(np.float32)
    far = rng.permutation(128)[:open_queries]
    y[far] += 3
    y[far[::3]] += 3
    ptr_x, ptr_y = [0, n], [0, 140]
    for limit in (1, 5, 20, 200):
        check(oracle, x, y, ptr_x, ptr_y, 1.0, limit)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 256, 1023, 1024, 1025, 2100])
@pytest.mark.parametrize("m", [1, 32, 33, 129, 160])
def test_few_queries_from_the_start(oracle, n, m):
    rng = np.random.default_rng(n + m)
    x = rng.random((n, 3)).astype(np.float32)
    y = rng.random((m, 3)).astype(np.float32)
    for r, limit in ((0.3, 32), (2.0, 70), (0.05, 3)):
        check(oracle, x, y, [0, n], [0, m], r, limit)


def test_clustered_graph(oracle):
    rng = np.random.default_rng(5)
    sizes = [5000, 0, 1300, 2500]
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    centres = rng.random((12, 3))
    x = (centres[rng.integers(0, 12, ptr[-1])]
         + 0.02 * rng.standard_normal((ptr[-1], 3))).astype(np.float32)
    x[7], x[1200, 1], x[6000] = np.nan, np.inf, 3e38
    for r, limit in ((0.05, 32), (0.02, 8), (0.1, 64), (np.inf, 16)):
        check(oracle, x, x, ptr, ptr, r, limit, ignore_same=True)


@pytest.mark.parametrize("d", [2, 3, 4, 8])
@pytest.mark.parametrize("share", [0.002, 0.03, 0.06, 0.3, 1.0])
def test_open_queries_by_share_of_rows_in_reach(oracle, d, share):
    """Few neighbours (rows shared by the waves), many (query by query), and
    the one after the other, at ends of a wave's rows and of a round."""
    rng = np.random.default_rng(int(share * 1000) + d)
    for n, m in ((31, 5), (513, 32), (2047, 17), (2049, 4), (6500, 29)):
        x = rng.random((n, d)).astype(np.float32)
        near = rng.random(n) < np.where(np.arange(n) < n // 2, share / 8, share)
        x[~near] += 5
        y = rng.random((m, d)).astype(np.float32)
        y[::7] += 5
        y[m // 2, d - 1] = np.nan
        k = min(n, m)
        x[:k:3] = y[:k:3]
        for limit in (7, 100, 3000):
            check(oracle, x, y, [0, n], [0, m], 0.5 * d ** 0.5, limit,
                  ignore_same=limit == 100)


@pytest.mark.parametrize("rows", [1, 31, 33, 511, 512, 513, 1025, 1999, 2047])
@pytest.mark.parametrize("d", [3, 6])
def test_last_rows_of_the_open_queries(oracle, rows, d):
    """Rounds that end inside a wave's rows or leave less than a wave's: the last
    row in reach of one query, of all, of none; lists that are full early."""
    rng = np.random.default_rng(rows + d)
    for round_rows in (2048, 4096):
        n = round_rows + rows
        for m in (5, 32):
            x = (0.2 * rng.random((n, d)) + 3).astype(np.float32)
            y = rng.random((m, d)).astype(np.float32)
            x[rng.integers(0, n, 40)] = y[rng.integers(0, m, 40)]
            for last in (y[m - 1], y.mean(0), np.full(d, 9)):
                x[-1] = last
                for r, limit in ((0.01, 32), (1.0, 4), (1.0, 32), (9.0, 60)):
                    check(oracle, x, y, [0, n], [0, m], r, limit)
