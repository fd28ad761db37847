"""The kNN search of small calls, one wave per query (csrc/knn_wave.hip),
against the oracle: numbers of rows around a round of 1,024 and a lane's share,
more candidates than a wave sorts at once, ties, ragged examples."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from pytorch_cluster_amd import capi  # noqa: E402
from gpu_common import dev, gpu_knn, oracle_knn_edges, ragged_ptrs  # noqa: E402


@pytest.fixture(autouse=True)
def always(monkeypatch):
    monkeypatch.setenv("PCA_KNN_WAVE", "1")


def check(oracle, x, y, ptr_x, ptr_y, k):
    e, d = gpu_knn(x, y, ptr_x, ptr_y, k)
    px = [0, len(x)] if ptr_x is None else ptr_x
    py = [0, len(y)] if ptr_y is None else ptr_y
    want, dist = oracle_knn_edges(oracle, x, y, px, py, k)
    assert e.shape == want.shape and (e == want).all()
    assert (d == dist).all()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 3100])
@pytest.mark.parametrize("d,k", [(1, 1), (2, 5), (3, 17), (4, 33), (3, 64)])
def test_numbers_of_rows(oracle, n, d, k):
    rng = np.random.default_rng(n + k)
    check(oracle, rng.random((n, d)).astype(np.float32),
          rng.random((37, d)).astype(np.float32), None, None, k)


@pytest.mark.parametrize("segments", [1, 2, 64, 65, 66, 300, 5000])
def test_ragged_examples(oracle, segments):
    rng = np.random.default_rng(segments)
    x = rng.random((6000, 3)).astype(np.float32)
    y = rng.random((700, 3)).astype(np.float32)
    ptr_x = ragged_ptrs(rng, 6000, segments)
    ptr_y = ragged_ptrs(rng, 700, segments)
    if segments == 1:
        ptr_x = ptr_y = None
    check(oracle, x, y, ptr_x, ptr_y, 9)
    # graph options, example ids in place of pointers
    if segments > 1:
        ids = dev(np.repeat(np.arange(segments), np.diff(ptr_x)))
        got, _ = capi.knn_edges(dev(x), dev(x), ids, ids, 6, drop_self=True,
                                x_first=True, ids_examples=segments)
        _, col, _ = oracle.knn_dense(x, x, ptr_x, ptr_x, 6, False, fma_mode=1)
        col = col.reshape(6000, 6)
        keep = (col != -1) & (col != np.arange(6000)[:, None])
        rows = np.broadcast_to(np.arange(6000)[:, None], (6000, 6))[keep]
        assert (got.cpu().numpy() == np.stack([col[keep], rows])).all()


def test_candidates_on_one_lane_and_ties(oracle):
    # all near rows 64 apart: they fall to one lane, whose 16 rows the bound
    # from the other lanes lets through together with theirs
    rng = np.random.default_rng(3)
    x = (50 + rng.random((2048, 3))).astype(np.float32)
    x[::64] = rng.random((32, 3))
    check(oracle, x, rng.random((20, 3)).astype(np.float32), None, None, 24)
    # hundreds of equal distances, lowest rows first
    x = rng.integers(0, 2, (3000, 3)).astype(np.float32)
    check(oracle, x, x[:50].copy(), None, None, 64)
    check(oracle, np.zeros((2000, 3), np.float32), x[:5].copy(), None, None,
          40)


def test_rows_without_a_distance(oracle):
    rng = np.random.default_rng(4)
    x = rng.random((1200, 3)).astype(np.float32)
    x[5] = np.nan
    x[6] = np.inf
    x[100:1100] = 2e5  # beyond the limit of 1e10
    y = rng.random((9, 3)).astype(np.float32)
    y[2, 1] = np.nan
    y[3, 0] = -np.inf
    for k in (3, 64):
        check(oracle, x, y, None, None, k)


def test_graph_of_more_queries_than_the_compaction_adds_up(oracle):
    # beyond 8,192 queries the edges are counted in a launch of their own
    rng = np.random.default_rng(5)
    sizes = rng.integers(1, 400, 60)
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(ptr[-1])
    assert n > 8192
    x = rng.integers(0, 6, (n, 3)).astype(np.float32)
    got, _ = capi.knn_edges(dev(x), dev(x), dev(ptr), dev(ptr), 7,
                            drop_self=True, x_first=True)
    _, col, _ = oracle.knn_dense(x, x, ptr, ptr, 7, False, fma_mode=1)
    col = col.reshape(n, 7)
    keep = (col != -1) & (col != np.arange(n)[:, None])
    rows = np.broadcast_to(np.arange(n)[:, None], (n, 7))[keep]
    assert (got.cpu().numpy() == np.stack([col[keep], rows])).all()
