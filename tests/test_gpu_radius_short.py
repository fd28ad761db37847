"""The radius search of many short examples, one lane per query
(csrc/radius_short.hip), against the oracle: examples around a round of eight
rows and a wave, one far longer than the others, ids and pointers, examples
without rows, ids beyond the number of examples, limits, rows without a
distance."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import pytorch_cluster_amd as pca  # noqa: E402
from pytorch_cluster_amd import capi  # noqa: E402
from gpu_common import dev, gpu_radius  # noqa: E402


@pytest.fixture(autouse=True)
def always(monkeypatch):
    monkeypatch.setenv("PCA_RADIUS_SHORT", "1")


def ids_of(ptr):
    return np.repeat(np.arange(len(ptr) - 1), np.diff(ptr)).astype(np.int64)


def check(oracle, x, y, ptr_x, ptr_y, r, limit, ignore_same=False):
    want = oracle.radius_op(x, y, ptr_x, ptr_y, r, limit,
                            ignore_same_index=ignore_same)
    got = gpu_radius(x, y, ptr_x, ptr_y, r, limit, ignore_same)
    assert got.shape == want.shape and (got == want).all()
    if len(ptr_x) > 2:
        got = capi.radius_edges(dev(x), dev(y), dev(ids_of(ptr_x)),
                                dev(ids_of(ptr_y)), r, limit, ignore_same,
                                ids_examples=len(ptr_x) - 1)
        assert (got.cpu().numpy() == want).all()


def pointers(sizes):
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)


@pytest.mark.parametrize("d", [1, 2, 3, 4])
@pytest.mark.parametrize("smallest,largest,examples", [
    (0, 1, 70), (1, 9, 400), (7, 9, 1), (60, 70, 65), (0, 300, 40),
    (5, 65, 1000)])
def test_sizes(oracle, d, smallest, largest, examples):
    rng = np.random.default_rng(d * 100 + largest)
    ptr_x = pointers(rng.integers(smallest, largest + 1, examples))
    ptr_y = pointers(rng.integers(smallest, largest + 1, examples))
    if ptr_x[-1] == 0 or ptr_y[-1] == 0:
        pytest.skip("no rows")
    x = rng.random((ptr_x[-1], d)).astype(np.float32)
    y = rng.random((ptr_y[-1], d)).astype(np.float32)
    for r, limit in ((0.3, 32), (2.0, 7), (0.5, 1000)):
        check(oracle, x, y, ptr_x, ptr_y, r, limit)
    check(oracle, x, x, ptr_x, ptr_x, 0.6, 16, ignore_same=True)


@pytest.mark.parametrize("longest", [1024, 1025, 3000])
def test_one_long_example(oracle, longest):
    rng = np.random.default_rng(longest)
    ptr = pointers([3, 10, longest, 0, 40, 1])
    x = rng.random((ptr[-1], 3)).astype(np.float32)
    for r, limit in ((0.2, 32), (0.05, 4), (2.0, 100)):
        check(oracle, x, x, ptr, ptr, r, limit, ignore_same=True)


def test_rows_without_a_distance(oracle):
    rng = np.random.default_rng(4)
    ptr = pointers([9, 30, 64, 17])
    x = rng.integers(0, 3, (ptr[-1], 3)).astype(np.float32)
    x[5], x[12], x[40] = np.nan, np.inf, 3e38
    check(oracle, x, x, ptr, ptr, 1.0, 5)
    check(oracle, x, x, ptr, ptr, np.inf, 50)
    check(oracle, x, x, ptr, ptr, 0.0, 5)


def test_examples_the_call_was_not_told_of(oracle):
    # the number of examples as an earlier call met it is too small, then too
    # large
    rng = np.random.default_rng(6)
    for examples in (3, 500, 20):
        ptr = pointers(rng.integers(1, 30, examples))
        x = rng.random((ptr[-1], 3)).astype(np.float32)
        want = oracle.radius_op(x, x, ptr, ptr, 0.4, 8, ignore_same_index=True)[::-1]
        got = pca.radius_graph(dev(x), 0.4, dev(ids_of(ptr)),
                               max_num_neighbors=8)
        assert (got.cpu().numpy() == want).all()


def test_ids_beyond_the_number_of_examples():
    # such queries search the last example, such rows of x are in none
    x = torch.arange(12, dtype=torch.float32, device="cuda")[:, None]
    ids = torch.tensor([0] * 4 + [1] * 4 + [2] * 4, device="cuda")
    got = pca.radius(x, x, 100.0, ids, ids, batch_size=2).cpu()
    rows = [[q, c] for q in range(12) for c in (range(4) if q < 4
                                                else range(4, 8))]
    assert got.t().tolist() == rows
