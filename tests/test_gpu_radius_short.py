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


# around the length up to which a lane searches by itself, and around one and
# several tiles of 512 rows; short ones in between, queries of several long
# examples in one workgroup, far fewer queries than rows
@pytest.mark.parametrize("d", [1, 2, 3, 4])
@pytest.mark.parametrize("sizes", [
    [256, 257, 3, 511, 512, 513], [40, 300, 0, 300, 1, 290, 7],
    [1, 1535, 64, 1537], [2300]])
def test_long_examples(oracle, d, sizes):
    rng = np.random.default_rng(d + len(sizes))
    ptr = pointers(sizes)
    x = rng.random((ptr[-1], d)).astype(np.float32)
    for r, limit in ((0.1, 32), (0.02, 5), (3.0, 70)):
        check(oracle, x, x, ptr, ptr, r, limit, ignore_same=limit == 32)
    few = pointers([min(n, 11) for n in sizes])
    y = rng.random((few[-1], d)).astype(np.float32)
    check(oracle, x, y, ptr, few, 0.2, 16)
    grid = rng.integers(0, 5, x.shape).astype(np.float32)
    check(oracle, grid, grid, ptr, ptr, 1.0, 1000)  # (distances of r^2 itself)
    check(oracle, grid * 3e4 + 1e6, grid * 3e4 + 1e6, ptr, ptr, 4e4, 9)


@pytest.mark.parametrize("scale", [1e-25, 1e-12, 1e3, 1e14, 3e17])
def test_long_example_at_the_edges_of_fp32(oracle, scale):
    rng = np.random.default_rng(8)
    ptr = pointers([5, 900, 30])
    x = (rng.standard_normal((ptr[-1], 3)) * scale).astype(np.float32)
    x[100], x[150, 1], x[200], x[250, 2] = np.nan, np.inf, 2e38, -np.inf
    x[300:340] = np.float32(3e15)  # |x|^2 beyond 1e30
    x[400] = x[401] = np.float32(1e19)
    for r in (0.3 * scale, 3 * scale, np.inf, 0.0):
        check(oracle, x, x, ptr, ptr, r, 20)


def test_time_of_one_long_example(monkeypatch):
    """Not much more than the kernel that gives an example its workgroups
    (it was 18 times that; the bound leaves room for noise)."""
    sizes = [35] * 300 + [20000]
    ids = dev(ids_of(pointers(sizes)))
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(sum(sizes), 3, generator=g, device="cuda") * 58

    def least():
        times = []
        for _ in range(8):
            begin, end = (torch.cuda.Event(enable_timing=True)
                          for _ in range(2))
            begin.record()
            pca.radius_graph(x, 2.0, ids)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    here = least()
    monkeypatch.setenv("PCA_RADIUS_SHORT", "0")
    assert here < 4 * least()


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
