"""``nearest`` and ``fps`` given example ids: pointers, checks and numbers of
samples from the device (csrc/segments.hip), against the operators that take
pointers and against torch's arithmetic."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import pytorch_cluster_amd as pca  # noqa: E402
from gpu_common import dev  # noqa: E402


def pointers(sizes):
    return np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)


def ids_of(ptr):
    return np.repeat(np.arange(len(ptr) - 1), np.diff(ptr)).astype(np.int64)


# (numbers of examples that make the guess from the call before too small and
# too large; 0: examples without rows on both sides)
@pytest.mark.parametrize("examples,low,high,d", [
    (5, 1, 60, 3), (700, 1, 9, 3), (1, 40, 40, 2), (64, 0, 5, 3),
    (3, 900, 3000, 64), (9, 20000, 40000, 3)])
def test_nearest_by_id(examples, low, high, d):
    rng = np.random.default_rng(examples)
    sizes = rng.integers(low, high + 1, examples)
    sizes[-1] = max(sizes[-1], 1)
    ptr_x = pointers(sizes)
    ptr_y = pointers((sizes + 3) // 4)
    x = dev(rng.random((ptr_x[-1], d)).astype(np.float32))
    y = dev(rng.random((ptr_y[-1], d)).astype(np.float32))
    want = torch.ops.torch_cluster.nearest(x, y, dev(ptr_x), dev(ptr_y))
    got = pca.nearest(x, y, dev(ids_of(ptr_x)), dev(ids_of(ptr_y)))
    assert (got == want).all()
    # int32 ids, every other entry of a longer vector
    strided = dev(ids_of(ptr_x)).repeat_interleave(2).int()[::2]
    got = pca.nearest(x, y, strided, dev(ids_of(ptr_y)))
    assert (got == want).all()
    # one example
    want = torch.ops.torch_cluster.nearest(
        x, y, dev(np.array([0, len(x)])), dev(np.array([0, len(y)])))
    assert (pca.nearest(x, y) == want).all()


@pytest.mark.parametrize("rows", [2, 63, 64, 65, 5000])
def test_nearest_refuses(rows):
    x = torch.rand(rows, 3, device="cuda")
    y = torch.rand(6, 3, device="cuda")
    ids_x = torch.zeros(rows, dtype=torch.long, device="cuda")
    ids_x[-1] = 1
    ids_y = torch.tensor([0, 0, 0, 1, 1, 1], device="cuda")
    for at in {1, rows // 2, rows - 1}:
        bad = ids_x.clone()
        bad[at - 1] = 2
        with pytest.raises(ValueError, match="'batch_x' is not sorted"):
            pca.nearest(x, y, bad, ids_y)
    with pytest.raises(ValueError, match="'batch_y' is not sorted"):
        pca.nearest(x, y, ids_x, ids_y.flip(0))
    with pytest.raises(ValueError, match="do not occur"):
        pca.nearest(x, y, ids_x, torch.zeros_like(ids_y))
    with pytest.raises(ValueError, match="do not occur"):
        pca.nearest(x, y, ids_x * 3, ids_y)
    with pytest.raises(ValueError, match="do not occur"):
        pca.nearest(x, y, ids_x, ids_y + 4)
    with pytest.raises(ValueError, match="do not occur"):
        pca.nearest(x, y, ids_x - 7, ids_y - 7)
    assert pca.nearest(x, y, ids_x, ids_y).numel() == rows


@pytest.mark.parametrize("examples", [1, 2, 40, 1100, 3000])
@pytest.mark.parametrize("ratio", [None, 0.25, 0.3, 1.0 / 3.0, 1.0, 1e-6])
def test_fps_sizes(examples, ratio):
    rng = np.random.default_rng(examples)
    sizes = rng.integers(0, 40, examples)
    sizes[-1] = 17
    ptr = pointers(sizes)
    x = dev(rng.random((ptr[-1], 3)).astype(np.float32))
    share = torch.full((), 0.5 if ratio is None else ratio, device="cuda")
    for known in (None, examples, examples + 5):
        told = np.append(ptr, [ptr[-1]] * ((known or examples) - examples))
        for random_start in (False, True):
            torch.manual_seed(3)
            want = torch.ops.torch_cluster.fps(x, dev(told), share,
                                               random_start)
            torch.manual_seed(3)
            got = pca.fps(x, dev(ids_of(ptr)), ratio, random_start, known)
            assert got.shape == want.shape and (got == want).all()
    torch.manual_seed(4)
    want = torch.ops.torch_cluster.fps(x, dev(np.array([0, len(x)])), share,
                                       True)
    torch.manual_seed(4)
    assert (pca.fps(x, ratio=ratio) == want).all()


def test_fps_fewer_examples_than_ids():
    x = torch.rand(30, 3, device="cuda")
    ids = torch.arange(3, device="cuda").repeat_interleave(10)
    want = torch.ops.torch_cluster.fps(
        x, torch.tensor([0, 10, 20], device="cuda"),
        torch.full((), 0.5, device="cuda"), False)
    assert (pca.fps(x, ids, 0.5, False, 2) == want).all()
    with pytest.raises(RuntimeError):
        pca.fps(x, ids - 5, 0.5, False)


@pytest.mark.parametrize("call", ["nearest", "nearest_mismatch", "fps", "knn",
                                  "radius"])
def test_a_refused_call_leaves_no_number_of_examples_behind(call):
    """A call with one huge id fails; the next one, which starts with the
    number of examples of an earlier call, must not start with that id."""
    x = torch.rand(40, 3, device="cuda")
    ids = torch.arange(4, device="cuda").repeat_interleave(10)
    searches = [lambda: pca.nearest(x, x[::2], ids, ids[::2]),
                lambda: pca.fps(x, ids, 0.5, random_start=False),
                lambda: pca.knn_graph(x, 3, ids),
                lambda: pca.radius_graph(x, 0.4, ids)]
    want = [search() for search in searches]
    bad = ids.clone()
    bad[-1] = 10**12
    with pytest.raises((RuntimeError, ValueError)):
        if call == "nearest":
            falls = bad.clone()
            falls[3] = 2
            pca.nearest(x, x[::2], falls, ids[::2])
        elif call == "nearest_mismatch":
            pca.nearest(x, x[10:20], bad, ids[10:20])
        elif call == "fps":
            pca.fps(x, bad, 0.5, random_start=False)
        elif call == "knn":
            pca.knn_graph(x, 3, bad)
        else:
            pca.radius_graph(x, 0.4, bad)
    for search, rows in zip(searches, want):
        assert (search() == rows).all()


def test_examples_of_a_much_larger_batch_before():
    many = torch.arange(5000, device="cuda").repeat_interleave(3)
    x = torch.rand(15000, 3, device="cuda")
    ids = torch.tensor([0] * 30 + [2] * 10, device="cuda")
    y = torch.rand(40, 3, device="cuda")
    want = [pca.knn_graph(y, 3, ids, batch_size=3),
            pca.radius_graph(y, 0.4, ids, batch_size=3),
            pca.fps(y, ids, 0.5, random_start=False, batch_size=3)]
    waits = torch.ops.pytorch_cluster_amd.host_waits
    for i, search in enumerate((lambda: pca.knn_graph(y, 3, ids),
                                lambda: pca.radius_graph(y, 0.4, ids),
                                lambda: pca.fps(y, ids, 0.5,
                                                random_start=False))):
        pca.radius_graph(x, 0.1, many)
        pca.radius_graph(x, 0.1, many)
        before = waits()
        assert (search() == want[i]).all()
        assert waits() - before == 2  # (more examples than rows: looked up)
