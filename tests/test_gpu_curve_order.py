"""The sort of rows along the curve in front of the binned searches and of fps
over large examples: what it leaves, not only that a search over it is right (any
order of the rows gives the same neighbours).  Per segment the rows are a
permutation of the segment's, keys ascend and rows of equal keys ascend."""
import ctypes

import pytest
import torch

from pytorch_cluster_amd import _native, capi

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
LIB = ctypes.CDLL(_native.CAPI_PATH)


def align(size):
    return (size + 255) // 256 * 256


def words(scratch, offset, count):
    """`count` unsigned 32-bit words of the scratch as int64."""
    part = scratch[offset:offset + 4 * count].view(torch.int32).long()
    return torch.where(part < 0, part + (1 << 32), part)


def curve_order(x, ptr):
    """(keys, rows) of pca::launch_curve_order; its scratch starts with the
    segments' boxes (24 bytes each), the keys, the rows."""
    size = LIB._ZN3pca17curve_order_bytesEii
    size.restype = ctypes.c_size_t
    order = LIB._ZN3pca18launch_curve_orderEPKfPKliiiPvPPKjP12ihipStream_t
    n, segments = x.shape[0], ptr.numel() - 1
    scratch = torch.empty(size(ctypes.c_int(n), ctypes.c_int(segments)),
                          dtype=torch.uint8, device=DEV)
    perm = ctypes.c_void_p()
    stream = torch.cuda.current_stream().cuda_stream
    assert order(ctypes.c_void_p(x.data_ptr()),
                 ctypes.c_void_p(ptr.data_ptr()), ctypes.c_int(n),
                 ctypes.c_int(x.shape[1]), ctypes.c_int(segments),
                 ctypes.c_void_p(scratch.data_ptr()), ctypes.byref(perm),
                 ctypes.c_void_p(stream)) == 0
    at_keys = align(24 * segments)
    at_perm = at_keys + align(4 * n)
    assert perm.value == scratch.data_ptr() + at_perm
    return words(scratch, at_keys, n), words(scratch, at_perm, n)


def check(keys, rows, ptr):
    n, segments = rows.numel(), ptr.numel() - 1
    sizes = (ptr[1:] - ptr[:-1]).to(DEV)
    segment = torch.repeat_interleave(torch.arange(segments, device=DEV),
                                      sizes)
    everyone = torch.arange(n, device=DEV)
    assert torch.equal(rows.sort().values, everyone)
    assert torch.equal(segment[rows], segment)
    bits = max(segments - 1, 0).bit_length()
    axis = min(10, (32 - bits) // 3)
    assert torch.equal(keys >> (3 * axis), segment)
    equal = keys[1:] == keys[:-1]
    assert bool(((keys[1:] > keys[:-1])
                 | equal & (rows[1:] > rows[:-1])).all())


def points(kind, n, d, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.rand(n, d, generator=g, device=DEV)
    if kind == "equal":
        x[:] = 0.25
    elif kind == "two_places":
        x = (x[:, :1] < 0.5).float().expand(n, d).contiguous()
    elif kind == "clump":  # a third of the rows share few places
        x[::3] *= 1e-3
    elif kind == "in_order":
        x = x.sort(dim=0).values
    elif kind == "not_finite":
        x[::5, 0] = float("nan")
        x[1::7, d - 1] = float("inf")
    return x


KINDS = ["uniform", "equal", "two_places", "clump", "in_order", "not_finite"]
# one bucket of 768 rows and one row more or less, a workgroup's 512, 1,024, 2,048
# and 4,096 places, tiles of 2,048 rows, empty segments
SIZES = [1, 511, 512, 513, 767, 768, 769, 0, 1024, 1025, 1536, 1537, 2048,
         2049, 0, 4096, 4097, 5000, 3, 40000, 0]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("d", [1, 2, 3])
@pytest.mark.parametrize("sizes", [SIZES, [300000], [1], [0, 7, 0]])
def test_rows_in_the_order_of_their_keys(kind, d, sizes):
    ptr = torch.tensor([0] + sizes).cumsum(0)
    x = points(kind, int(ptr[-1]), d, 31 + d)
    check(*curve_order(x, ptr.to(DEV)), ptr)


# Sorted by samples: a segment of 750,000 rows, 4,000,000 rows, most of them in one
# segment (buckets of 2,000 rows, some of more than the 4,096 that fit on the chip).
# By digits: one row more than either; a tile of 4,096 rows more and less, segments
# that start and end within tiles; keys of 30, 31 and 32 bits.
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("sizes", [
    [750000], [750001], [4096 * 184 - 1], [4096 * 184], [4096 * 184 + 1],
    [0, 40, 0, 3999959, 1, 0], [0, 40, 0, 3999960, 1, 0],
    [1000000, 0, 5, 3500000], [750001, 750001], [30011] * 140, [9000000]])
def test_many_rows_in_the_order_of_their_keys(kind, sizes):
    ptr = torch.tensor([0] + sizes).cumsum(0)
    x = points(kind, int(ptr[-1]), 3, 7)
    check(*curve_order(x, ptr.to(DEV)), ptr)


@pytest.mark.parametrize("kind", ["uniform", "clump"])
@pytest.mark.parametrize("rows,queries", [
    ([5000, 0, 40000], [700, 3, 1]), ([800, 300000], [100000, 20000]),
    ([40, 1600000], [1, 3000]), ([3000, 10], [1600000, 50000])])
def test_two_sides_of_different_size(kind, rows, queries):
    """Both sides of a search, each in the box of the rows: in the workspace of
    the kNN search, which starts as the scratch above does."""
    ptr_x, ptr_y = (torch.tensor([0] + s).cumsum(0) for s in (rows, queries))
    x = points(kind, int(ptr_x[-1]), 3, 1)
    y = points(kind, int(ptr_y[-1]), 3, 2)
    n, m, segments = x.shape[0], y.shape[0], len(rows)
    ws = capi.knn_launch(x, y, ptr_x.to(DEV), ptr_y.to(DEV), 4,
                         binned=True)[3]
    at = align(24 * segments)
    found = []
    for count in (n, m, n, m):
        found.append(words(ws, at, count))
        at += align(4 * count)
    keys_x, keys_y, rows_x, rows_y = found
    check(keys_x, rows_x, ptr_x)
    check(keys_y, rows_y, ptr_y)
