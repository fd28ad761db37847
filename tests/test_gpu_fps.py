"""GPU parity of `fps` (pca_fps through the C ABI, the TorchScript operator
and the Python entry point) against the oracle's play-through of the reference
kernel (csrc/cuda/fps_cuda.cu:10-66).  The sampled rows and their order must
be identical, ties and the 5e4 clipping included."""
import numpy as np
import pytest
import torch
from torch import Tensor

pytestmark = pytest.mark.gpu

import pytorch_cluster_amd as pca  # noqa: E402
from pytorch_cluster_amd import capi  # noqa: E402
from gpu_common import DEV, dev  # noqa: E402

TORCH_DTYPE = {np.float32: torch.float32, np.float64: torch.float64,
               np.float16: torch.float16}


def gpu_fps(oracle, x, ptr, ratio, start=None, max_rows=None):
    """pca_fps through the C ABI with the oracle's output positions."""
    dt = x.dtype.type
    out_ptr = oracle.fps_out_ptr(ptr, ratio, dt)
    if max_rows is None:
        max_rows = int(np.diff(ptr).max())
    out, _ws = capi.fps_launch(dev(x), dev(ptr, torch.long),
                               dev(out_ptr, torch.long), int(out_ptr[-1]),
                               dev(start, torch.long), max_rows)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.float16])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 33])
def test_random_points(oracle, dtype, d):
    rng = np.random.default_rng(100 * d)
    ptr = np.array([0, 900, 900, 3000, 8000], dtype=np.int64)
    x = rng.standard_normal((8000, d)).astype(dtype)
    ratio = np.array([0.1, 0.5, 0.05, 0.02])
    got = gpu_fps(oracle, x, ptr, ratio)
    want = oracle.fps_op(x, ptr, ratio)
    assert (got == want).all()


@pytest.mark.parametrize("dtype,d", [(np.float32, 3), (np.float32, 2),
                                     (np.float32, 7), (np.float64, 3),
                                     (np.float16, 3)])
def test_ties_and_clipping_follow_the_reference_block(oracle, dtype, d):
    rng = np.random.default_rng(23 + d)
    ptr = np.array([0, 900, 1500, 6000], dtype=np.int64)
    x = rng.integers(0, 5, (6000, d)).astype(dtype)
    x[900:1500] *= 60  # most running minima stay at the 5e4 they start from
    ratio = np.array([0.05, 0.1, 0.01])
    got = gpu_fps(oracle, x, ptr, ratio)
    want = oracle.fps_op(x, ptr, ratio)
    assert (got == want).all()


@pytest.mark.parametrize("rows", [1, 200, 256, 257, 512, 1000, 1024, 2047,
                                  2048, 3000, 4096, 4097, 8192, 8193, 12000,
                                  16384])
@pytest.mark.parametrize("d", [2, 3, 4])
def test_every_register_shape_resolves_ties_like_the_reference(oracle, rows, d):
    """The register kernel's launch shape follows the largest example; points
    on a coarse integer grid make most maxima ties, which go by
    (row - start) % 256 first and the row second."""
    rng = np.random.default_rng(rows + d)
    small = max(1, rows // 3)
    ptr = np.array([0, small, small + rows], dtype=np.int64)
    x = rng.integers(0, 4, (ptr[-1], d)).astype(np.float32)
    ratio = np.array([0.5, min(1.0, 150.0 / rows)])
    start = np.array([small - 1, rows // 2], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, ratio, start)
    want = oracle.fps_op(x, ptr, ratio, start)
    assert (got == want).all()


def test_register_and_streaming_kernels_agree(oracle):
    """Examples of up to 4,096 / 16,384 rows are sampled from registers,
    larger ones (or an unknown bound) from memory: same samples."""
    rng = np.random.default_rng(5)
    for n_big in (4096, 16384, 16385, 30000):
        ptr = np.array([0, 1000, 1000 + n_big], dtype=np.int64)
        x = rng.standard_normal((ptr[-1], 3)).astype(np.float32)
        ratio = np.array([0.2, 300.0 / n_big])
        want = oracle.fps_op(x, ptr, ratio)
        assert (gpu_fps(oracle, x, ptr, ratio) == want).all()
        assert (gpu_fps(oracle, x, ptr, ratio, max_rows=0) == want).all()


# 1,025 / 4,097 / 8,193: where the kernels that skip rows change; 16,385: from
# memory on; 65,537 and 131,073: two and four slots per lane; 262,145: several
# pieces of 64 rows to a bucket
@pytest.mark.parametrize("kind", ["grid", "far", "odd"])
@pytest.mark.parametrize("rows,d", [(1025, 3), (4097, 3), (4097, 4), (8193, 2),
                                    (16385, 3), (65537, 1), (131073, 2),
                                    (262145, 3)])
def test_skipped_rows_change_nothing(oracle, rows, d, kind):
    """Rows in buckets, whole buckets left alone: ties (a coarse grid, and
    distances beyond the 5e4 cap), rows with NaN and infinite coordinates,
    examples of very different sizes, rows in front of the first example."""
    rng = np.random.default_rng(rows + d)
    ptr = np.cumsum([5, 70, rows, 1, 300]).astype(np.int64)
    n = ptr[-1] + 3
    x = (rng.integers(0, 9, (n, d)) if kind == "grid" else
         rng.standard_normal((n, d)) * (300 if kind == "far" else 1))
    x = x.astype(np.float32)
    if kind == "odd":
        x[100] = np.nan
        x[rows // 2, 0] = np.inf
    share = np.array([0.5, 60.0 / rows, 1.0, 0.1])
    start = np.array([3, rows - 1, 0, 12], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, share, start)
    want = oracle.fps_op(x, ptr, share, start)
    assert (got == want).all()


# 1,025 / 2,048 / 4,097: rows per lane of a wave's stretch; 32,768 / 65,536 / 262,144:
# of one, two, four pieces of 64 rows in memory and of several times four; hundreds
# of samples, most of them several to a step
@pytest.mark.parametrize("kind", ["uniform", "grid", "copies", "clusters"])
@pytest.mark.parametrize("rows,d", [(1025, 3), (2048, 2), (4096, 4), (4097, 1),
                                    (8192, 3), (16385, 3), (32769, 3),
                                    (65537, 2), (262145, 3)])
def test_several_samples_per_step_are_those_one_by_one(oracle, rows, d, kind):
    rng = np.random.default_rng(rows)
    second = max(1000, rows // 16)
    ptr = np.cumsum([0, 40, rows, second]).astype(np.int64)
    n = ptr[-1]
    if kind == "uniform":
        x = rng.random((n, d))
    elif kind == "grid":  # most largest minima are ties
        x = rng.integers(0, 24, (n, d))
    elif kind == "copies":  # samples whose neighbours come to a minimum of 0
        x = rng.random((700, d))[rng.integers(0, 700, n)]
    else:
        x = rng.random((12, d))[rng.integers(0, 12, n)]
        x = x + 0.003 * rng.standard_normal((n, d))
    x = x.astype(np.float32)
    share = np.array([1.0, 750.0 / rows, 800.0 / second])
    start = np.array([7, rows - 1, 0], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, share, start)
    want = oracle.fps_op(x, ptr, share, start)
    assert (got == want).all()


# 255 / 256 rows: fewest of which the waves have stretches; 1,024 to 8,192: rows per
# lane; stretches of equal and of unequal length, all examples in one call
@pytest.mark.parametrize("kind", ["uniform", "grid"])
@pytest.mark.parametrize("sizes,d", [
    ([255, 256, 271, 1024, 1025, 2048, 4096], 3), ([2049, 300, 3000], 2),
    ([4096, 1023, 2047], 4), ([8192, 4097, 4096, 1024, 260], 3),
    ([8191, 5000], 1)])
def test_stretches_of_every_length(oracle, sizes, d, kind):
    rng = np.random.default_rng(sum(sizes) + d)
    ptr = np.cumsum([0] + sizes).astype(np.int64)
    x = rng.random((ptr[-1], d)) if kind == "uniform" else \
        rng.integers(0, 13, (ptr[-1], d))
    x = x.astype(np.float32)
    # (more samples than rows: the smallest tie among minima of 0, again and again)
    share = np.array([520.0 / n for n in sizes])
    start = np.array([n // 2 for n in sizes], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, share, start)
    assert (got == oracle.fps_op(x, ptr, share, start)).all()


# An example by several workgroups, one for 1,024 rows up to 32 of them, up to 256 of
# all examples; 2, 4, 8, 16 rows of a lane; 4, 8, 16 entries told (17, 9, fewer
# workgroups).  Examples of fewer than 1,024 rows, and those beyond 16,384 rows of a
# workgroup, are one workgroup's.
SHARED = [([16384, 1023, 1024, 2047, 2048, 40], 3),
          ([9215, 9216, 16385, 17407, 17408], 2), ([65536, 65537, 33000], 3),
          ([131073, 1100], 1), ([262144, 262145], 3), ([524288], 3),
          ([524289], 3), ([40] * 63 + [32769], 3), ([1500] * 63 + [65537], 3),
          ([1025] * 24 + [16500], 2)]


@pytest.mark.parametrize("kind", ["uniform", "grid", "odd"])
@pytest.mark.parametrize("sizes,d", SHARED)
def test_examples_of_several_workgroups(oracle, sizes, d, kind):
    rng = np.random.default_rng(sum(sizes) + d)
    ptr = np.cumsum([0] + sizes).astype(np.int64)
    n = ptr[-1]
    x = rng.integers(0, 17, (n, d)) if kind == "grid" else rng.random((n, d))
    x = x.astype(np.float32)
    if kind == "odd":
        x[rng.random(n) < 0.1] *= 400.0  # minima clipped at first
        x[rng.random(n) < 0.01, 0] = np.nan
        x[rng.random(n) < 0.001] = np.inf
    samples = 120 if n > 300000 else 500
    share = np.array([min(samples, 2 * s) / s for s in sizes])
    start = np.array([s // 2 for s in sizes], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, share, start, max(max(sizes), 16385))
    assert (got == oracle.fps_op(x, ptr, share, start)).all()


# More than 64 examples in curve order, not shared: stretches of 8, 12 and 16 rows of
# a lane (8,192 and 12,288 rows), other examples beside them.
@pytest.mark.parametrize("kind", ["uniform", "grid", "odd"])
@pytest.mark.parametrize("d", [2, 3])
def test_stretches_of_rows_in_memory(oracle, d, kind):
    rng = np.random.default_rng(70 + d)
    sizes = [16384, 12289, 16383, 12288, 8193, 8192, 256, 255] + [300] * 57
    ptr = np.cumsum([0] + sizes).astype(np.int64)
    n = ptr[-1]
    x = rng.integers(0, 17, (n, d)) if kind == "grid" else rng.random((n, d))
    x = x.astype(np.float32)
    if kind == "odd":
        x[rng.random(n) < 0.1] *= 400.0
        x[rng.random(n) < 0.01, 0] = np.nan
        x[rng.random(n) < 0.001] = np.inf
    share = np.array([min(400, 2 * s) / s for s in sizes])
    start = np.array([s // 2 for s in sizes], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, share, start, 16385)
    assert (got == oracle.fps_op(x, ptr, share, start)).all()


# 4,096 rows, 1,100 and 1,600 samples, 16 and 64 examples: where rows that fit one
# workgroup are shared all the same; 8,192 rows, 170 and 220 samples: where larger
# ones go through memory; 16,384 / 16,385: rows that are ordered in LDS
@pytest.mark.parametrize("rows,examples,samples", [
    (4096, 2, 1100), (4097, 2, 1099), (4097, 2, 1100), (8192, 16, 1100),
    (8192, 17, 1100), (5000, 17, 1599), (5000, 64, 1600), (5000, 65, 1600),
    (9000, 16, 169), (9000, 16, 170), (9000, 17, 219), (8193, 65, 220),
    (12288, 3, 250), (12289, 3, 250), (16384, 3, 250), (16385, 3, 250)])
def test_entry_points_where_examples_are_shared(oracle, rows, examples, samples):
    rng = np.random.default_rng(rows + samples)
    sizes = [rows] + [300] * (examples - 2) + [rows // 3]
    ptr = np.cumsum([0] + sizes).astype(np.int64)
    x = rng.random((ptr[-1], 3)).astype(np.float32)
    batch = np.repeat(np.arange(examples), sizes)
    ratio = (samples - 0.5) / rows
    want = oracle.fps_op(x, ptr, np.float32(ratio))
    got = pca.fps(dev(x), dev(batch, torch.long), ratio, random_start=False)
    assert (got.cpu().numpy() == want).all()
    got = torch.ops.torch_cluster.fps(
        dev(x), dev(ptr, torch.long),
        torch.tensor(ratio, dtype=torch.float32, device=DEV), False)
    assert (got.cpu().numpy() == want).all()


def probe_library():
    import ctypes
    import os
    return ctypes.CDLL(os.path.join(os.path.dirname(pca.__file__),
                                    "libpca_probe.so"))


def probe_fps(oracle, x, ptr, ratio, max_rows, told=-1, came=-1,
              before=lambda: None):
    """launch_fps with a patience (-1: its own); samples, and which examples
    one workgroup sampled after all.  `before` is called right before it."""
    import ctypes
    lib = probe_library()
    count = len(ptr) - 1
    out_ptr = oracle.fps_out_ptr(ptr, ratio, np.float32)
    bytes_ = capi.capi.pca_fps_workspace_bytes(len(x), x.shape[1], count,
                                               max_rows, 0)
    held = [dev(x), dev(ptr, torch.long), dev(out_ptr, torch.long),
            torch.full((int(out_ptr[-1]),), -1, dtype=torch.long, device=DEV),
            torch.empty(bytes_, dtype=torch.uint8, device=DEV),
            torch.zeros(count, dtype=torch.int32, device=DEV)]
    src, ptr_, out_ptr_, out, work, states = [ctypes.c_void_p(t.data_ptr())
                                              for t in held]
    torch.cuda.current_stream().synchronize()
    before()
    assert lib.pca_probe_fps(src, ptr_, out_ptr_, ctypes.c_int64(len(x)),
                             ctypes.c_int64(x.shape[1]), ctypes.c_int64(count),
                             ctypes.c_int64(max_rows), ctypes.c_int(told),
                             ctypes.c_int(came), out, work,
                             ctypes.c_size_t(bytes_), states) == 0
    return held[3].cpu().numpy(), (held[5].cpu().numpy() >> 30 & 1).tolist()


@pytest.mark.parametrize("told,came", [(0, -1), (1, -1), (3, -1), (-1, 0),
                                       (-1, 1), (-1, -1)])
def test_workgroups_that_do_not_wait(oracle, told, came):
    """A workgroup that does not hear from the others in time marks its example
    and ends; another kernel samples that one from the start.  One that does not
    see the others come goes to work with those that did, if they are enough."""
    rng = np.random.default_rng(5)
    ptr = np.array([0, 20000, 21500, 61500], dtype=np.int64)
    x = rng.random((ptr[-1], 3)).astype(np.float32)
    ratio = 0.02
    got, marked = probe_fps(oracle, x, ptr, ratio, 40000, told, came)
    assert (got == oracle.fps_op(x, ptr, np.float32(ratio))).all()
    if told == 0:  # (nobody hears 31 others at the first look, 50 times over)
        assert marked[2] == 1
    if told == came == -1:
        assert marked == [0, 0, 0]


@pytest.mark.parametrize("kind", ["uniform", "grid"])
@pytest.mark.parametrize("told,came", [(0, -1), (-1, -1)])
def test_examples_given_up_are_sampled_in_stretches(oracle, told, came, kind):
    """The same where the other kernel holds the rows in registers (a bound of
    16,385): 16, 12 and 8 rows of a lane."""
    rng = np.random.default_rng(8)
    ptr = np.cumsum([0, 16384, 12289, 12288, 8192, 700]).astype(np.int64)
    x = rng.random((ptr[-1], 3)) if kind == "uniform" else \
        rng.integers(0, 17, (ptr[-1], 3))
    x = x.astype(np.float32)
    got, marked = probe_fps(oracle, x, ptr, 0.03, 16385, told, came)
    assert (got == oracle.fps_op(x, ptr, np.float32(0.03))).all()
    assert marked[:4] == [int(told == 0)] * 4
    assert told == 0 or marked[4] == 0


def streams_beside(count):
    """Streams whose work does not hold up the current one (streams share a few
    queues of the hardware)."""
    found = []
    for _ in range(32):
        stream = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            torch.cuda._sleep(2400000)  # (1 ms)
        torch.zeros(1, device=DEV)
        torch.cuda.current_stream().synchronize()
        if not stream.query():
            found.append(stream)
        if len(found) == count:
            torch.cuda.synchronize()
            return found
    pytest.skip("no %d streams beside the current one" % count)


def test_units_that_are_held_cost_workgroups_not_the_sharing(oracle):
    """A wave of another stream's kernel leaves no room on its compute unit: the
    example goes to the workgroups that came."""
    rng = np.random.default_rng(6)
    ptr = np.arange(9, dtype=np.int64) * 33000
    x = rng.random((ptr[-1], 3)).astype(np.float32)
    want = oracle.fps_op(x, ptr, np.float32(0.01))
    probe_fps(oracle, x, ptr, 0.01, 33000)
    side = streams_beside(3)
    for streams in (1, 3):
        for stream in side[:streams]:
            with torch.cuda.stream(stream):
                torch.cuda._sleep(24000000)  # (10 ms)
        got, marked = probe_fps(oracle, x, ptr, 0.01, 33000)
        asleep = not side[0].query()
        torch.cuda.synchronize()
        assert (got == want).all()
        assert asleep and marked == [0] * 8


@pytest.mark.parametrize("came", [0, -1])
def test_workgroups_wait_for_as_many_as_hold_the_rows(oracle, came):
    """32 units are free, a workgroup's each: 28 take the first example, the four
    that begin the second wait for a fifth until the first one is done."""
    import ctypes
    rng = np.random.default_rng(9)
    ptr = np.cumsum([0, 70000, 70000] + [40] * 7).astype(np.int64)
    x = rng.random((ptr[-1], 3)).astype(np.float32)
    ratio = np.float32(1999.5 / 70000)
    want = oracle.fps_op(x, ptr, ratio)
    side, = streams_beside(1)

    def hold(us):
        assert probe_library().pca_probe_hold(
            224, us, ctypes.c_void_p(side.cuda_stream)) == 0

    hold(1)
    assert probe_fps(oracle, x, ptr, ratio, 70000)[1] == [0] * 9
    got, marked = probe_fps(oracle, x, ptr, ratio, 70000, -1, came,
                            lambda: hold(4000))
    held = not side.query()
    torch.cuda.synchronize()
    assert held and (got == want).all()
    assert marked == [0, int(came == 0)] + [0] * 7


@pytest.mark.parametrize("kind", ["uniform", "grid"])
def test_short_examples_among_shared_ones_do_not_wait_for_them(oracle, kind):
    """Examples of fewer rows than two workgroups share are sampled beside the
    others, by the same kernel."""
    rng = np.random.default_rng(7)
    sizes = [20000, 1, 255, 256, 257, 0, 1023, 1024, 2047, 2048]
    ptr = np.cumsum([0] + sizes).astype(np.int64)
    x = rng.random((ptr[-1], 3)) if kind == "uniform" else \
        rng.integers(0, 9, (ptr[-1], 3))
    x = x.astype(np.float32)
    share = np.array([0.02] + [0.7] * 9).astype(np.float32)
    got, marked = probe_fps(oracle, x, ptr, share, 20000)
    assert (got == oracle.fps_op(x, ptr, share)).all()
    assert marked == [0] * 10


def test_shared_examples_on_several_streams():
    """Calls that each ask for every compute unit, side by side: the workgroups
    of one wait for units that the other holds."""
    g = torch.Generator(device=DEV).manual_seed(3)
    ids = torch.arange(8, device=DEV).repeat_interleave(40000)
    xs = [torch.rand(320000, 3, generator=g, device=DEV) for _ in range(3)]
    want = [pca.fps(x, ids, 0.01, random_start=False) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    got = []
    for _ in range(3):
        for x, stream in zip(xs, streams):
            with torch.cuda.stream(stream):
                got.append(pca.fps(x, ids, 0.01, random_start=False))
    torch.cuda.synchronize()
    for i, rows in enumerate(got):
        assert torch.equal(rows, want[i % 3])


# 8,192 rows, 170 samples: where the entry points change, for few examples of up to
# 3 dimensions, between the kernels on the chip and rows in curve order
@pytest.mark.parametrize("rows,samples", [(8192, 400), (8193, 169), (8193, 170),
                                          (16384, 169), (16384, 170),
                                          (16384, 485)])
@pytest.mark.parametrize("d", [3, 4])
def test_entry_points_where_the_kernels_change(oracle, rows, samples, d):
    rng = np.random.default_rng(rows + samples)
    ptr = np.array([0, rows, rows + 500, 2 * rows + 400], dtype=np.int64)
    x = rng.random((ptr[-1], d)).astype(np.float32)
    batch = np.repeat(np.arange(3), np.diff(ptr))
    ratio = (samples - 0.5) / rows
    want = oracle.fps_op(x, ptr, np.float32(ratio))
    got = pca.fps(dev(x), dev(batch, torch.long), ratio, random_start=False)
    assert (got.cpu().numpy() == want).all()
    got = torch.ops.torch_cluster.fps(
        dev(x), dev(ptr, torch.long),
        torch.tensor(ratio, dtype=torch.float32, device=DEV), False)
    assert (got.cpu().numpy() == want).all()


# whole buckets (64 or 128 consecutive rows along the curve) at an infinite
# distance: rows without a finite coordinate on an axis, rows and first samples
# at infinity, squared gaps beyond the fp32 range
@pytest.mark.parametrize("kind", ["nan", "nan_axis", "all_nan", "all_nan_axis",
                                  "inf", "inf_start", "far", "mixed"])
@pytest.mark.parametrize("rows,d", [(1025, 3), (4096, 4), (4097, 3), (4097, 4),
                                    (8193, 2), (16385, 3), (20000, 1),
                                    (262145, 3)])
def test_rows_out_of_reach_keep_their_place(oracle, rows, d, kind):
    rng = np.random.default_rng(rows + d)
    begin, first = 70, 5
    ptr = np.array([0, begin, begin + rows], dtype=np.int64)
    x = rng.standard_normal((ptr[-1], d)).astype(np.float32)
    some = begin + rng.permutation(rows)[:rows // 3]
    if kind == "nan":
        x[some] = np.nan
    elif kind == "nan_axis":
        x[some, d - 1] = np.nan
    elif kind == "all_nan":
        x[begin:] = np.nan
    elif kind == "all_nan_axis":
        x[begin:, 0] = np.nan
    elif kind == "inf":
        x[some, 0] = np.inf
        x[some[:200], 0] = -np.inf
        x[begin + first] = 0
    elif kind == "inf_start":
        x[begin + first, d - 1] = np.inf
    elif kind == "far":
        x[some] += np.float32(3e19)
        x[begin + first] = 0
    else:
        x[some] = np.nan
        x[some[:300]] = np.inf
        x[some[300:]] *= np.float32(1e25)
    share = np.array([0.1, 130.0 / rows])
    start = np.array([0, first], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, share, start)
    assert got.min() >= 0 and (got[7:] >= begin).all()
    assert got.max() < ptr[-1]
    assert (got == oracle.fps_op(x, ptr, share, start)).all()


# one sample more or fewer decides whether every row is looked at (up to `few`
# samples, by rows and dimensions) or the rows are put in order; examples on both
# sides in one call
@pytest.mark.parametrize("rows,d,few", [
    (257, 3, 119), (512, 2, 119), (513, 3, 89), (1024, 1, 89), (1025, 3, 129),
    (2048, 2, 129), (4096, 1, 129), (4097, 3, 169), (8192, 3, 169),
    (257, 4, 139), (2048, 4, 139), (2049, 4, 169), (8192, 4, 169),
    (8193, 3, 339), (16384, 2, 339), (8193, 4, 479), (16384, 4, 479)])
def test_few_samples_and_many(oracle, rows, d, few):
    rng = np.random.default_rng(rows + d)
    ptr = np.cumsum([0, rows, 7, rows, rows // 2, rows]).astype(np.int64)
    samples = np.array([few, 7, few + 1, rows // 200 + 1, 1])
    for grid in (False, True):
        x = rng.standard_normal((ptr[-1], d)).astype(np.float32)
        if grid:
            x = rng.integers(0, 6, x.shape).astype(np.float32)
        share = ((samples - 0.5) / np.diff(ptr)).astype(np.float32)
        assert (np.diff(oracle.fps_out_ptr(ptr, share, np.float32)) ==
                samples).all()
        start = np.array([rows - 1, 6, 0, 1, 5], dtype=np.int64)
        got = gpu_fps(oracle, x, ptr, share, start)
        assert (got == oracle.fps_op(x, ptr, share, start)).all()


@pytest.mark.parametrize("rows,samples", [(16385, 8), (16385, 9), (16384, 8),
                                          (60000, 3), (60000, 4), (140000, 1)])
def test_a_handful_of_samples_from_large_examples(oracle, rows, samples):
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((2 * rows, 3)).astype(np.float32)
    ptr = np.array([0, rows, 2 * rows], dtype=np.int64)
    ratio = (samples - 0.5) / rows
    want = oracle.fps_op(x, ptr, ratio)
    ids = torch.arange(2, device=DEV).repeat_interleave(rows)
    got = pca.fps(dev(x), ids, ratio, random_start=False)
    assert (got.cpu().numpy() == want).all()
    got = pca.fps(dev(x), ptr=dev(ptr), ratio=ratio, random_start=False)
    assert (got.cpu().numpy() == want).all()
    one = pca.fps(dev(x[:rows]), None, ratio, random_start=False)
    assert (one.cpu().numpy() == want[:samples]).all()


# (bytes of a row: 0 on the chip, 8 with every row looked at, 24 in curve order)
@pytest.mark.parametrize("sizes,samples,least", [
    ([17000] * 64, 4, 8), ([16384, 17000, 40], 8, 8), ([16384, 17000, 40], 9, 24),
    ([16000] + [500] * 15, 169, 0), ([16000] + [500] * 15, 170, 24),
    ([16000] + [500] * 16, 219, 0), ([16000] + [500] * 16, 220, 24),
    ([8193] * 65, 219, 0), ([8193] * 65, 220, 24), ([9000] * 8, 450, 24),
    ([8192] * 16, 1099, 0), ([8192] * 16, 1100, 24), ([4097] * 2, 1100, 24),
    ([4096] * 16, 1700, 0), ([8192] * 17, 1599, 0), ([8192] * 17, 1600, 24),
    ([5000] * 64, 1600, 24), ([5000] * 65, 1600, 0)])
def test_both_entry_points_take_the_same_kernel(sizes, samples, least):
    """The kernel follows the largest example, the most samples of one and the
    number of examples, whoever asks: seen by the workspace it takes."""
    n, longest = sum(sizes), max(sizes)
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.rand(n, 3, generator=g, device=DEV)
    batch = torch.arange(len(sizes)).repeat_interleave(torch.tensor(sizes))
    batch = batch.to(DEV)
    ptr = torch.tensor(np.cumsum([0] + sizes), device=DEV)
    ratio = (samples - 0.5) / longest
    ratios = torch.full((len(sizes),), ratio, device=DEV)
    taken, rows = [], []
    for call in (lambda: pca.fps(x, batch, ratio, random_start=False),
                 lambda: torch.ops.torch_cluster.fps(x, ptr, ratios, False)):
        call()
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        rows.append(call())
        taken.append((torch.cuda.max_memory_allocated() - before) / n)
    assert torch.equal(rows[0], rows[1])
    for bytes_per_row in taken:  # (4: the result, most of what else is taken)
        assert least < bytes_per_row if least == 24 else \
            least <= bytes_per_row < least + 4


def test_captured_into_a_graph(oracle):
    """While its stream is being captured the search does without the sort of
    the large examples; every replay samples the same rows."""
    rng = np.random.default_rng(8)
    x = rng.standard_normal((18000, 3)).astype(np.float32)
    ptr = np.array([0, 18000], dtype=np.int64)
    want = oracle.fps_op(x, ptr, 40.0 / 18000)
    out_ptr = oracle.fps_out_ptr(ptr, 40.0 / 18000, np.float32)
    args = (dev(x), dev(ptr, torch.long), dev(out_ptr, torch.long),
            int(out_ptr[-1]), None, 18000)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, _ws = capi.fps_launch(*args)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert (out.cpu().numpy() == want).all()
        eager, _ws2 = capi.fps_launch(*args)
        torch.cuda.synchronize()
        assert (eager.cpu().numpy() == want).all()


def test_start_offsets_nan_rows_and_oversampling(oracle):
    rng = np.random.default_rng(6)
    x = rng.standard_normal((700, 3)).astype(np.float32)
    ptr = np.array([0, 300, 700], dtype=np.int64)
    got = gpu_fps(oracle, x, ptr, 0.1, start=np.array([17, 250]))
    assert (got == oracle.fps_op(x, ptr, 0.1, start=[17, 250])).all()
    # rows with NaN coordinates keep the value they start from
    x[5] = np.nan
    x[400, 1] = np.nan
    for max_rows in (None, 0):
        got = gpu_fps(oracle, x, ptr, 0.2, max_rows=max_rows)
        assert (got == oracle.fps_op(x, ptr, 0.2)).all()
    # more samples than rows: the arg-max over zeros follows the tie rule
    y = rng.standard_normal((40, 2)).astype(np.float32)
    p = np.array([0, 40], dtype=np.int64)
    for max_rows in (None, 0):
        got = gpu_fps(oracle, y, p, 1.5, max_rows=max_rows)
        assert (got == oracle.fps_op(y, p, 1.5)).all()
    # every value NaN: the reference's index 0
    z = np.full((10, 3), np.nan, dtype=np.float32)
    p = np.array([0, 4, 10], dtype=np.int64)
    for max_rows in (None, 0):
        got = gpu_fps(oracle, z, p, 0.5, max_rows=max_rows)
        assert (got == oracle.fps_op(z, p, 0.5)).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16])
def test_entry_point_fixture(dtype):
    # test/test_fps.py:16-63 of the reference
    x = torch.tensor([[-1, -1], [-1, +1], [+1, +1], [+1, -1],
                      [-2, -2], [-2, +2], [+2, +2], [+2, -2]],
                     dtype=dtype, device=DEV)
    batch = torch.tensor([0, 0, 0, 0, 1, 1, 1, 1], device=DEV)
    ptr_list = [0, 4, 8]
    ptr = torch.tensor(ptr_list, device=DEV)
    out = pca.fps(x, batch, random_start=False)
    assert out.dtype == torch.long and out.device == x.device
    assert out.tolist() == [0, 2, 4, 6]
    assert pca.fps(x, batch, ratio=0.5,
                   random_start=False).tolist() == [0, 2, 4, 6]
    ratio = torch.tensor(0.5, device=DEV)
    assert pca.fps(x, batch, ratio=ratio,
                   random_start=False).tolist() == [0, 2, 4, 6]
    assert pca.fps(x, ptr=ptr_list, ratio=0.5,
                   random_start=False).tolist() == [0, 2, 4, 6]
    assert pca.fps(x, ptr=ptr, ratio=0.5,
                   random_start=False).tolist() == [0, 2, 4, 6]
    ratio = torch.tensor([0.5, 0.5], device=DEV)
    assert pca.fps(x, batch, ratio=ratio,
                   random_start=False).tolist() == [0, 2, 4, 6]
    assert sorted(pca.fps(x, random_start=False).tolist()) == [0, 5, 6, 7]
    assert sorted(pca.fps(x, ratio=0.5,
                          random_start=False).tolist()) == [0, 5, 6, 7]
    assert sorted(pca.fps(x, ratio=torch.tensor([0.5], device=DEV),
                          random_start=False).tolist()) == [0, 5, 6, 7]

    @torch.jit.script
    def fps2(x: Tensor, ratio: Tensor) -> Tensor:
        return pca.fps(x, None, ratio, False)

    out = fps2(x, torch.tensor([0.5], device=DEV))
    assert sorted(out.tolist()) == [0, 5, 6, 7]


def test_random_start():
    # test/test_fps.py:66-75 of the reference
    N = 1024
    for _ in range(5):
        pos = torch.randn((2 * N, 3), device=DEV)
        batch = torch.cat([torch.zeros(N, dtype=torch.long, device=DEV),
                           torch.ones(N, dtype=torch.long, device=DEV)])
        idx = pca.fps(pos, batch, ratio=0.5)
        assert idx.numel() == N
        assert idx.min() >= 0 and idx.max() < 2 * N
        assert (idx[:N // 2] < N).all() and (idx[N // 2:] >= N).all()
        assert idx.unique().numel() == N


def test_operator_against_oracle_with_ratio_types(oracle):
    """The sample counts come from ceil(deg * ratio) in the ratio's type."""
    rng = np.random.default_rng(9)
    x = rng.standard_normal((3013, 3)).astype(np.float32)
    ptr = np.array([0, 10, 13, 3013], dtype=np.int64)
    for ratio in (0.3, 0.001):
        got = torch.ops.torch_cluster.fps(
            dev(x), dev(ptr, torch.long),
            torch.tensor(ratio, dtype=torch.float32, device=DEV), False)
        want = oracle.fps_op(x, ptr, ratio)
        assert got.cpu().numpy().tolist() == want.tolist()
    with pytest.raises(RuntimeError, match="BFloat16"):
        pca.fps(dev(x).to(torch.bfloat16), random_start=False)


def test_set_abstraction_sizes(oracle):
    """16 clouds of 4,096 points, a quarter sampled (the step that precedes
    radius / knn in a PointNet++ layer): every cloud against the oracle."""
    g = torch.Generator().manual_seed(0)
    x = torch.rand(16 * 4096, 3, generator=g)
    ptr = torch.arange(17) * 4096
    out = torch.ops.torch_cluster.fps(
        x.to(DEV), ptr.to(DEV), torch.tensor(0.25, device=DEV), False)
    want = oracle.fps_op(x.numpy(), ptr.numpy(), 0.25)
    assert out.cpu().numpy().tolist() == want.tolist()
