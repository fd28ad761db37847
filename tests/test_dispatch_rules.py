"""Which kernel a call takes, as the libraries decide it on the host (no GPU)."""
import ctypes

import pytest

from pytorch_cluster_amd import _native


def rule(mangled, *args):
    function = getattr(ctypes.CDLL(_native.CAPI_PATH), mangled)
    function.restype = ctypes.c_bool
    function.argtypes = [ctypes.c_int] * len(args)
    return function(*args)


def knn_wave(n, m, k, examples=1, d=3):
    # bool pca::knn_wave_supported(n, m, d, num_segments, k, cosine)
    return rule("_ZN3pca18knn_wave_supportedEiiiiib", n, m, d, examples, k, 0)


@pytest.mark.parametrize("n,m,k", [
    (50000, 4000, 4), (50000, 8000, 16), (100000, 64, 4), (100000, 2000, 16),
    (100000, 4000, 32), (200000, 64, 16), (200000, 1000, 4),
    (200000, 4000, 16), (524288, 4096, 1), (20000, 8000, 16),
    (1000000, 1, 8)])
def test_few_queries_among_many_rows_take_the_sliced_scan(monkeypatch, n, m,
                                                          k):
    # (1.1 to 4.6 times slower with a wave per query)
    monkeypatch.delenv("PCA_KNN_WAVE", raising=False)
    assert not knn_wave(n, m, k)
    assert not knn_wave(n, m, k, d=4)


@pytest.mark.parametrize("n,m,k,examples", [
    (1024, 1024, 16, 1), (4096, 4096, 16, 1), (8192, 8192, 16, 1),
    (8192, 8192, 16, 8), (16384, 64, 16, 1), (16384, 2048, 32, 1),
    (4096, 1, 1, 1), (1024, 1024, 33, 1), (65536, 65536, 33, 16)])
def test_small_calls_take_a_wave_per_query(monkeypatch, n, m, k, examples):
    monkeypatch.delenv("PCA_KNN_WAVE", raising=False)
    assert knn_wave(n, m, k, examples)


# Uniform clouds: calls of both searches on an MI355X, us.
GRAPHS = [
    # clouds, rows each, k, scan, binned
    (1, 23000, 4, 109, 123), (1, 23000, 17, 209, 167), (1, 23000, 25, 257, 195),
    (1, 25000, 17, 236, 168), (1, 25000, 25, 289, 192), (1, 27000, 17, 252, 171),
    (1, 27000, 25, 319, 200), (1, 32768, 4, 155, 125), (1, 32768, 17, 297, 178),
    (1, 16000, 4, 94, 113), (1, 16000, 8, 107, 124), (1, 19000, 9, 132, 142),
    (1, 22000, 32, 282, 199), (1, 22000, 33, 633, 221), (2, 17500, 4, 124, 134),
    (2, 17500, 16, 205, 160), (2, 17500, 24, 268, 183), (2, 23000, 4, 158, 135),
    (8, 12000, 24, 334, 214), (8, 12000, 8, 190, 158), (8, 12000, 16, 246, 188),
    (8, 4096, 16, 90, 157), (64, 4096, 16, 232, 272), (64, 6500, 4, 341, 251),
    (8, 9000, 33, 645, 322), (32, 4096, 33, 532, 350)]
FEW_QUERIES = [
    # rows, queries, clouds, k, scan, binned
    (1000000, 1954, 1, 4, 384, 1122), (1000000, 1954, 1, 32, 670, 2210),
    (1000000, 3907, 1, 4, 448, 814), (300000, 4688, 1, 16, 318, 512),
    (1000000, 15625, 8, 16, 348, 605), (3000000, 5860, 8, 32, 549, 2176),
    (3000000, 11719, 8, 16, 545, 1246), (3000000, 2930, 1, 16, 1269, 2466)]


@pytest.mark.parametrize("queries,rows,clouds,scan,binned", [
    (3000, 1000000, 1, 358, 683),
    (1000, 100000, 1, 61, 352), (300000, 30000, 1, 580, 135),
    (100000, 300000, 1, 1711, 137), (1000000, 100000, 8, 871, 239)])
def test_auto_of_nearest_scans_for_few_queries(queries, rows, clouds, scan,
                                               binned):
    import torch
    import pytorch_cluster_amd as pca
    before = pca.get_search_strategy()
    pca.set_search_strategy("auto")
    try:
        assert torch.ops.pytorch_cluster_amd.strategy_for(
            "nearest", rows, queries, clouds) == \
            ("binned" if binned < scan else "scan")
    finally:
        pca.set_search_strategy(before)


@pytest.mark.parametrize("rows,queries,clouds,k,scan,binned", FEW_QUERIES)
def test_auto_scans_for_few_queries_among_many_rows(rows, queries, clouds, k,
                                                    scan, binned):
    import torch
    import pytorch_cluster_amd as pca
    before = pca.get_search_strategy()
    pca.set_search_strategy("auto")
    try:
        assert torch.ops.pytorch_cluster_amd.strategy_for(
            "knn", rows, queries, clouds, k) == "scan"
    finally:
        pca.set_search_strategy(before)


@pytest.mark.parametrize("clouds,rows,k,scan,binned", GRAPHS)
def test_auto_follows_the_length_of_the_lists(clouds, rows, k, scan, binned):
    import torch
    import pytorch_cluster_amd as pca
    pick = torch.ops.pytorch_cluster_amd.strategy_for
    before = pca.get_search_strategy()
    pca.set_search_strategy("auto")
    try:
        n = clouds * rows
        assert pick("knn", n, n, clouds, k) == \
            ("binned" if binned < scan else "scan")
        # longer lists of up to 32 places never turn a binned search into a scan
        picks = [pick("knn", n, n, clouds, i) for i in range(1, 33)]
        assert "scan" not in picks[picks.index("binned"):] \
            if "binned" in picks else True
        assert pick("knn", n, n, clouds) == pick("knn", n, n, clouds, 16)
    finally:
        pca.set_search_strategy(before)
