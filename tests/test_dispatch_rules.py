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
