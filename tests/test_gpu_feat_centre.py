"""Feature-space rows away from the origin (feat_centre, csrc/knn_feat.hip): the
one-kernel search filters them less a mean row; what it returns is what the
oracle's exhaustive scan of the rows as they are returns, and it takes the time
of rows around the origin."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import pytorch_cluster_amd as pca  # noqa: E402
from gpu_common import (gpu_knn, gpu_radius, oracle_knn_edges,  # noqa: E402
                        ragged_ptrs)


@pytest.fixture(autouse=True)
def always(monkeypatch):
    monkeypatch.setenv("PCA_KNN_FEAT_SMALL", "1")


def rows(rng, kind, n, d):
    x = rng.standard_normal((n, d))
    if kind == "offset":
        x += 5.0
    elif kind == "far":
        x = x + 1000.0 * rng.standard_normal(d)
    elif kind == "at_the_limit":  # the mean is beyond 1e18 in some components
        x = x * 1e14 + 1e18
    elif kind == "grid":  # ties, and differences that are exact
        x = rng.integers(0, 3, (n, d)) + 100.0
    elif kind == "a_few_large":  # rows that leave the scale, and the samples
        x += 5.0
        x[:: max(1, n // 3)] *= 1e5
    elif kind == "not_finite":
        x += 5.0
        x[1::5, d // 2] = np.nan
        x[2::7, 0] = np.inf
        x[0] = np.nan  # (the first row is one of the samples)
    elif kind == "not_finite_elsewhere":
        x += 5.0
        x[n // 32 + 1::n // 16 + 1, d - 1] = -np.inf
    elif kind == "overflow":  # squares that overflow beside ordinary rows
        x += 5.0
        x[n // 2] = 3e38
    elif kind == "examples":  # two places
        x[: n // 2] += 8.0
        x[n // 2:] -= 2.0
    return x.astype(np.float32)


KINDS = ["offset", "far", "at_the_limit", "grid", "a_few_large", "not_finite",
         "not_finite_elsewhere", "overflow", "examples"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,m,d,k", [(700, 150, 64, 20), (33, 33, 9, 5),
                                     (900, 300, 127, 40), (31, 5, 30, 8),
                                     (1, 3, 128, 1)])
def test_knn_is_the_oracle_s(oracle, kind, n, m, d, k):
    rng = np.random.default_rng(n + d)
    x = rows(rng, kind, n, d)
    y = x if m == n else rows(rng, kind, m, d)
    for segments in ((1, 3) if n > 100 else (1,)):
        ptr_x, ptr_y = ragged_ptrs(rng, n, segments), ragged_ptrs(
            rng, m, segments)
        if m == n:
            ptr_y = ptr_x
        edges, dist = gpu_knn(x, y, ptr_x, ptr_y, k)
        want, want_dist = oracle_knn_edges(oracle, x, y, ptr_x, ptr_y, k)
        assert edges.shape == want.shape and (edges == want).all()
        assert (dist.view(np.uint32) == want_dist.view(np.uint32)).all()


@pytest.mark.parametrize("kind", ["offset", "grid", "not_finite", "overflow"])
@pytest.mark.parametrize("d", [12, 64, 128])
def test_radius_is_the_plain_scan_s(monkeypatch, kind, d):
    rng = np.random.default_rng(d)
    x, y = rows(rng, kind, 800, d), rows(rng, kind, 200, d)
    r = float(np.sqrt(1.6 * d))
    ptr = [0, 800], [0, 200]
    monkeypatch.setenv("PCA_RADIUS_FEAT", "1")
    got = gpu_radius(x, y, *ptr, r, 24)
    monkeypatch.setenv("PCA_RADIUS_FEAT", "0")
    want = gpu_radius(x, y, *ptr, r, 24)
    assert got.shape == want.shape and (got == want).all()
    assert kind == "overflow" or got.shape[1] > 0


def test_rows_away_from_the_origin_take_no_longer(monkeypatch):
    monkeypatch.delenv("PCA_KNN_FEAT_SMALL")
    x = torch.randn(32 * 1024, 128, device="cuda")
    batch = torch.arange(32, device="cuda").repeat_interleave(1024)

    def us(v):
        best = float("inf")
        for _ in range(12):
            torch.cuda.synchronize()
            t = time.perf_counter()
            pca.knn_graph(v, 20, batch)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        return 1e6 * best

    # (without the centre 20 standard deviations took several times as long)
    there, here = us(x + 20.0), us(x)
    assert there < 1.3 * here, (there, here)
