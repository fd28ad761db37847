"""The work a user has this package do: sizes, inputs and calls to be timed.

A case is a dict of plain values; ``"path"`` says which entry point it goes
through, the rest are its sizes and options.  Inputs are on the GPU before a
pass starts; a pass is one call of ``knn``, ``knn_graph``, ``radius_graph``,
``nearest`` or ``fps`` under the default search strategy, as a training or
inference step makes it.  All outputs are row numbers, so any two correct
implementations return the same ones.

The sizes of ragged batches belong to the case and the points to the seed, so
that a case has the same number of edges whatever the seed.
"""
import math

import torch

import pytorch_cluster_amd as pca

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one point cloud without a batch vector, as an interactive program or
        # an inference call on a single object builds its graph: all latency
        {"name": "one_cloud", "path": "knn_graph", "clouds": 1,
         "points": 1024, "ragged": False, "k": 16},
        # input layer of a point-cloud network: a batch of objects, one graph
        {"name": "clouds", "path": "knn_graph", "clouds": 16, "points": 4096,
         "ragged": False, "k": 20},
        # neighbourhoods of fixed radius in larger, unevenly filled clouds,
        # many more rows in range than the limit lets through
        {"name": "clustered_radius", "path": "radius_graph", "clouds": 8,
         "points": 16384, "ragged": False, "r": 0.05, "limit": 32},
        # a mini-batch of many small graphs (molecule-sized point sets) whose
        # edges come from a cutoff radius
        {"name": "many_tiny_graphs", "path": "tiny_graphs", "graphs": 1000,
         "smallest": 5, "largest": 65, "r": 5.0, "limit": 32},
        # ragged LiDAR-like scans, every fourth point looks for neighbours:
        # large, very uneven density
        {"name": "lidar_knn", "path": "lidar_knn", "scans": 8,
         "smallest": 60000, "largest": 200000, "stride": 4, "k": 16},
        # the largest call: neighbours of query vectors among stored ones
        {"name": "feature_search", "path": "features", "rows": 200000,
         "queries": 50000, "d": 128, "k": 32, "cosine": False},
        # dynamic graph of a point-cloud network: every layer of every step
        # builds it again, in feature space
        {"name": "feature_graph", "path": "feature_graph", "clouds": 32,
         "points": 1024, "ragged": False, "d": 64, "k": 20, "dtype": "f32"},
        # the same under mixed precision, clouds of different sizes
        {"name": "feature_graph_f16", "path": "feature_graph", "clouds": 24,
         "points": 1300, "ragged": True, "d": 64, "k": 20, "dtype": "f16"},
        # every point of the scans is assigned to the nearest sampled one
        # (pooling, label transfer)
        {"name": "nearest_points", "path": "lidar_nearest", "scans": 8,
         "smallest": 60000, "largest": 200000, "stride": 8},
        # feature vectors assigned to the entries of a code book
        {"name": "nearest_codes", "path": "codes", "rows": 1 << 20,
         "codes": 4096, "d": 64},
        # sampling of a set-abstraction layer
        {"name": "fps_clouds", "path": "fps", "clouds": 16, "points": 4096,
         "ragged": False, "ratio": 0.25},
        # key points of whole scans: a few thousand out of a hundred thousand
        {"name": "fps_scans", "path": "lidar_fps", "scans": 8,
         "smallest": 60000, "largest": 200000, "ratio": 0.02},
    ]


def _log(rng, low, high):
    """A whole number between low and high, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    path = rng.choice(["knn_graph", "radius_graph", "tiny_graphs",
                       "lidar_knn", "features", "feature_graph",
                       "lidar_nearest", "codes", "fps", "lidar_fps"])
    c = {"path": path}
    if path in ("knn_graph", "radius_graph", "fps"):
        top = {"knn_graph": 65536, "radius_graph": 32768, "fps": 16384}[path]
        c["points"] = _log(rng, 300, top)
        c["clouds"] = _log(rng, 1, max(1.0, min(64, 262144 // c["points"])))
        c["ragged"] = rng.random() < 0.5
        if path == "knn_graph":
            c["k"] = rng.randint(4, 32)
        elif path == "radius_graph":
            c["r"] = round(rng.uniform(0.02, 0.1), 4)
            c["limit"] = rng.choice([8, 16, 32, 64])
        else:
            c["ratio"] = round(rng.uniform(0.05, 0.5), 3)
    elif path == "tiny_graphs":
        c["graphs"] = _log(rng, 16, 4096)
        c["smallest"] = rng.randint(1, 12)
        c["largest"] = rng.randint(20, 120)
        c["r"] = round(rng.uniform(2.0, 8.0), 2)
        c["limit"] = rng.choice([16, 32, 32, 64])
    elif path in ("lidar_knn", "lidar_nearest", "lidar_fps"):
        c["scans"] = rng.randint(1, 8)
        c["smallest"] = _log(rng, 18000, 60000)
        c["largest"] = _log(rng, 60000, 200000)
        if path == "lidar_fps":
            c["ratio"] = round(rng.uniform(0.004, 0.02), 4)
        else:
            c["stride"] = rng.randint(2, 16)
        if path == "lidar_knn":
            c["k"] = rng.randint(3, 32)
    elif path == "features":
        c["rows"] = _log(rng, 5000, 200000)
        c["queries"] = _log(rng, 500, 50000)
        c["d"] = rng.randint(12, 128)
        c["k"] = rng.randint(5, 32)
        c["cosine"] = rng.random() < 0.4
    elif path == "feature_graph":
        c["points"] = _log(rng, 200, 2048)
        c["clouds"] = _log(rng, 4, min(64, 65536 // c["points"]))
        c["ragged"] = rng.random() < 0.5
        c["d"] = rng.choice([32, 48, 64, 64, 96, 128])
        c["k"] = rng.randint(8, 40)
        c["dtype"] = rng.choice(["f32", "f32", "f16", "bf16"])
    else:
        c["rows"] = _log(rng, 10000, 1 << 20)
        c["codes"] = _log(rng, 64, 4096)
        c["d"] = rng.randint(16, 128)
    return c


# ---- inputs -----------------------------------------------------------------


def _sizes(count, low, high):
    g = torch.Generator().manual_seed(count * 1000003 + low * 1009 + high)
    return torch.randint(low, high + 1, (count,), generator=g).tolist()


def _cloud_sizes(case):
    if not case["ragged"]:
        return [case["points"]] * case["clouds"]
    return _sizes(case["clouds"], max(1, case["points"] // 2),
                  case["points"] + case["points"] // 2)


def _batch(sizes):
    ids = torch.arange(len(sizes)).repeat_interleave(torch.tensor(sizes))
    return ids.cuda()


def _shuffled(points, ids, g):
    """The rows of every example in another order and mirrored along some
    axes: other points, and exactly as many pairs within any distance."""
    order = torch.randperm(ids.numel(), generator=g, device="cuda")
    order = order[torch.argsort(ids[order], stable=True)]
    signs = torch.randint(0, 2, (int(ids[-1]) + 1, 3), generator=g,
                          device="cuda") * 2.0 - 1.0
    return (points[order] * signs[ids]).contiguous()


def _clustered(sizes):
    """Every cloud a mixture of 32 narrow Gaussians in the unit cube."""
    g = torch.Generator(device="cuda").manual_seed(len(sizes))
    ids = _batch(sizes)
    centres = torch.rand(len(sizes) * 32, 3, generator=g, device="cuda")
    which = torch.randint(0, 32, (ids.numel(),), generator=g, device="cuda")
    noise = torch.randn(ids.numel(), 3, generator=g, device="cuda")
    return centres[ids * 32 + which] + 0.02 * noise, ids


def _scans(case, g):
    """LiDAR-like scans: ranges with density proportional to 1 / rho^2 on
    [1, 80] m, 64 elevation beams, 2 cm vertical noise."""
    sizes = _sizes(case["scans"], case["smallest"], case["largest"])
    ids = _batch(sizes)
    n = ids.numel()
    theta = torch.linspace(math.radians(-25.0), math.radians(3.0), 64,
                           device="cuda")
    theta = theta[torch.randint(0, 64, (n,), generator=g, device="cuda")]
    u = torch.rand(n, generator=g, device="cuda")
    rho = 1.0 / (1.0 - u * (1.0 - 1.0 / 80.0))
    phi = 2.0 * math.pi * torch.rand(n, generator=g, device="cuda")
    z = rho * torch.tan(theta)
    z = z + 0.02 * torch.randn(n, generator=g, device="cuda")
    points = torch.stack([rho * torch.cos(phi), rho * torch.sin(phi), z], 1)
    return points.contiguous(), ids, sizes


def _every(points, ids, sizes, stride):
    """Every stride-th point of each scan."""
    starts = [0]
    for n in sizes:
        starts.append(starts[-1] + n)
    rows = torch.cat([torch.arange(a, b, stride)
                      for a, b in zip(starts, starts[1:])]).cuda()
    return points[rows].contiguous(), ids[rows].contiguous()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    path = case["path"]
    s = {"case": case}
    if path in ("knn_graph", "fps"):
        sizes = _cloud_sizes(case)
        s["x"] = torch.rand(sum(sizes), 3, generator=g, device="cuda")
        s["batch"] = _batch(sizes) if case["clouds"] > 1 else None
    elif path == "radius_graph":
        x, s["batch"] = _clustered(_cloud_sizes(case))
        s["x"] = _shuffled(x, s["batch"], g)
    elif path == "tiny_graphs":
        sizes = _sizes(case["graphs"], case["smallest"], case["largest"])
        s["batch"] = _batch(sizes)
        # one point in ten cubic units, whatever the size of the graph
        edge = (10.0 * torch.tensor(sizes, dtype=torch.float32)) ** (1.0 / 3)
        fixed = torch.Generator(device="cuda").manual_seed(len(sizes))
        x = torch.rand(sum(sizes), 3, generator=fixed, device="cuda")
        s["x"] = _shuffled(x * edge.cuda()[s["batch"], None], s["batch"], g)
    elif path in ("lidar_knn", "lidar_nearest"):
        s["x"], s["batch"], sizes = _scans(case, g)
        s["y"], s["batch_y"] = _every(s["x"], s["batch"], sizes,
                                      case["stride"])
    elif path == "lidar_fps":
        s["x"], s["batch"], _ = _scans(case, g)
    elif path == "features":
        s["x"] = torch.randn(case["rows"], case["d"], generator=g,
                             device="cuda")
        s["y"] = torch.randn(case["queries"], case["d"], generator=g,
                             device="cuda")
    elif path == "feature_graph":
        sizes = _cloud_sizes(case)
        s["batch"] = _batch(sizes)
        s["x"] = torch.randn(sum(sizes), case["d"], generator=g,
                             device="cuda").to(DTYPES[case["dtype"]])
    else:
        codes = torch.randn(case["codes"], case["d"], generator=g,
                            device="cuda")
        which = torch.randint(0, case["codes"], (case["rows"],), generator=g,
                              device="cuda")
        noise = torch.randn(case["rows"], case["d"], generator=g,
                            device="cuda")
        s["x"], s["y"] = codes[which] + 0.5 * noise, codes
    return s


# ---- one pass ---------------------------------------------------------------


def run(s):
    c = s["case"]
    path = c["path"]
    if path in ("knn_graph", "feature_graph"):
        return pca.knn_graph(s["x"], c["k"], s["batch"])
    if path in ("radius_graph", "tiny_graphs"):
        return pca.radius_graph(s["x"], c["r"], s["batch"],
                                max_num_neighbors=c["limit"])
    if path == "lidar_knn":
        return pca.knn(s["x"], s["y"], c["k"], s["batch"], s["batch_y"])
    if path == "features":
        return pca.knn(s["x"], s["y"], c["k"], cosine=c["cosine"])
    if path == "lidar_nearest":
        return pca.nearest(s["x"], s["y"], s["batch"], s["batch_y"])
    if path == "codes":
        return pca.nearest(s["x"], s["y"])
    return pca.fps(s["x"], s["batch"], c["ratio"], random_start=False)


def work(case):
    """Points, example ids and queries read once, row numbers written once.
    In feature space the distances of all pairs are a contraction (2 d per
    pair); points of three dimensions need the distances of what is returned
    (fps: one per row), since rows far away can be left out by their place."""
    path = case["path"]
    d = case.get("d", 3)
    size = {"f16": 2, "bf16": 2}.get(case.get("dtype"), 4)
    flops = 0.0
    if path in ("knn_graph", "radius_graph", "feature_graph", "fps"):
        rows = case["clouds"] * case["points"]
    elif path == "tiny_graphs":
        rows = case["graphs"] * (case["smallest"] + case["largest"]) / 2
    elif path in ("features", "codes"):
        rows = case["rows"]
    else:
        rows = case["scans"] * (case["smallest"] + case["largest"]) / 2
    read = rows * d * size
    if path not in ("features", "codes"):
        read += rows * 8
    if path in ("knn_graph", "feature_graph"):
        out = rows * case["k"] * 16
        flops = 3 * d * rows * case["k"]
        if path == "feature_graph":
            flops = 2.0 * d * rows * case["points"]
    elif path in ("radius_graph", "tiny_graphs"):
        found = case["limit"]
        if path == "tiny_graphs":  # at most the other points of the graph
            found = min(found, (case["smallest"] + case["largest"]) / 2)
        out = rows * found * 16
        flops = 3 * d * rows * found
    elif path == "lidar_knn":
        read += rows / case["stride"] * 20
        out = rows / case["stride"] * case["k"] * 16
        flops = 3 * d * rows / case["stride"] * case["k"]
    elif path == "features":
        read += case["queries"] * d * size
        out = case["queries"] * case["k"] * 16
        flops = 2.0 * d * rows * case["queries"]
    elif path == "lidar_nearest":
        read += rows / case["stride"] * 20
        out = rows * 8
        flops = 3 * d * rows
    elif path == "codes":
        read += case["codes"] * d * size
        out = rows * 8
        flops = 2.0 * d * rows * case["codes"]
    else:
        out = rows * case["ratio"] * 8
        flops = 3 * d * rows
    return {"bytes": read + out, "flops": flops}


def tolerance(case):
    return "exact"
