"""The calls by which this framework's speed is followed over its whole range.

Every case goes through a public entry point the way a program calls it: host arrays into
``fps_sampling``, ``bucket_fps_kdline_sampling`` and ``fps_npdu_sampling``, GPU tensors into
``fps_sampling_tensor``, many clouds in one ``DeviceBatch``, and a burst of requests on a serving
loop.  ``listed()`` holds one case for each use, ``draw()`` further sizes of the same ranges.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import fpsample_amd as fpsample
from fpsample_amd import device as D
from fpsample_amd.batch import DeviceBatch
from fpsample_amd.serve import Server


def listed():
    return [
        # A region crop inside a network's forward pass: the smallest call, all latency.
        {"name": "crop1k", "entry": "host", "shape": "uniform", "n": 1024, "d": 3, "m": 256},
        # One object of a shape dataset as numpy hands it over (float64): the small bench case.
        {"name": "object4k", "entry": "host", "shape": "uniform", "n": 4096, "d": 3, "m": 1024,
         "f64": True},
        # A lidar-sized scan that is already on the GPU, picks and their coordinates wanted.
        {"name": "scan50k", "entry": "tensor", "shape": "uniform", "n": 50_000, "d": 3, "m": 4096,
         "points": True},
        # Thinning a cloud to half its points: long runs of picks over a mid-sized cloud.
        {"name": "half100k", "entry": "host", "shape": "uniform", "n": 100_000, "d": 3,
         "m": 50_000, "f64": True},
        # The KD-line order and its tie rule on host arrays, with the tree built per call.
        {"name": "kdline50k", "entry": "kdline", "shape": "uniform", "n": 50_000, "d": 3,
         "m": 4096, "h": 7},
        # The windowed update at its default window.
        {"name": "npdu50k", "entry": "npdu", "shape": "uniform", "n": 50_000, "d": 3, "m": 4096},
        # The headline cloud: a million clustered points on the GPU.
        {"name": "gauss1m", "entry": "tensor", "shape": "gauss", "n": 1 << 20, "d": 3,
         "m": 16_384},
        # The largest cloud, beyond the register file, full of equal distances and duplicates.
        {"name": "lattice16m", "entry": "tensor", "shape": "lattice", "n": 1 << 24, "d": 3,
         "m": 4096},
        # Points with normals: six coordinates, a ragged number of points.
        {"name": "normals6d", "entry": "tensor", "shape": "surface", "n": 100_003, "d": 6,
         "m": 4096},
        # Feature vectors, for a subset that covers them: beyond the dimensions with own kernels.
        {"name": "feature32d", "entry": "tensor", "shape": "normal", "n": 20_000, "d": 32,
         "m": 2000},
        # A training batch of ragged clouds in one launch.
        {"name": "batch256", "entry": "batch", "clouds": 256, "lo": 1024, "hi": 65_536, "d": 3,
         "part": 4},
        # A burst of mixed requests on the serving loop.
        {"name": "serve24", "entry": "serve", "requests": 24, "lo": 1024, "hi": 131_072},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    entry = rng.choice(["host", "host", "tensor", "tensor", "tensor", "kdline", "npdu", "batch",
                        "serve"])
    if entry == "batch":
        d = rng.choice([3, 3, 2])
        return {"entry": entry, "clouds": _log_int(rng, 8, 256 if d == 3 else 48), "lo": 1024,
                "hi": rng.choice([4096, 16_384, 65_536] if d == 3 else [4096, 16_384]), "d": d,
                "part": rng.choice([4, 8, 16])}
    if entry == "serve":
        return {"entry": entry, "requests": rng.randint(4, 24), "lo": 1024,
                "hi": _log_int(rng, 16_384, 131_072)}
    if entry == "tensor":
        d = rng.choice([3, 3, 3, 2, 4, 6, 8, 32])
        n = _log_int(rng, 2048, {3: 4_000_000, 32: 60_000}.get(d, 300_000))
        shape = {3: rng.choice(["uniform", "gauss", "surface", "lattice"]), 6: "surface",
                 32: "normal"}.get(d, "uniform")
        m = min(n // 2, _log_int(rng, 256, 2048 if d == 32 else 16_384))
        return {"entry": entry, "shape": shape, "n": n, "d": d, "m": m,
                "points": rng.random() < 0.3, "soa": rng.random() < 0.3}
    n = _log_int(rng, 1024, 150_000)
    m = min(_log_int(rng, 128, 20_000), n // 2)
    case = {"entry": entry, "shape": rng.choice(["uniform", "gauss", "surface"]), "n": n,
            "d": 3, "m": m}
    if entry == "host":
        case["f64"] = rng.random() < 0.5
        case["starts"] = rng.choice([1, 1, 4])
    if entry == "kdline":
        case["h"] = rng.choice([3, 5, 7, 9])
    return case


def _cloud(rng: np.random.Generator, shape: str, n: int, d: int) -> np.ndarray:
    """A host cloud, float64."""
    if shape == "gauss":  # 64 clusters in the unit cube
        centers = rng.random((64, d))
        return centers[rng.integers(0, 64, n)] + 0.02 * rng.standard_normal((n, d))
    if shape == "surface":  # a sphere seen with noise
        v = rng.standard_normal((n, d))
        return v / np.linalg.norm(v, axis=1, keepdims=True) + 0.01 * rng.standard_normal((n, d))
    return rng.random((n, d))


def _tensor_cloud(seed: int, shape: str, n: int, d: int) -> torch.Tensor:
    """The same distributions made on the GPU, (n, d) float32."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if shape == "gauss":
        centers = torch.rand((64, d), generator=g, device="cuda")
        label = torch.randint(0, 64, (n,), generator=g, device="cuda")
        return centers[label] + 0.02 * torch.randn((n, d), generator=g, device="cuda")
    if shape == "surface":  # positions on a noisy sphere and, in 6-D, their unit normals
        v = torch.randn((n, 3), generator=g, device="cuda")
        v = v / v.norm(dim=1, keepdim=True)
        p = v + 0.01 * torch.randn((n, 3), generator=g, device="cuda")
        return torch.cat([p, v], dim=1).contiguous() if d == 6 else p
    if shape == "lattice":  # integer sites of a cube, a quarter of the points exact copies
        side = max(2, round(n ** (1.0 / 3.0)))
        sites = torch.randperm(side ** 3, generator=g, device="cuda")[: n * 3 // 4]
        more = torch.randint(0, sites.numel(), (n - sites.numel(),), generator=g, device="cuda")
        code = torch.cat([sites, sites[more]])
        code = code[torch.randperm(n, generator=g, device="cuda")]
        return torch.stack([code // (side * side), code // side % side, code % side],
                           dim=1).float().contiguous()
    if shape == "normal":
        return torch.randn((n, d), generator=g, device="cuda")
    return torch.rand((n, d), generator=g, device="cuda")


def _ragged(rng: np.random.Generator, count: int, lo: int, hi: int, d: int):
    """Clouds of sizes spread evenly over the logarithm of lo..hi (the same for every seed) in a
    mixed order, cubes and noisy spheres in turn; with each its rank by size from the largest."""
    sizes = [int(lo * (hi / lo) ** ((count - i) / count)) for i in range(count)]
    ranks = np.random.default_rng(count).permutation(count)
    clouds = [_cloud(rng, "surface" if i % 2 else "uniform", sizes[r], d).astype(np.float32)
              for i, r in enumerate(ranks)]
    return clouds, [int(r) for r in ranks]


_SERVER = None


def _server() -> Server:
    """The one serving loop that a serving program keeps."""
    global _SERVER
    if _SERVER is None:
        _SERVER = Server(hbm_budget_bytes=4 << 30)
    return _SERVER


def prepare(case, seed):
    entry = case["entry"]
    rng = np.random.default_rng(seed)
    state = {"case": case, "entry": entry}
    if entry == "tensor":
        pc = _tensor_cloud(seed, case["shape"], case["n"], case["d"])
        # Column-major storage (one array per coordinate), as some loaders keep it.
        state["pc"] = pc.t().contiguous().t() if case.get("soa") else pc
        state["start"] = int(rng.integers(0, case["n"]))
    elif entry == "batch":
        clouds, _ = _ragged(rng, case["clouds"], case["lo"], case["hi"], case["d"])
        picks = [max(1, c.shape[0] // case["part"]) for c in clouds]
        state["batch"] = DeviceBatch(clouds, picks, [0] * len(clouds))
        # The object's own output buffer, seen as a tensor (uint64 picks, cloud after cloud).
        # The object frees that buffer when it goes, so the tensor keeps the object.
        state["out"] = torch.as_tensor(_Int64View(state["batch"]), device="cuda")
        state["out"].owner = state["batch"]
    elif entry == "serve":
        clouds, ranks = _ragged(rng, case["requests"], case["lo"], case["hi"], 3)
        state["requests"] = [(c, c.shape[0] // (2, 4, 8)[r % 3]) for c, r in zip(clouds, ranks)]
        state["server"] = _server()
    else:
        pc = _cloud(rng, case["shape"], case["n"], case["d"])
        state["pc"] = pc if case.get("f64") else pc.astype(np.float32)
        starts = rng.choice(case["n"], case.get("starts", 1), replace=False)
        state["start"] = int(starts[0]) if len(starts) == 1 else [int(s) for s in starts]
    return state


class _Int64View:
    """A batch's uint64 output buffer shown to torch as int64 (the bits are the same)."""

    def __init__(self, batch):
        self.batch = batch
        self.__cuda_array_interface__ = {**batch.d_out.__cuda_array_interface__,
                                         "typestr": "<i8"}


def run(state):
    case, entry = state["case"], state["entry"]
    if entry == "host":
        return fpsample.fps_sampling(state["pc"], case["m"], start_idx=state["start"]).view(np.int64)
    if entry == "kdline":
        return fpsample.bucket_fps_kdline_sampling(state["pc"], case["m"], case["h"],
                                                   start_idx=state["start"]).view(np.int64)
    if entry == "npdu":
        return fpsample.fps_npdu_sampling(state["pc"], case["m"],
                                          start_idx=state["start"]).view(np.int64)
    if entry == "tensor":
        idx, points = D.fps_sampling_tensor(state["pc"], case["m"], state["start"],
                                            return_points=bool(case.get("points")))
        return [idx] if points is None else [idx, points]
    if entry == "batch":
        # The picks stay on the GPU; status() is what tells the caller that they are there.
        state["batch"].run()
        state["batch"].status()
        return state["out"]
    server = state["server"]
    ids = [server.submit(pc, m) for pc, m in state["requests"]]
    return [server.wait(i)[0].view(np.int64) for i in ids]


def work(case):
    """Every coordinate read once and every pick written once; one distance for each point.

    That is all that no order of the work can avoid: how many further distances a run takes
    depends on how it prunes, and what its picks cost is a chain of m - 1 dependent steps.
    """
    if case["entry"] in ("batch", "serve"):
        count = case.get("clouds") or case["requests"]
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        n, d = count * mean, case.get("d", 3)
        m = n / case.get("part", 4)
    else:
        n, d, m = case["n"], case["d"], case["m"]
    points = d * 4 * m if case.get("points") else 0
    return {"bytes": 4 * n * d + 8 * m + points, "flops": n * (3 * d - 1)}


def exact(case, seed):
    """The outputs are indices and copies of input rows: nothing in them is rounded."""
    return None
