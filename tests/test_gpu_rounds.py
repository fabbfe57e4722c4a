"""GPU tests of the threshold rounds: every pick against the oracle at the sizes where the
blocks, the candidate lists and the bound can go wrong.  Picks are indices: they are equal."""
import os

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def log(msg):
    print(msg, flush=True)


@pytest.fixture
def rounds_env(monkeypatch):
    def set_(value):
        monkeypatch.setenv("FPSX_ROUNDS", value)
    return set_


def run(pc, m, starts, lowest=False):
    """(picks, their coordinates) by the device entry, row-major points in place."""
    from fpsample_amd import device as D

    n, d = pc.shape
    st = np.atleast_1d(np.asarray(starts, np.uint64))
    rows, ds = D.DeviceArray.from_numpy(pc), D.DeviceArray.from_numpy(st)
    out, pts = D.DeviceArray((m,), np.uint64), D.DeviceArray((m, d), np.float32)
    tie = D.TIE_LOWEST if lowest else D.TIE_HIGHEST
    init = float(np.finfo(np.float32).max) if lowest else float("inf")
    assert D.call_info(n, d, tie=tie, n_samples=m)["kind"] == "rounds"
    D.fps_sampling_device_strided(rows, d, 1, n, d, m, ds, st.size, out, pts, tie=tie, init=init)
    D.device_status()
    return out.numpy(), pts.numpy()


def check(pc, m, starts, name):
    log(f"rounds {name} n={len(pc)} d={pc.shape[1]} m={m} env={os.environ.get('FPSX_ROUNDS')}")
    got, pts = run(pc, m, starts)
    want = O.fps(pc, m, starts)
    np.testing.assert_array_equal(got, want, err_msg=name)
    np.testing.assert_array_equal(pts, pc[want.astype(np.int64)], err_msg=name + " coordinates")
    if np.size(starts) == 1:
        got, _ = run(pc, m, starts, lowest=True)
        want = O.fps_ex(pc, m, int(starts), lowest=True, init=float(np.finfo(np.float32).max))
        np.testing.assert_array_equal(got, want, err_msg=name + " lowest")


# Points per lane : workgroups, with and without spatial order.
SHAPES = ["1:1", "1:3", "1:64:160:1", "1:200", "4:5", "4:64:256:0", "8:2:1", "8:16"]


@pytest.mark.parametrize("shape", SHAPES)
def test_rounds_block_edges(gpu, rounds_env, shape):
    # Around whole blocks of 64, 256 and 512 points and the smallest clouds.
    rounds_env(shape)
    rng = np.random.default_rng(60)
    for n, m in ((1, 1), (2, 2), (63, 63), (64, 40), (65, 65), (257, 100), (511, 300), (513, 513),
                 (4097, 700)):
        check(rng.random((n, 3)).astype(np.float32), m, int(rng.integers(n)), "edge")


@pytest.mark.parametrize("shape", SHAPES)
def test_rounds_ties_special_values_and_prefixes(gpu, rounds_env, shape):
    # Far more equal distances than a round's candidates, duplicates to the last pick (the
    # best key stays), NaN and infinite coordinates, squares that overflow, and forced
    # prefixes below, at and beyond the 256 picks a round can hold.
    rounds_env(shape)
    rng = np.random.default_rng(61)
    check(rng.integers(0, 24, (9000, 3)).astype(np.float32), 3000, 5, "lattice")
    check(np.repeat(rng.integers(0, 5, (700, 3)), 3, axis=0).astype(np.float32), 2100, 7, "dups")
    check(np.ones((3000, 3), np.float32), 400, 11, "same")
    sp = (rng.random((5000, 3)) * 4e19).astype(np.float32)
    sp[9] = np.inf
    sp[10, 1] = -np.inf
    check(sp, 500, 0, "overflow")
    sp[[5, 700, 4000]] = np.nan
    check(sp, 500, 0, "nan")
    check((rng.random((5000, 3)) * 1e-21).astype(np.float32), 500, 3, "denormal")
    pc = rng.random((6000, 3)).astype(np.float32)
    for count in (2, 255, 256, 257, 700):
        check(pc, 700, [int(v) for v in rng.integers(0, 6000, count)], f"prefix {count}")


def test_rounds_planner_sizes(gpu):
    # The planner's own shapes on both sides of each of its lines.
    rng = np.random.default_rng(62)
    for n, d, m in ((512, 3, 192), (512, 8, 64), (1024, 3, 256), (1025, 3, 600), (4097, 3, 600),
                    (8193, 3, 700), (16385, 2, 600), (65536, 3, 1500), (65537, 3, 1500),
                    (262145, 3, 300), (524289, 3, 600), (300000, 7, 70), ((1 << 22) + 1, 3, 192)):
        check(rng.random((n, d)).astype(np.float32), m, int(rng.integers(n)), "planner")


@pytest.mark.parametrize("d", [1, 2, 4, 5, 6, 7, 8])
def test_rounds_dimensions(gpu, rounds_env, d):
    # Every dimension with a kernel, one and several blocks per wave, with and without order.
    rng = np.random.default_rng(63 + d)
    for shape in ("4:3:100:1" if d == 1 else "1:40:100:1", "4:2:160:1", "4:64:60:0"):
        rounds_env(shape)
        check(rng.random((9001, d)).astype(np.float32), 900, int(rng.integers(9001)), "uniform")
        check(rng.integers(0, 4, (3000, d)).astype(np.float32), 1500, 5, "lattice")
        sp = (rng.random((3000, d)) * 4e19).astype(np.float32)
        sp[[7, 900]] = np.nan
        sp[11, d - 1] = np.inf
        check(sp, 300, 1, "special")


@pytest.mark.parametrize("d", [9, 32, 63, 256])
def test_rounds_any_dimension(gpu, rounds_env, d):
    # Beyond eight dimensions: one and several workgroups, several blocks of one workgroup,
    # dimensions around the unrolled four, the largest; prefixes beyond a round's 128 picks.
    rng = np.random.default_rng(80 + d)
    for shape in ("1:1", "1:3:100", "1:40:30"):
        rounds_env(shape)
        for n, m in ((1, 1), (65, 65), (2001, 300)):
            check(rng.standard_normal((n, d)).astype(np.float32), m, int(rng.integers(n)), "any")
        check(rng.integers(0, 2, (700, d)).astype(np.float32), 700, 5, "ties")
        sp = (rng.random((900, d)) * 4e19).astype(np.float32)
        sp[11, d - 1] = np.inf
        check(sp, 100, 1, "overflow")
        sp[[7, 800], 0] = np.nan
        check(sp, 100, 1, "nan")
        pc = rng.random((1500, d)).astype(np.float32)
        for count in (128, 129, 300):
            check(pc, 330, [int(v) for v in rng.integers(0, 1500, count)], f"prefix {count}")


@pytest.mark.parametrize("n", [8191, 8192, 8193, 20000, 70001])
def test_rounds_order_sizes(gpu, rounds_env, n):
    # The order's one-workgroup form, its last size, several chunks, a ragged last chunk;
    # clouds in one bucket but for an outlier, on a line, and with values it cannot place.
    rounds_env("1:16:160:1")
    rng = np.random.default_rng(n)
    tight = (0.5 + 1e-4 * rng.random((n, 3))).astype(np.float32)
    tight[n // 2] = 1e6
    line = np.zeros((n, 3), np.float32)
    line[:, 1] = rng.random(n)
    odd = rng.random((n, 3)).astype(np.float32)
    odd[[3, n - 1], 0] = np.nan
    odd[5, 2] = np.inf
    odd[6] = -np.inf
    for name, pc in (("tight", tight), ("line", line), ("odd", odd)):
        check(pc, 400, 9, name)


@pytest.mark.parametrize("n,d,m", [(1000, 3, 250), (20_001, 3, 700), (70_001, 6, 300),
                                   (3001, 20, 200)])
def test_rounds_under_capture(gpu, n, d, m):
    # A call captured after one that left its buffers, replayed on new points each time.
    import torch

    from fpsample_amd import device as D

    log(f"capture n={n} d={d} m={m}")
    rng = np.random.default_rng(66)
    pts = torch.zeros((n, d), dtype=torch.float32, device="cuda")
    start = torch.zeros(1, dtype=torch.int64, device="cuda")
    out = torch.zeros(m, dtype=torch.int64, device="cuda")

    def call(stream):
        D.fps_sampling_device_strided(pts.data_ptr(), d, 1, n, d, m, start.data_ptr(), 1,
                                      out.data_ptr(), stream=stream)

    side = torch.cuda.Stream()
    pts.copy_(torch.from_numpy(rng.random((n, d), dtype=np.float32)))
    torch.cuda.synchronize()
    call(side.cuda_stream)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(torch.cuda.current_stream().cuda_stream)
    for rep in range(3):
        pc = rng.random((n, d), dtype=np.float32)
        pts.copy_(torch.from_numpy(pc))
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy().astype(np.uint64), O.fps(pc, m, 0),
                                      err_msg=f"replay {rep}")
