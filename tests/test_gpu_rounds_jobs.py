"""GPU tests of the threshold rounds over many clouds in one launch (fps_rounds_jobs)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_teams_and_a_queue_of_clouds(gpu):
    # More members than workgroups: some workgroups form teams, which wait for each other, and
    # go on to clouds of their own afterwards.
    from fpsample_amd.batch import DeviceBatch

    rng = np.random.default_rng(20)
    sizes = [50_000] * 12 + [9000] * 30 + [int(n) for n in rng.integers(1, 900, 500)]
    clouds = [rng.random((n, 3)).astype(np.float32) for n in sizes]
    ms = [max(1, n // 8) for n in sizes]
    b = DeviceBatch(clouds, ms, [0] * len(sizes))
    info = b.info()
    print(f"queue: {info}", flush=True)
    assert info["ppt"] == 4 and info["members"] > info["grid"] and info["members"] > len(sizes)
    want = [O.fps(pc, m, 0) for pc, m in zip(clouds, ms)]
    for rep in range(3):
        b.run()
        b.status()
        for i, (g, w) in enumerate(zip(b.picks(), want)):
            np.testing.assert_array_equal(g, w, err_msg=f"run {rep} cloud {i} n={sizes[i]}")
    b.close()


@pytest.mark.parametrize("d", [2, 3])
@pytest.mark.parametrize("passes", [False, True], ids=["rounds", "passes"])
def test_status_before_the_first_run(gpu, monkeypatch, d, passes):
    # On memory that held other values before: a batch that has not run has not failed.
    from fpsample_amd import device as D
    from fpsample_amd.batch import DeviceBatch

    if passes:
        monkeypatch.setenv("FPSX_NO_ROUNDS", "1")
    rng = np.random.default_rng(21)
    clouds = [rng.random((n, d)).astype(np.float32) for n in (5000, 300)]
    for size in (4096, 16_384, 65_536, 1 << 18, 1 << 20, 1 << 22):
        filled = [D.DeviceArray.from_numpy(np.full(size, 255, np.uint8)) for _ in range(4)]
        for a in filled:
            a.free()
        b = DeviceBatch(clouds, [500, 100], [0, 0], graph=False)
        b.status()
        b.close()


@pytest.mark.parametrize("n,m,rounds", [(5000, 63, False), (5000, 64, True), (8193, 95, False),
                                        (8193, 96, True), (300, 8, False)])
def test_batches_of_few_picks(gpu, n, m, rounds):
    # Both sides of the line below which 3-D batches take the pass kernels (8 points a thread).
    import fpsample_amd as F
    from fpsample_amd.batch import DeviceBatch

    rng = np.random.default_rng(n + m)
    clouds = [rng.random((k, 3)).astype(np.float32) for k in (n, 200, n // 2)]
    ms = [m, 7, m // 2]
    want = [O.fps(pc, k, 1) for pc, k in zip(clouds, ms)]
    b = DeviceBatch(clouds, ms, [1, 1, 1])
    assert b.info()["ppt"] == (4 if rounds else 8)
    b.run()
    b.status()
    for g, o, w in zip(b.picks(), F.fps_sampling_batch(clouds, ms, 1), want):
        np.testing.assert_array_equal(g, w)
        np.testing.assert_array_equal(o, w)
    b.close()


def special_clouds():
    """NaN, infinite and overflowing coordinates, and clouds whose last points are at distance 0,
    so that a run ends on one point taken again and again."""
    rng = np.random.default_rng(22)
    for n in (200, 3000, 40_000):
        sp = (rng.random((n, 3)) * 4e19).astype(np.float32)
        sp[9] = np.inf
        sp[10, 1] = -np.inf
        yield sp, min(n, 300), 0
        sp = sp.copy()
        sp[[5, 70, n - 1]] = np.nan
        yield sp, min(n, 300), 3
        yield (rng.random((n, 3)) * 1e-21).astype(np.float32), min(n, 400), 1
        yield np.ones((n, 3), np.float32), 77, n // 2
        yield rng.integers(0, 4, (n, 3)).astype(np.float32), min(n, 103), 2  # 64 places
        yield rng.integers(0, 30, (n, 3)).astype(np.float32), min(n, 1500), 2


@pytest.mark.parametrize("chunk", [5, 64, 1 << 20])
def test_special_values_on_the_serving_loop(gpu, chunk):
    # In one part and in many: a run may end on one point in the middle of a part.
    from fpsample_amd.serve import Server

    clouds = list(special_clouds())
    print(f"special values, serving loop, {chunk} picks a launch", flush=True)
    with Server(hbm_budget_bytes=128 << 20, chunk_passes=chunk) as srv:
        ids = [srv.submit(pc, m, s) for pc, m, s in clouds]
        outs = [srv.wait(r)[0] for r in ids]
    for i, (g, (pc, m, s)) in enumerate(zip(outs, clouds)):
        np.testing.assert_array_equal(g, O.fps(pc, m, s), err_msg=f"request {i} n={len(pc)} m={m}")


def test_special_values_in_a_batch(gpu):
    # With enough small clouds beside them that the large ones get one workgroup each and keep
    # their min-distances in memory, and alone, as teams.
    from fpsample_amd.batch import DeviceBatch

    special = list(special_clouds())
    rng = np.random.default_rng(23)
    many = special + [(rng.random((9000, 3)).astype(np.float32), 900, 0) for _ in range(400)]
    for name, work in (("teams", special), ("one workgroup each", many)):
        print(f"special values, batch, {name}", flush=True)
        b = DeviceBatch([w[0] for w in work], [w[1] for w in work], [w[2] for w in work])
        assert b.info()["ppt"] == 4
        b.run()
        b.status()
        for i, (g, (pc, m, s)) in enumerate(zip(b.picks(), work)):
            np.testing.assert_array_equal(g, O.fps(pc, m, s), err_msg=f"{name} cloud {i} n={len(pc)}")
        b.close()
