"""GPU tests of the threshold rounds on clouds that one round can hold whole: the first pick at
distance 0 is the best of all such points, those that the same picks brought there included."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def small_clouds(d=3):
    """Clouds of duplicates and wide scales, with the picks to take of each."""
    rng = np.random.default_rng(90 + d)
    ladder = np.zeros((80, d), np.float32)
    ladder[40:, 0] = 2.0 ** -np.arange(40)
    three = np.zeros((3, d), np.float32)
    three[2, 0] = 1e-20
    out = [(ladder, 60), (three, 3)]
    for _ in range(60):
        n = int(rng.integers(2, 500))
        pc = rng.uniform(-1, 1, (n, d)) * 10.0 ** rng.uniform(-12, 0, (n, 1))
        copies = rng.integers(0, n, int(rng.integers(1, 30)))
        pc[copies] = pc[rng.integers(0, n, copies.size)]
        out.append((pc.astype(np.float32), n))
    return out


def check(got, pc, m, start, name):
    np.testing.assert_array_equal(got, O.fps(pc, m, start), err_msg=f"{name} n={len(pc)} m={m}")


@pytest.mark.parametrize("d", [1, 2, 3, 4])
def test_small_clouds_in_a_batch(gpu, d):
    import fpsample_amd as F

    clouds = small_clouds(d)
    print(f"batch d={d}", flush=True)
    got = F.fps_sampling_batch([c for c, _ in clouds], [m for _, m in clouds], 0)
    for i, (g, (pc, m)) in enumerate(zip(got, clouds)):
        check(g, pc, m, 0, f"cloud {i}")


@pytest.mark.parametrize("chunk", [5, 256])
def test_small_clouds_on_the_serving_loop(gpu, chunk):
    from fpsample_amd.serve import Server

    clouds = small_clouds()
    print(f"serve chunk={chunk}", flush=True)
    with Server(hbm_budget_bytes=64 << 20, chunk_passes=chunk) as srv:
        ids = [srv.submit(pc, m, 0) for pc, m in clouds]
        outs = [srv.wait(r)[0] for r in ids]
    for i, (g, (pc, m)) in enumerate(zip(outs, clouds)):
        check(g, pc, m, 0, f"request {i}")


@pytest.mark.parametrize("shape", ["1:1", "1:4"])
@pytest.mark.parametrize("d", [3, 6, 9, 40])
def test_small_clouds_one_call_each(gpu, monkeypatch, shape, d):
    import fpsample_amd as F
    from fpsample_amd import device as D

    monkeypatch.setenv("FPSX_ROUNDS", shape)
    print(f"calls d={d} shape={shape}", flush=True)
    for i, (pc, m) in enumerate(small_clouds(d)):
        assert D.call_info(len(pc), d, n_samples=m)["kind"] == "rounds"
        check(F.fps_sampling(pc, m, start_idx=0), pc, m, 0, f"cloud {i}")
