"""GPU tests of the threshold rounds on clouds that hold points many times over: every pick, and
no more rounds than picks."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def clouds(d):
    rng = np.random.default_rng(50 + d)
    sites = rng.random((250, d))
    yield "sites", sites[rng.integers(0, 250, 20_000)], 250
    x = rng.random((20_000, d))
    x[10_000:] = 0.0
    yield "padded", x, 300
    yield "padded in between", rng.permutation(x), 1200
    yield "lattice", rng.integers(0, 4, (30_000, d)), 1500
    y = rng.random((20_000, d))
    y[::3] = np.nan
    y[1::3] = np.inf
    yield "no distance", y, 200


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("d", [1, 3, 6, 9, 40])
def test_every_round_takes_a_pick(gpu, monkeypatch, d, order):
    from fpsample_amd import device as D

    for shape in (f"{4 if d == 1 else 1}:40:100:{order}", f"4:5:100:{order}"):
        monkeypatch.setenv("FPSX_ROUNDS", shape)
        for name, pc, m in clouds(d):
            pc = np.ascontiguousarray(pc, np.float32)
            print(f"copies d={d} {name} m={m} shape={shape}", flush=True)
            assert D.call_info(len(pc), d, n_samples=m)["kind"] == "rounds"
            rows = D.DeviceArray.from_numpy(pc)
            start, out = D.DeviceArray.from_numpy(np.zeros(1, np.uint64)), D.DeviceArray((m,), np.uint64)
            D.fps_sampling_device_strided(rows, d, 1, len(pc), d, m, start, 1, out)
            D.device_status()
            np.testing.assert_array_equal(out.numpy(), O.fps(pc, m, 0), err_msg=name)
            v = ctypes.c_uint64()
            assert D.lib().fpsx_launch_exchanges(ctypes.c_void_p(0), ctypes.byref(v)) == 0
            assert v.value <= m, f"{name}: {v.value} rounds for {m} picks"
