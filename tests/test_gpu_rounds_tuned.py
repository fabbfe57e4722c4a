"""GPU tests of the tuner with the threshold rounds among its plans."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_tuned_rounds_follow_the_calls_picks(gpu, monkeypatch):
    # Tuned for few picks; a call of many takes the candidates a round and the spatial order of
    # its own picks, and so as many rounds as before tuning.
    from fpsample_amd import device as D

    n, d, m = 90_001, 6, 4096
    rng = np.random.default_rng(14)
    pc = rng.random((n, d)).astype(np.float32)
    soa = D.DeviceArray.from_numpy(np.ascontiguousarray(pc.T))
    start = D.DeviceArray.from_numpy(np.array([3], np.uint64))
    want = O.fps(pc, m, 3)

    def call():
        out = D.DeviceArray((m,), np.uint64)
        D.fps_sampling_device(soa, n, d, m, start, 1, out)
        D.device_status()
        np.testing.assert_array_equal(out.numpy(), want)
        v = ctypes.c_uint64()
        assert D.lib().fpsx_launch_exchanges(ctypes.c_void_p(0), ctypes.byref(v)) == 0
        return v.value

    before = call()
    passes = D.plan_info(n, d, n_samples=m)
    tuned = D.autotune(soa, 1, n, n, d)
    info = D.call_info(n, d, n_samples=m)
    print(f"tuned {tuned}, a call runs {info}", flush=True)
    assert info["kind"] == "rounds" and info["grid"] == tuned["grid"]
    assert D.plan_info(n, d, n_samples=m) == info
    assert call() == before
    # Pass kernels asked for by name are what runs, and what is reported.
    for name in ("FPSX_NO_ROUNDS", "FPSX_NO_PAIR"):
        monkeypatch.setenv(name, "1")
        assert D.call_info(n, d, n_samples=m) == passes
        assert D.plan_info(n, d, n_samples=m) == passes
        monkeypatch.delenv(name)


def test_tuner_leaves_the_rounds_out_when_asked(gpu, monkeypatch):
    from fpsample_amd import device as D

    n, d = 30_011, 32
    soa = D.DeviceArray.from_numpy(np.random.default_rng(15).random((d, n)).astype(np.float32))
    monkeypatch.setenv("FPSX_NO_ROUNDS", "1")
    D.autotune(soa, 1, n, n, d, passes=64)
    monkeypatch.delenv("FPSX_NO_ROUNDS")
    assert D.call_info(n, d, n_samples=500)["kind"] != "rounds"  # the tuned plan serves


def test_batch_tuner_skips_rounds_that_gave_up(gpu):
    # Exchanges that may not wait at all: the rounds' teams give up at once, which is fast; clouds
    # that one workgroup holds need no exchange in the pass kernels.
    from fpsample_amd import device as D
    from fpsample_amd.batch import DeviceBatch

    rng = np.random.default_rng(16)
    clouds = [rng.random((16_000, 3)).astype(np.float32) for _ in range(2)]
    ms = [2000, 1500]
    D.exchange_timeout(1e-9)
    try:
        b = DeviceBatch(clouds, ms, [0, 0], autotune=True)
    finally:
        D.exchange_timeout(0)
    print(f"tuned batch: {b.info()}", flush=True)
    b.run()
    b.status()
    for i, (g, pc, m) in enumerate(zip(b.picks(), clouds, ms)):
        np.testing.assert_array_equal(g, O.fps(pc, m, 0), err_msg=f"cloud {i}")
    b.close()


@pytest.mark.parametrize("n,d,m,rounds", [
    (511, 3, 192, False), (512, 3, 191, False), (512, 3, 192, True), (512, 4, 63, False),
    (512, 4, 64, True), (513, 4, 111, False), (513, 8, 112, True), (8192, 6, 111, False),
    (8192, 6, 112, True), (8193, 6, 64, True), (600, 9, 63, False), (600, 9, 64, True)])
def test_which_calls_run_in_rounds(gpu, n, d, m, rounds):
    # Both sides of each line of the rule: what runs, and its picks.
    import fpsample_amd as F
    from fpsample_amd import device as D

    assert (D.call_info(n, d, n_samples=m)["kind"] == "rounds") is rounds
    pc = np.random.default_rng(n + d).random((n, d)).astype(np.float32)
    np.testing.assert_array_equal(F.fps_sampling(pc, m, start_idx=5), O.fps(pc, m, 5))
