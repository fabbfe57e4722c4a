"""The pass kernels in the plans and forms that calls took before the threshold rounds: single
clouds by the planner's own choice, the KD-line entry, batches, and the serving loop's paired
kernel.  FPSX_NO_ROUNDS=1 keeps them; without it the tests used here run the rounds."""
import numpy as np
import pytest

import bench
from oracle import oracle as O
from tests import test_gpu_fullsize as full
from tests import test_gpu_pair as pair
from tests import test_gpu_parity as parity
from tests import test_gpu_serve as serve

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_rounds(gpu, monkeypatch):
    from fpsample_amd import device as D

    monkeypatch.setenv("FPSX_NO_ROUNDS", "1")
    for n, d, m in ((4096, 3, 1024), (50_000, 3, 4096), (1 << 21, 3, 16_384), (9000, 6, 900)):
        assert D.call_info(n, d, n_samples=m) == D.plan_info(n, d, n_samples=m)


@pytest.fixture
def plan_env(monkeypatch):
    def set_plan(p):
        if p is None:
            monkeypatch.delenv("FPSX_PLAN", raising=False)
        else:
            monkeypatch.setenv("FPSX_PLAN", p)
    return set_plan


def test_small_clouds(gpu):
    parity.test_small_clouds_auto_plans(gpu)


def test_paired_plan_and_bucket_order(gpu):
    parity.test_pruned_auto_plan_and_bucket_order(gpu)


@pytest.mark.parametrize("d", [1, 2, 5, 8, 9, 40])
def test_dimensions(gpu, d):
    parity.test_dimensions_auto_plan(gpu, d)


def test_streaming_lattice(gpu, plan_env):
    parity.test_lattice_streaming_kernels_agree(gpu, plan_env)


@pytest.mark.parametrize("n", [(1 << 20) + 1, 64 * 17_408])
def test_paired_with_a_row_in_lds(gpu, plan_env, n):
    pair.test_pair_lds_row_planner_sizes(gpu, plan_env, n)


@pytest.mark.parametrize("n,name", [(1 << 20, "gauss1m"), ((1 << 20) + 1, "gauss1m1"),
                                    (1 << 21, "gauss2m")])
def test_clustered_every_pick(gpu, monkeypatch, n, name):
    full.check_single(gpu, monkeypatch, name, bench.gen_gauss_mixture(n), {})


@pytest.mark.parametrize("n", [50_000, 100_000])
def test_uniform_every_pick(gpu, monkeypatch, n):
    full.check_single(gpu, monkeypatch, f"uniform{n // 1000}k", bench.gen_uniform_n(n), {})


@pytest.mark.parametrize("n,name,h", [(4096, "kdline4k", 5), (50_000, "kdline50k", 7)])
def test_bucket_entry_every_pick(gpu, monkeypatch, n, name, h):
    full.test_reference_kdline_bench_cases_every_pick(gpu, monkeypatch, n, name, h)


def test_serving_in_short_chunks(gpu, monkeypatch):
    # The one-slot paired kernel; chunks of 5 passes end on both sides of its pairs.
    serve.test_serve_default_shape_short_chunks(gpu, monkeypatch, False)


def test_serving_whole_requests(gpu):
    serve.test_serve_pruned_whole_requests_against_oracle(gpu)


def test_serving_from_threads(gpu):
    serve.test_serve_mixed_from_threads(gpu)


def test_batch(gpu):
    from fpsample_amd.batch import DeviceBatch

    rng = np.random.default_rng(30)
    clouds = [rng.random((n, 3)).astype(np.float32) for n in (20_000, 300, 70_000, 5000)]
    ms = [2000, 300, 1500, 1250]
    b = DeviceBatch(clouds, ms, [0] * 4)
    assert b.info()["ppt"] == 8
    b.run()
    b.status()
    for g, pc, m in zip(b.picks(), clouds, ms):
        np.testing.assert_array_equal(g, O.fps(pc, m, 0))
    b.close()
