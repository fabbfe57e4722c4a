"""GPU tests of captured calls in threshold rounds whose scratch is of the cloud's size."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def exchanges(D):
    import ctypes

    v = ctypes.c_uint64()
    assert D.lib().fpsx_launch_exchanges(ctypes.c_void_p(0), ctypes.byref(v)) == 0
    return v.value


# The planner's own shape, in spatial order; several blocks a wave, so that min-distances go to
# memory, in order and not; rows of any dimension, turned into columns first.
CASES = [(20_001, 3, 2048, None), (20_001, 3, 1500, "1:4:100:1"), (20_001, 3, 1500, "1:4:100:0"),
         (3001, 20, 200, None)]


@pytest.mark.parametrize("n,d,m,shape", CASES)
def test_replay_after_a_larger_call(gpu, monkeypatch, n, d, m, shape):
    # The buffers that the graph refers to stay where they are when a larger call needs more.
    import torch

    from fpsample_amd import device as D

    if shape:
        monkeypatch.setenv("FPSX_ROUNDS", shape)
    rng = np.random.default_rng(n + d)
    side = torch.cuda.Stream()
    start = torch.zeros(1, dtype=torch.int64, device="cuda")

    def call(pts, picks, out, stream):
        D.fps_sampling_device_strided(pts.data_ptr(), d, 1, pts.shape[0], d, picks,
                                      start.data_ptr(), 1, out.data_ptr(), stream=stream)

    pts = torch.from_numpy(rng.random((n, d), dtype=np.float32)).cuda()
    out = torch.zeros(m, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    print(f"capture n={n} d={d} m={m} shape={shape}", flush=True)
    call(pts, m, out, side.cuda_stream)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(pts, m, out, torch.cuda.current_stream().cuda_stream)
    for rep in range(3):
        # A larger call each time, and other work on what memory there is.
        more = (rep + 2) * n
        big = rng.random((more, d), dtype=np.float32)
        big_out = torch.zeros(m, dtype=torch.int64, device="cuda")
        big_pts = torch.from_numpy(big).cuda()
        torch.cuda.synchronize()
        call(big_pts, m, big_out, side.cuda_stream)
        side.synchronize()
        np.testing.assert_array_equal(big_out.cpu().numpy().astype(np.uint64), O.fps(big, m, 0),
                                      err_msg=f"larger call {rep}")
        torch.full((1 << 22,), float("nan"), device="cuda")
        pc = rng.random((n, d), dtype=np.float32)
        pts.copy_(torch.from_numpy(pc))
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy().astype(np.uint64), O.fps(pc, m, 0),
                                      err_msg=f"replay {rep}")
        assert 0 < exchanges(D) < m // 4  # rounds, not a pick or two an exchange


FRESH = """
import sys
import numpy as np, torch
from fpsample_amd import device as D
from oracle import oracle as O
n, d, m1, m2 = [int(v) for v in sys.argv[1:5]]
rng = np.random.default_rng(8)
pc = rng.random((n, d), dtype=np.float32)
pts = torch.from_numpy(pc).cuda()
start = torch.zeros(1, dtype=torch.int64, device="cuda")
side = torch.cuda.Stream()
def call(m, out, stream):
    D.fps_sampling_device_strided(pts.data_ptr(), d, 1, n, d, m, start.data_ptr(), 1,
                                  out.data_ptr(), stream=stream)
first = torch.zeros(m1, dtype=torch.int64, device="cuda")
out = torch.zeros(m2, dtype=torch.int64, device="cuda")
torch.cuda.synchronize()
call(m1, first, side.cuda_stream)
side.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph, stream=side):
    call(m2, out, torch.cuda.current_stream().cuda_stream)
want = O.fps(pc, m2, 0)
for rep in range(3):
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().astype(np.uint64), want), rep
print("ok")
"""


# The earlier call took so few picks that it made no spatial order, where the captured one would
# make one; or the captured call takes so few that alone it would run a pass kernel, whose scratch
# the earlier one, in rounds, did not need.
@pytest.mark.parametrize("n,d,first,captured", [(20_001, 3, 1100, 2048), (3001, 20, 200, 50),
                                                (4_500_000, 3, 200, 100)])
def test_capture_after_a_call_of_other_picks(gpu, n, d, first, captured):
    # In a process of its own, whose library has made no call before.
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", FRESH, str(n), str(d), str(first), str(captured)],
                         cwd=root, capture_output=True, text=True, timeout=100,
                         env=dict(os.environ, PYTHONPATH=root))
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout + out.stderr
