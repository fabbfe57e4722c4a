"""GPU test of calls in threshold rounds where the GPU's memory is nearly full."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

# In a process of its own, whose library holds no buffers yet.  Besides the points there is room
# for min-distances (8 MB), as the pass kernels need it, but not for the records in spatial order.
FULL = """
import numpy as np, torch
from fpsample_amd import device as D
from fpsample_amd.batch import DeviceBatch
from oracle import oracle as O
n, m = 1 << 21, 600
rng = np.random.default_rng(3)
pc = rng.random((n, 4), dtype=np.float32)
flat = rng.random((n, 2), dtype=np.float32)
want, want2 = O.fps(pc, m, 0), O.fps(flat, m, 0)
D.fps_sampling_tensor(D.DeviceArray.from_numpy(pc[:600]), 300, 0)  # loads what there is to load
D.device_status()
rows, soa = D.DeviceArray.from_numpy(pc), D.DeviceArray.from_numpy(np.ascontiguousarray(pc.T))
start = D.DeviceArray.from_numpy(np.zeros(1, np.uint64))
out = D.DeviceArray((m,), np.uint64)
batch_room = D.DeviceArray((16 << 20,), np.uint8)
full = []
while len(full) < 8 and torch.cuda.mem_get_info()[0] > 40 << 20:
    full.append(D.DeviceArray((torch.cuda.mem_get_info()[0] - (32 << 20),), np.uint8))
print("free", torch.cuda.mem_get_info()[0] >> 20, "MiB", flush=True)
for form in ("rows", "columns"):
    sp, ld = (4, 1) if form == "rows" else (1, n)
    D.fps_sampling_device_strided(rows if form == "rows" else soa, sp, ld, n, 4, m, start, 1, out)
    D.device_status()
    assert np.array_equal(out.numpy(), want), form
print("calls ok", flush=True)
batch_room.free()
b = DeviceBatch([flat], [m], [0], graph=False)
b.run()
b.status()
assert np.array_equal(b.picks()[0], want2)
print("batch ok", flush=True)
for a in full:
    a.free()
D.fps_sampling_device_strided(rows, 4, 1, n, 4, m, start, 1, out)
D.device_status()
assert np.array_equal(out.numpy(), want)
print("ok")
"""


def test_calls_on_a_nearly_full_gpu(gpu):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", FULL], cwd=root, capture_output=True, text=True,
                         timeout=110, env=dict(os.environ, PYTHONPATH=root))
    print(out.stdout, flush=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout + out.stderr
