"""Batches of one, two and four dimensions read the caller's points on every run, at its place in
the stream, and not before."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [20_001, 700, 1, 8193, 64, 3000, 8192]


@pytest.mark.parametrize("graph", [False, True], ids=["launches", "graph"])
@pytest.mark.parametrize("d", [1, 2, 4])
def test_points_changed_between_runs(gpu, d, graph):
    import torch

    from fpsample_amd import batch as Bt

    rng = np.random.default_rng(70 + d)
    ms = [max(1, n // 8) for n in SIZES]
    starts = [n // 3 for n in SIZES]
    offsets = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.uint64)
    total = int(offsets[-1])
    u64p = ctypes.POINTER(ctypes.c_uint64)
    ms_, starts_ = np.array(ms, np.uint64), np.array(starts, np.uint64)
    stream = torch.cuda.Stream()
    # Values no order can be made of until the first run.
    pts = torch.full((d, total), float("nan"), device="cuda")
    out = torch.zeros(sum(ms), dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    handle = ctypes.c_void_p()
    L = Bt._lib()
    rc = L.fpsx_batch_create(pts.data_ptr(), total, d, offsets.ctypes.data_as(u64p), len(SIZES),
                             ms_.ctypes.data_as(u64p), starts_.ctypes.data_as(u64p),
                             out.data_ptr(), Bt.GRAPH if graph else 0, ctypes.byref(handle))
    assert rc == 0, L.fpsx_last_error()
    try:
        for rep in range(3):
            print(f"d={d} graph={graph} run {rep}", flush=True)
            soa = (rng.integers(0, 30, (d, total)) if rep == 1 else rng.random((d, total)))
            soa = np.ascontiguousarray(soa, np.float32)
            host = torch.from_numpy(soa).pin_memory()
            with torch.cuda.stream(stream):
                pts.copy_(host, non_blocking=True)
            assert L.fpsx_batch_run(handle, stream.cuda_stream) == 0
            assert L.fpsx_batch_status(handle, stream.cuda_stream) == 0
            got = np.split(out.cpu().numpy().astype(np.uint64), np.cumsum(ms)[:-1])
            for i, (lo, n) in enumerate(zip(offsets[:-1].astype(int), SIZES)):
                want = O.fps(np.ascontiguousarray(soa[:, lo:lo + n].T), ms[i], starts[i])
                np.testing.assert_array_equal(got[i], want, err_msg=f"run {rep} cloud {i} n={n}")
    finally:
        L.fpsx_batch_destroy(handle)
