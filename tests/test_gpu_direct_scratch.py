"""The scratch of the direct sums: taking it leaves a graph alone that another host
thread is capturing."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_direct_sum_beside_another_threads_capture(gpu):
    from sbh_amd import ffi
    from sbh_amd._lib import buf, call, f32, i32, stream_handle

    rng = np.random.default_rng(5)
    p = torch.tensor(rng.uniform(0, 1, (5000, 3)).astype(np.float32), device=gpu)
    m = torch.full((5000,), 1.0 / 5000, device=gpu)
    want = ffi.softened_direct_force(p, m, p, cutoff_scale=float("inf"))
    out = torch.zeros_like(p)
    x = torch.ones(1000, device=gpu)
    other, result = torch.cuda.Stream(), []
    torch.cuda.synchronize()

    def work():
        torch.cuda.set_device(gpu)
        try:
            with torch.cuda.stream(other):
                handle = stream_handle()
            call("sbh_direct_force_soft", handle, buf(p), buf(m), buf(p), buf(out),
                 f32(1e-2), f32(float("inf")), i32(0), f32(1.0), i32(256))
            result.append(None)
        except Exception as e:  # reported by the test's own thread
            result.append(e)

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="global"):
        y = x * 2.0
        t = threading.Thread(target=work)
        t.start()
        t.join()
        z = y + 1.0
    torch.cuda.synchronize()
    assert result == [None]
    torch.testing.assert_close(out, want, rtol=1e-4, atol=2e-6 * float(want.abs().max()))
    for _ in range(2):
        g.replay()
        torch.cuda.synchronize()
        assert bool((z == 3.0).all())
