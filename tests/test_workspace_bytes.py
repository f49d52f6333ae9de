"""A workspace made for some size also serves every smaller one: the sizes that
the library asks for never fall as the number of points or queries grows."""
import ctypes

import numpy as np
import pytest
import torch


def _bytes(name):
    from sbh_amd import _lib as L

    fn = getattr(L.load_library(), name)
    fn.restype = ctypes.c_int64
    return lambda *a: fn(*(ctypes.c_int64(x) for x in a[:-2]), *map(ctypes.c_int32, a[-2:]))


def _sets(name, sets):
    from sbh_amd import _lib as L

    fn = getattr(L.load_library(), name)
    fn.restype = ctypes.c_int64
    return lambda n: fn(ctypes.c_int64(n), ctypes.c_int32(sets), ctypes.c_int32(10),
                        ctypes.c_int32(32))


# across the sizes where the sort's tiles change, and odd sizes over the range
SIZES = sorted({n + d for n in (1024, 4096, 1 << 15, 1 << 16, 1 << 17, 1 << 18, 1 << 20)
                for d in (*range(-3, 4), 132, 1024, 2049, 4095)} |
               {int(x) for x in np.geomspace(1, 5e6, 300)})


@pytest.mark.parametrize("fn", [
    lambda: (lambda n: _bytes("sbh_gravity_workspace_bytes")(n, 10, 32)),
    lambda: _sets("sbh_gravity_batch_workspace_bytes", 1),
    lambda: _sets("sbh_gravity_batch_workspace_bytes", 300),
    lambda: (lambda n: _bytes("sbh_winding_number_workspace_bytes")(n, 1000, 10, 16)),
    lambda: (lambda n: _bytes("sbh_winding_number_workspace_bytes")(1000, n, 10, 16)),
    lambda: (lambda n: _bytes("sbh_stochastic_workspace_bytes")(n, 1000, 10, 32)),
    lambda: (lambda n: _bytes("sbh_stochastic_workspace_bytes")(1000, n, 10, 32)),
], ids=["gravity", "one set", "300 sets", "elements", "wn queries", "sources",
        "stochastic queries"])
def test_workspace_bytes_never_fall(fn):
    need = fn()
    got = [need(n) for n in SIZES]
    assert got[0] > 0
    falls = [(a, b) for a, b, x, y in zip(SIZES, SIZES[1:], got, got[1:]) if y < x]
    assert not falls


@pytest.mark.gpu
@pytest.mark.parametrize("made,used", [(131400, 131072), (32900, 32768)])
def test_workspace_serves_a_smaller_call(gpu, made, used):
    from sbh_amd import gravity as G

    rng = np.random.default_rng(used)
    p = torch.tensor(rng.uniform(size=(used, 3)).astype(np.float32), device=gpu)
    m = torch.full((used,), 1.0 / used, device=gpu)
    ws = G.new_workspace(made, 10, 32)
    f = G.gravity_force(p, m, workspace=ws)
    assert torch.equal(f, G.gravity_force(p, m))
