"""The autotuner's candidates and cache keys, with the timings faked (no device):
by default only what the walks of the batch react to is timed, and a result tuned
with one build of the library is not taken for another's."""
import pytest
import torch


@pytest.fixture()
def tuner(monkeypatch):
    from sbh_amd import autotune as A

    class Gate:
        sets, rows = [], None

        def __init__(self, *a, **k):
            pass

        def errors(self, *a):
            return {"force": 0.0}

    timed = []

    def build_step(P, M, C, offsets, leaf, blocks, kw, threads=0):
        timed.append((kw["fwd_multipole_order"], kw["multipole_order"], leaf, blocks, threads))
        return (lambda: None), (None, None, None), None

    monkeypatch.setattr(A, "_Gate", Gate)
    monkeypatch.setattr(A, "build_step", build_step)
    monkeypatch.setattr(A, "time_graph", lambda step, reps=3: 1.0 + len(timed))
    monkeypatch.setattr(A, "_CACHE", {})
    monkeypatch.setattr(A, "_set_boxes", lambda p, o: torch.zeros(o.shape[0] - 1, 6))
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda d: "card")
    return A, timed


def _tune(A, sizes, **kw):
    offs = torch.tensor([0] + sizes, dtype=torch.int32).cumsum(0).to(torch.int32)
    x = torch.zeros(1, 3)
    return A.tune_batch(x, x[:, 0], x, offs, softening_scale=0.01, **kw)


# the first set for single waves, the last total for teams alone, and a set of that
# size whose walks have no monopole terms
@pytest.mark.parametrize("sizes,orders,single", [
    ([699999, 5, 0], {}, False), ([700000, 5], {}, True), ([500000] * 5 + [499999], {}, False),
    ([500000] * 6, {}, True), ([1000000], dict(fwd_orders=(2,), vjp_orders=(2, 3)), False)])
def test_defaults_time_what_the_walks_react_to(tuner, sizes, orders, single):
    A, timed = tuner
    res = _tune(A, sizes, **orders)
    blocks, threads = {t[3] for t in timed}, {t[4] for t in timed}
    assert len(timed) == len(set(timed)) == len(res["table"])
    if single:
        assert blocks == set(A.DEFAULT_BLOCKS) and threads == set(A.DEFAULT_THREADS)
    else:
        assert blocks == set(A.TEAM_BLOCKS) and threads == {256}
        # a grid of 256 caps the teams' own of 512 and 1024 blocks, of 1024 does not
        assert all(b < 512 for b in blocks)
    first = 10
    assert len(timed) == first + (0 if orders else 1) + (2 + 3 if single else 1)


def test_lines_are_the_library_s():
    import os
    import re

    from sbh_amd import autotune as A

    src = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       "barnes-hut_amd", "csrc")
    text = open(os.path.join(src, "tree.hpp")).read() + open(os.path.join(src, "tree.hip")).read()
    line = lambda name: int(re.search(r"constexpr \w+ " + name + r" = (\d+);", text).group(1))
    assert line("kSinglePoints") == A.SINGLE_WAVE_SET
    assert line("kAlonePoints") == A.SINGLE_WAVE_POINTS


def test_given_candidates_are_all_timed(tuner):
    A, timed = tuner
    _tune(A, [1000, 20], leaf_sizes=(16,), walk_blocks=(0, 4096), walk_threads=(256, 64))
    assert {t[3:] for t in timed} == {(0, 256), (4096, 256), (0, 64)}


def test_results_belong_to_a_build_of_the_library(tuner, monkeypatch, tmp_path):
    A, timed = tuner
    lib = tmp_path / "lib.so"
    lib.write_bytes(b"one")
    monkeypatch.setattr(A, "library_path", lambda: str(lib))
    cache = str(tmp_path / "tuned.json")
    _tune(A, [1000, 20], cache_file=cache)
    n = len(timed)
    A._CACHE.clear()
    _tune(A, [1000, 20], cache_file=cache)
    assert len(timed) == n  # from the file
    A._CACHE.clear()
    other = tmp_path / "other.so"
    other.write_bytes(b"two")
    monkeypatch.setattr(A, "library_path", lambda: str(other))
    _tune(A, [1000, 20], cache_file=cache)
    assert len(timed) == 2 * n
