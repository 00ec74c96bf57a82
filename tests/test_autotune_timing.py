"""The tuner times the build that programs run, and the shipped table holds no
tile cap that was ranked on a kernel which no longer runs there (no GPU)."""

import torch

from forte2_amd import autotune


def test_candidates_are_timed_without_phase_events(monkeypatch):
    import forte2_amd.jkbuilder as jkb
    import forte2_amd.workloads as wl

    seen = []

    class FB:
        timing, last_timings = False, {"total": 0.0}

        def __init__(self, **kw):
            pass

        def set_tuning(self, k, v):
            pass

        def build_JK(self, Cs, precision):
            seen.append(self.timing)

    class Event:
        def __init__(self, enable_timing=False):
            pass

        def record(self):
            pass

        def synchronize(self):
            pass

        def elapsed_time(self, other):
            return 1.0

    monkeypatch.setattr(jkb, "FockBuilder", FB)
    monkeypatch.setattr(wl, "synthetic_B", lambda *a, **k: None)
    monkeypatch.setattr(wl, "orthonormal_C", lambda *a, **k: None)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "empty_cache", lambda: None)
    table = autotune.tune([(24, 139, 5)], ("fp64",), device="cpu", log=None)
    assert table["fp64:24:139"]["ms"] == 1.0
    # F2JK_TIMING keeps J off the side stream
    assert len(seen) >= 2 * 28 and not any(seen)


def test_tile_rows_are_offered_where_the_library_chooses():
    rows = lambda n: {c.get("kx_rows") for c in autotune._candidates("bf16x3", grouped=False, nbf=n)}
    assert rows(144) == {None} and rows(192) == rows(384) == rows(960) == {128, 256}


def test_no_cap_of_the_128_row_kernel_from_nbf_192_on():
    for key, e in autotune.load().items():
        prec, nbf = key.split(":")[-3], int(key.split(":")[-2])
        if not key.startswith("group:") and prec == "bf16x3" and nbf >= 192 and e.get("kx_rows") != 128:
            assert e.get("bf16_nbw_max", 10) == 10, key
