"""The tuner's decisions, with the library and the timings replaced."""
import pytest


class Lib:
    def __init__(self):
        self.conv = {}
        self.caps = {}
        self.calls = []

    def csipm_tune_bluestein(self, L, m):
        if m:
            self.conv[L] = m
        else:
            self.conv.pop(L, None)
        return 0

    def csipm_tune_set(self, kind, elem, w, r, cap, nt):
        self.calls.append((kind, cap, nt))
        self.caps[kind] = None if cap < 0 else cap
        return 0


# ms of the library's own plan, of the smallest convolution length and of the others
@pytest.mark.parametrize("own,smallest,other,chosen", [
    (1.0, 2.0, 1.5, False),     # the dense form beats every length
    (1.0, 2.0, 0.99, False),    # one beats it by 1%: within the threshold
    (1.0, 2.0, 0.8, True),
    (1.0, 0.7, 0.9, True),
])
def test_bluestein_lengths_compete_with_the_plan_in_use(monkeypatch, own, smallest, other, chosen):
    from csipm import tune
    lib = Lib()
    L = 111
    m0, cands = tune.bluestein_candidates(L)
    assert m0 == 221 and len(set(cands)) > 1

    def best(dims, count, reps, lib):
        m = lib.conv.get(L, 0)
        ms = own if m == 0 else smallest if m == m0 else other
        return {1: (ms / 2, None, ms / 2), 0: (ms / 2, None, ms / 2)}, {1: (m, m, 1), 0: (m, m, 1)}

    monkeypatch.setattr(tune, "_shape_best", best)
    entry, launch = tune.tune_bluestein((L, L, L), 1, 1, lib, lambda m: None)
    assert (entry is not None) == chosen and not launch
    if chosen:
        assert (entry["conv_len"] == m0) == (smallest < other)
        assert entry["ms_builtin"] == own
    assert lib.conv == {}


class Op:
    handle = None


@pytest.mark.parametrize("ms,cap", [
    ({None: [1.0, 1.0], 3: [0.8, 0.8], 2: [0.9], 1: [1.2]}, 3),
    ({None: [1.0, 0.8], 3: [0.8, 0.8], 2: [0.9], 1: [1.2]}, None),   # won once, by chance
    ({None: [1.0], 3: [1.1], 2: [1.0], 1: [1.2]}, None),
])
def test_one_timing_per_launch_shape(monkeypatch, ms, cap):
    from csipm import tune
    lib = Lib()
    left = {k: list(v) for k, v in ms.items()}
    monkeypatch.setattr(tune, "_batch", lambda dims, count: ([], [Op()]))
    monkeypatch.setattr(tune, "fft_shape", lambda op, axis: (64, 64, 0))
    monkeypatch.setattr(tune, "_time", lambda *a: left[lib.caps.get(1)].pop(0))
    out = tune.tune_shape((64,), 1, 1, lib, lambda m: None)
    assert [e["lg_cap"] for e in out] == ([] if cap is None else [cap])
    # the workgroup size is the library's: no two candidates differ in it alone
    first = [c for c in lib.calls if c[1] >= 0][:3]
    assert sorted(c[1] for c in first) == [1, 2, 3] and {c[2] for c in lib.calls} == {0}
    assert lib.caps[1] is None


def test_tables_with_and_without_thread_counts_load(tmp_path):
    import json

    from csipm import tune
    lib = Lib()
    path = tmp_path / "t.json"
    e = {"kind": 0, "elem_bytes": 8, "fft_len": 64, "rows": 64, "lg_cap": 2}
    path.write_text(json.dumps({"entries": [e, dict(e, fft_len=80, rows=80, nt=128)]}))
    assert tune.load(lib, str(path)) == 2
    assert [c[2] for c in lib.calls] == [0, 128]


def test_plan_order_is_the_library_s():
    from csipm import tune
    assert tune.radix_stages(2 * 3 * 5 * 31 * 16) == [31, 15, 16, 2]
    assert tune.radix_stages(391) == [23, 17] and tune.radix_stages(37) is None
