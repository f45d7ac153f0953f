"""The launch-shape autotuner's choice and cache, with given times in place of
the device: the plan's own shapes are among what is compared, every stage-1
shape the plan may pick is, and another build's results are not reused."""
import json

import numpy as np
import pytest

from transientx_amd import _lib, autotune

ROW = (0.0, 1.0, 100, 8)


@pytest.fixture
def tune(monkeypatch, tmp_path):
    """tune(times) runs tune_row with times[stage](shapes) as the stage's ms."""
    class Lib:
        @staticmethod
        def tx_stage2_shapes(out, n):
            return 6

    monkeypatch.setenv("TX_AUTOTUNE_CACHE", str(tmp_path / "autotune.json"))
    monkeypatch.setattr(autotune, "_device_id", lambda: "gfx950/256CU")
    monkeypatch.setattr(autotune, "_library_id", lambda: "a")
    monkeypatch.setattr(autotune, "_blocks", lambda nchans, ndump, dtype: [None, None])
    monkeypatch.setattr(_lib, "lib", lambda: Lib)
    asked = []

    def run(times, **kw):
        def time_stage(nchans, freqs, tsamp, ndump, row, vwn, overlap, shapes, data, stage, nblocks, dtype="u8"):
            asked.append((stage, dict(shapes)))
            return times(stage, shapes)

        monkeypatch.setattr(autotune, "_time_stage", time_stage)
        asked.clear()
        return autotune.tune_row(64, np.linspace(1500, 1200, 64), 1e-3, 512, ROW, [1, 2], **kw), list(asked)

    return run


def test_plans_choice_is_kept_unless_beaten(tune):
    shapes, asked = tune(lambda stage, s: 1.0 if not s else 1.2, use_cache=False)
    assert shapes == {}
    assert ("stage1", {}) in asked and ("stage2", {}) in asked
    # within the noise of a timing: kept
    assert tune(lambda stage, s: 1.0 if not s else 0.995, use_cache=False)[0] == {}
    # one stage beaten
    fast = {"s1_ncc": 2, "s1_q": 1}
    assert tune(lambda stage, s: 0.8 if s == fast else 1.0, use_cache=False)[0] == fast
    # the fastest of several that beat it, and shapes that do not fit
    t = {2: 0.9, 3: 0.7, 4: 0.8}
    shapes, _ = tune(lambda stage, s: None if s.get("s2_lds") == 163840 else t.get(s.get("s2_shape"), 1.0),
                     use_cache=False)
    assert shapes == {"s2_shape": 3, "s2_lds": 81920}


@pytest.mark.parametrize("dtype,widest", [("u8", 16), ("f32", 8)])
def test_every_stage1_shape_is_tried(tune, dtype, widest):
    _, asked = tune(lambda stage, s: 1.0, use_cache=False, dtype=dtype)
    tried = {(s["s1_ncc"], s["s1_q"]) for stage, s in asked if stage == "stage1" and s}
    ncc = [n for n in (1, 2, 4, 8, 16) if n <= widest]
    assert tried == {(n, q) for n in ncc for q in (1, 2)}


def test_cache_of_another_build_is_not_used(tune, monkeypatch, tmp_path):
    fast = {"s1_ncc": 8, "s1_q": 2}
    shapes, asked = tune(lambda stage, s: 0.5 if s == fast else 1.0)
    assert shapes == fast and asked
    shapes, asked = tune(lambda stage, s: 1.0)  # from the cache
    assert shapes == fast and not asked
    monkeypatch.setattr(autotune, "_library_id", lambda: "b")
    shapes, asked = tune(lambda stage, s: 1.0)
    assert shapes == {} and asked
    assert len(json.loads((tmp_path / "autotune.json").read_text())) == 2


def test_library_id_follows_the_file(monkeypatch, tmp_path):
    f = tmp_path / "lib.so"
    monkeypatch.setattr(_lib, "LIBPATH", f)
    f.write_bytes(b"one")
    a = autotune._library_id()
    f.write_bytes(b"two")
    assert autotune._library_id() != a
