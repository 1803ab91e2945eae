"""What the autotuner's cache is keyed by, and its candidates (no device)."""
import types

import pytest


def _problem(N, dense):
    return types.SimpleNamespace(nspins=N, maxnb=N - 1 if dense else 4, zmax=7, ncolors=N if dense else 2,
                                 pm_j=not dense, pm_j_fields=False, exact_rows=True)


def test_cached_tiles_belong_to_the_build_they_were_timed_on(monkeypatch, tmp_path):
    from piqmc import _lib, autotune
    monkeypatch.setattr(autotune, "_arch", lambda: "gfx950")
    pb = _problem(64, True)
    batch = types.SimpleNamespace(jobs=[{"problem": pb, "P": 16, "R": 2, "sched": [0.0, 1.0]}])
    keys = []
    for k in range(2):
        lib = tmp_path / ("lib%d.so" % k)
        lib.write_bytes(b"build %d" % k)
        monkeypatch.setattr(_lib, "LIB_PATH", str(lib))
        keys.append((autotune.key(pb, 16, 2), autotune.batch_key(batch)))
        assert keys[-1] == (autotune.key(pb, 16, 2), autotune.batch_key(batch))
    assert keys[0][0] != keys[1][0] and keys[0][1] != keys[1][1]


@pytest.mark.parametrize("N,fields", [(64, 1), (256, 1), (257, 2)])
def test_dense_candidates_differ(N, fields):
    from piqmc import autotune
    c = autotune.candidates(_problem(N, True), 16, 8)
    assert len(set(c)) == len(c)
    assert sum(v == "fields" for _, v in c) == fields
