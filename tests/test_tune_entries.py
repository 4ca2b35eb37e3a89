"""The autotuner against the tables it keeps: its recorded results leave every
entry where it is (entries they did not measure included), and each entry of
the single-value tables is one of its candidates, so a new run can weigh it."""
import importlib.util
import json
import os
import re
import shutil

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gilaelectromagnetics.jl_amd")


@pytest.fixture()
def tune(tmp_path):
    spec = importlib.util.spec_from_file_location("gla_tune_entries", os.path.join(PKG, "tune.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    shutil.copy(os.path.join(PKG, "csrc", "gla_tune.hpp"), tmp_path / "gla_tune.hpp")
    mod.CSRC = str(tmp_path)
    return mod


def test_recorded_results_keep_the_tables(tune, tmp_path):
    before = (tmp_path / "gla_tune.hpp").read_text()
    tune.table(os.path.join(PKG, "tune", "shapes_mi355x.jsonl"), 0.05)
    assert (tmp_path / "gla_tune.hpp").read_text() == before


def test_entries_are_candidates(tune, tmp_path):
    src = (tmp_path / "gla_tune.hpp").read_text()
    for part, tag in (("gg", "GG"), ("xk", "XK"), ("yk", "YK"), ("rl", "RELOAD"), ("plan", "PLAN")):
        for dt in ("c64", "c128"):
            have = {d[dt] for _, _, d in tune.candidates() if d["part"] == part}
            body = re.search(rf"// BEGIN TUNED {tag} {dt.upper()}\n(.*?)// END TUNED", src, flags=re.S).group(1)
            assert {int(v) for v in re.findall(r"return (\d+);", body)} <= have, (part, dt)


def test_a_measured_entry_can_lose(tune, tmp_path):
    path = tmp_path / "res.jsonl"
    path.write_text("\n".join(json.dumps({"part": "gg", "dtype": "c128", "n": 64, "choice": c,
                                          "large_us": [0, 0, t, 0, 0]}) for c, t in ((3, 80.0), (7, 90.0), (15, 100.0))))
    tune.table(str(path), 0.05)
    body = re.search(r"// BEGIN TUNED GG C128\n(.*?)// END TUNED", (tmp_path / "gla_tune.hpp").read_text(), flags=re.S)
    assert "case 64:" not in body.group(1) and "case 128: return 15;" in body.group(1)


def test_wave_lengths_are_timed_with_and_without(tune, tmp_path, capsys):
    # at the wave form's lengths pass 3's shapes time k_zpass, so that they
    # differ, and the wave form itself is compared and reported
    assert all("-DGLA_WT_F=0" in flags for _, flags, d in tune.candidates() if d["part"] == "zpass")
    assert {flags for _, flags, d in tune.candidates() if d["part"] == "wave"} == {"-DGLA_WT_F=0", ""}
    before = (tmp_path / "gla_tune.hpp").read_text()
    assert "GLA_WT_F == 0" in before
    path = tmp_path / "res.jsonl"
    path.write_text("\n".join(json.dumps({"part": "wave", "dtype": "c64", "n": n, "choice": c,
                                          "large_us": [0, 0, t, 0, 0], "small_us": [0, 0, t / 4, 0, 0]})
                              for n in (96, 128) for c, t in ((0, 60.0), (1, 50.0))))
    tune.table(str(path), 0.05)
    out = capsys.readouterr().out
    assert "c64 wave 96 large: wave form 50.0 us, without 60.0 us" in out and "wave 128" not in out
    assert (tmp_path / "gla_tune.hpp").read_text() == before


def test_rows_of_plane_lengths_by_the_apply(tune, tmp_path):
    # 16: the plane kernels' apply decides, whatever the five separate passes
    # say; 80: the passes decide; entries that were set are candidates
    recs = []
    for (ex, ey, pxy), t in (((4, 4, 16), 30.0), ((8, 8, 16), 20.0), ((8, 4, 16), 25.0)):
        recs.append({"part": "rows", "dtype": "c64", "n": 16, "choice": [ex, ey, pxy], "apply_us": t,
                     "rows_us": [40 - t, 40 - t, 0, 0, 0]})
        recs.append({"part": "rows", "dtype": "c64", "n": 80, "choice": [ex, ey, pxy],
                     "rows_us": [40 - t, 40 - t, 0, 0, 0]})
    path = tmp_path / "res.jsonl"
    path.write_text("\n".join(map(json.dumps, recs)))
    tune.table(str(path), 0.05)
    src = (tmp_path / "gla_tune.hpp").read_text()
    body = re.search(r"// BEGIN TUNED ROWS C64\n(.*?)// END TUNED", src, flags=re.S).group(1)
    assert "case 16: return RShape{8, 8, 16};" in body and "case 80:" not in body
    for k, dt in enumerate(("C64", "C128")):
        body = re.search(rf"// BEGIN TUNED ROWS {dt}\n(.*?)// END TUNED", src, flags=re.S).group(1)
        small = [tuple(map(int, v)) for v in re.findall(r"case (\d+): return RShape\{(\d+), (\d+), (\d+)\}", body)]
        assert {v[1:] for v in small if v[0] <= 64} <= {c[k] for c in tune.RCAND}
