"""The profile summary on small synthetic traces with the kernels that a step
launches: families, steps told apart by their k_publish, merged and separate
launches, one-off kernels left out."""
import csv
import json
import subprocess
import sys

import pytest

from lpa_amd.rocprof_summary import _headline, family

NAMES = {
    "bins": "void lpa::k_bins<1>(lpa::StepArgs, lpa::BinTable)",
    "lane": "void lpa::k_lane<8, false>(lpa::StepArgs)",
    "wave": "void lpa::k_group<8, false, 1, 8>(lpa::StepArgs, unsigned int, unsigned int)",
    "block": "void lpa::k_group<256, false, 1, 8>(lpa::StepArgs, unsigned int, unsigned int)",
    "decode1": "void lpa::k_heavy_decode<1>(lpa::HeavyArgs, lpa::DecodeTask const*, unsigned int, unsigned long const*, unsigned int*)",
    "chunks2": "void lpa::k_heavy_chunks<2, 1>(lpa::HeavyArgs)",
    "local0": "void lpa::k_heavy_local<0, 1, 4, false>(lpa::HeavyArgs, unsigned int const*, unsigned int)",
    "publish": "lpa::k_publish(unsigned long long*, unsigned int, unsigned int, unsigned long long*)",
    "fill": "lpa::k_fill_u64(unsigned long long*, unsigned long, unsigned long long)",
    "relayout": "lpa::k_relayout(unsigned long const*, unsigned long const*)",
    "copy": "lpa::k_calibration_copy(HIP_vector_type<unsigned int, 4u> const*, HIP_vector_type<unsigned int, 4u>*, unsigned long)",
    "cglp": "lpa::k_decode_bins(lpa::DecodeArgs, lpa::BinTable)",
    "labels": "lpa::k_labels_own(unsigned int*, unsigned int*, unsigned long, unsigned long, unsigned int, unsigned int)",
}
RUN = ["bins", "lane", "decode1", "chunks2", "local0", "publish", "publish", "publish"]
ALONE = ["lane", "lane", "wave", "block", "decode1", "chunks2", "local0", "publish"]


def test_families():
    want = dict(bins="bins", lane="lane", wave="wave", block="block", decode1="cms", chunks2="cms", local0="global",
                publish="step", fill="other", relayout="other", copy="copy", cglp="cglp-decode", labels="other")
    assert {k: family(NAMES[k]) for k in NAMES} == want


def _rows(keys):
    return [dict(Dispatch_Id=str(i), Kernel_Name=NAMES[k], Start_Timestamp=str(1000 * i),
                 End_Timestamp=str(1000 * i + 500), Counter_Name="", Counter_Value="") for i, k in enumerate(keys)]


def _keys(rows):
    names = {v: k for k, v in NAMES.items()}
    return [names[r["Kernel_Name"]] for r in rows]


def test_steps_are_told_apart():
    # two layouts; the counts are cleared once; two warm-up and two timed
    # iterations; rows out of order, as the file may hold them
    trace = ["relayout", "labels", "fill"] + RUN + ["relayout", "labels"] + 2 * RUN + 2 * (RUN + ALONE) + 3 * ["copy"]
    run, alone, copies = _headline(_rows(trace)[::-1], 2)
    assert _keys(run) == 2 * RUN and _keys(alone) == 2 * ALONE and len(copies) == 3
    # a trace that ends within a step
    run, alone, _ = _headline(_rows(trace[:-3] + RUN[:3]), 1)
    assert _keys(run) == RUN and _keys(alone) == ALONE


@pytest.mark.parametrize("trace", [["relayout"] + RUN, ["relayout"] + 4 * RUN])
def test_traces_without_timed_steps_are_refused(trace):
    with pytest.raises(SystemExit):
        _headline(_rows(trace), 1)


def test_summary_files(tmp_path):
    trace = ["relayout", "fill"] + RUN + RUN + ALONE + ["copy"]
    for d, counter in (("T", None), ("F", "FETCH_SIZE"), ("W", "WRITE_SIZE")):
        (tmp_path / d).mkdir()
        rows = _rows(trace)
        for r in rows:
            r["Counter_Name"] = counter or ""
            r["Counter_Value"] = str(256 * 1024 if "copy" in r["Kernel_Name"] else 4)
        with open(tmp_path / d / ("run_counter_collection.csv" if counter else "run_kernel_trace.csv"), "w", newline="") as f:
            w = csv.DictWriter(f, rows[0].keys())
            w.writeheader()
            w.writerows(rows)
    out = tmp_path / "s"
    subprocess.run([sys.executable, "-m", "lpa_amd.rocprof_summary", "--trace", tmp_path / "T", "--fetch", tmp_path / "F",
                    "--write", tmp_path / "W", "--steps", "1", "--command", "a;b", "--workload", "w", "--K", "1",
                    "--out", out], check=True)
    d = json.load(open(f"{out}_traffic.json"))
    assert d["traffic_per_iter"]["lane"]["fetch_bytes"] == 2 * 4096 and d["traffic_per_iter"]["cms"]["write_bytes"] == 2 * 4096
    assert set(d["ms_per_iter"]) == {"lane", "wave", "block", "cms", "global", "step"}
    assert "k_bins" in open(f"{out}_kernels.txt").read()
