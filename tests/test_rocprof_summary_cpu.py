"""The HBM traffic record is the mean over launches of one problem size, scaled by a copy of known size."""
import json

import pytest

from intra_amd import rocprof_summary

COPY_KIB = rocprof_summary.COPY_BYTES / 1024


def counter_run(path, counter, launches, copies):
    path.mkdir()
    rows = [("intra::intra_fwd_kernel<M>", v) for v in launches] + [("__amd_rocclr_copyBuffer", v) for v in copies]
    lines = ["Kernel_Name,Counter_Name,Counter_Value"] + [f"{kernel},{counter},{value}" for kernel, value in rows]
    (path / "r_counter_collection.csv").write_text("\n".join(lines) + "\n")


def record(tmp_path, monkeypatch, fetch):
    counter_run(tmp_path / "fetch", "FETCH_SIZE", fetch, [3.0, COPY_KIB / 2])
    counter_run(tmp_path / "write", "WRITE_SIZE", [300000.0, 302000.0], [3.0, COPY_KIB])
    out = tmp_path / "traffic.json"
    monkeypatch.setattr("sys.argv", ["rocprof_summary", "traffic", "--fetch", str(tmp_path / "fetch"), "--write",
                                     str(tmp_path / "write"), "--out", str(out)])
    rocprof_summary.main()
    return json.loads(out.read_text())


def test_mean_of_launches_scaled_by_the_copy(tmp_path, monkeypatch):
    got = record(tmp_path, monkeypatch, [240000.0, 250000.0])
    assert got["fetch_size"]["scale"] == 2.0 and got["write_size"]["scale"] == 1.0
    assert got["hbm_bytes_per_launch"] == (2 * 245000 + 301000) * 1024


def test_launches_of_several_sizes_are_refused(tmp_path, monkeypatch):
    with pytest.raises(SystemExit, match="several sizes"):
        record(tmp_path, monkeypatch, [240000.0, 250000.0, 60000.0])
