"""The benchmark reports counters from a committed profile: only for the workload, the sources and the compiler flags they were taken with."""
import importlib
import json

import bench


def test_traffic_record_follows_the_build(tmp_path, monkeypatch):
    flags, record = tmp_path / "device_flags.txt", tmp_path / "traffic.json"
    monkeypatch.setattr(bench, "BUILD_FLAGS", str(flags))
    monkeypatch.setattr(bench, "PROFILED_TRAFFIC", str(record))
    workload = dict(config=4, n_train=100, k=128, seed=1, workers=16)

    flags.write_text("a.hip: -O3\n")
    record.write_text(json.dumps(dict(workload, kernel_build_sha256=bench.kernel_build_digest(), bytes_per_epoch=7)))
    assert bench.profiled_traffic(4, 100, 128, 1, 16)["bytes_per_epoch"] == 7
    assert bench.profiled_traffic(4, 100, 64, 1, 16) is None
    flags.write_text("a.hip: -O3 -mllvm -enable-tail-merge=false\n")
    assert bench.profiled_traffic(4, 100, 128, 1, 16) is None
    flags.unlink()
    assert bench.profiled_traffic(4, 100, 128, 1, 16) is None
    record.write_text(json.dumps(dict(workload, kernel_build_sha256=None, bytes_per_epoch=7)))
    assert bench.profiled_traffic(4, 100, 128, 1, 16) is None


def test_the_build_records_every_files_flags(tmp_path, monkeypatch):
    builder = importlib.import_module("icdm-2021_mascot_amd.build")
    lines = dict(line.split(": ", 1) for line in builder.flags_record().splitlines())
    assert sorted(lines) == sorted(builder.KERNEL_SOURCES)
    for src, flags in lines.items():
        assert flags.split() == builder.device_flags(src)
    assert builder.STRUCTURISED < set(lines)
    assert {src for src, flags in lines.items() if builder.UNIFORM_BRANCH_FLAGS[1] not in flags} == builder.STRUCTURISED
    monkeypatch.setattr(builder, "EXTRA_FLAGS", ["-DX=1"])
    assert all(line.endswith(" -DX=1") for line in builder.flags_record().splitlines())
