"""bench.py's roofline block: counters of a profile stand beside a run only if
both had the same tuning."""
import json

import bench


def block(tmp_path, monkeypatch, counted, ran):
    f = tmp_path / "traffic.json"
    f.write_text(json.dumps({"tuning": counted, "per_launch": {"raster_g1": {"read_bytes": 7, "write_bytes": 5, "valu_instr": 900}}}))
    monkeypatch.setitem(bench.TRAFFIC_FILES, "c3", str(f))
    return bench.roofline("c3", {"raster_g0": 0.1, "raster_g1": 0.4}, {"raster_g1": 2}, {"raster_g1": 1e6}, ran)


def test_counters_of_the_same_tuning(tmp_path, monkeypatch):
    ran = {"tile_size": 16, "raster_wgs_per_cu": 0, "parts": 4, "raster_waves": 2, "ms": 1.2}
    out = block(tmp_path, monkeypatch, [16, 0, 4, 2], ran)
    assert out["traffic"] == 12 and out["valu"]["wave_instr_per_launch"] == 900 and out["launch_us"] == 200.0


def test_no_counters_of_another_tuning(tmp_path, monkeypatch):
    ran = {"tile_size": 32, "raster_wgs_per_cu": 0, "parts": 4, "raster_waves": 4, "ms": 1.2}
    for counted in ([16, 0, 4, 2], None):
        out = block(tmp_path, monkeypatch, counted, ran)
        assert out["traffic"] is None and out["traffic_source"] is None and "valu" not in out
        assert out["launch_us"] == 200.0
