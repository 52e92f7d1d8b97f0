"""bench.py's roofline takes the kernels' counters from a committed file only while the kernels' sources
are those that the counters were taken of."""

import json

import bench


def test_counters_of_other_sources_are_not_reported(tmp_path, monkeypatch):
    e = {"fetch_kib": 2.0, "write_kib": 1.0, "valu_busy": 0.5, "flops": 3.0}
    doc = {"fetch_scale": 2.0, "write_scale": 1.0, "runs": {"w/fp64/grad": e},
           "kernel_sources_sha256": bench.kernel_sources_sha256()}
    path = tmp_path / "counters.json"
    monkeypatch.setattr(bench, "TRAFFIC_FILE", str(path))
    path.write_text(json.dumps(doc))
    assert bench.traffic_of("w", "fp64", True) == (5.0 * 1024, 0.5, 3.0)
    assert bench.traffic_of("w", "mixed", True) == (None, None, None)
    path.write_text(json.dumps(dict(doc, kernel_sources_sha256="0" * 64)))
    assert bench.traffic_of("w", "fp64", True) == (None, None, None)
