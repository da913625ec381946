"""bench.py's HBM traffic figure belongs to the kernels it runs: a record made with other sources under
csrc/ is not reported."""
import bench


def _record(tmp_path, monkeypatch, digest):
    (tmp_path / "profiles").mkdir()
    (tmp_path / "profiles" / "scene_hbm_traffic.md").write_text(
        f"# a record\n\nkernel_sources: {digest}\ntraffic_bytes_per_frame_exact: 1000\n")
    digest_now = bench.kernel_sources_digest()
    monkeypatch.setattr(bench, "kernel_sources_digest", lambda: digest_now)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))


def test_record_of_these_sources(tmp_path, monkeypatch):
    _record(tmp_path, monkeypatch, bench.kernel_sources_digest())
    assert bench.measured_traffic("scene", "exact") == (1000.0, "profiles/scene_hbm_traffic.md")
    assert bench.measured_traffic("scene", "coloured") == (None, None)
    assert bench.measured_traffic("other", "exact") == (None, None)


def test_record_of_other_sources(tmp_path, monkeypatch):
    _record(tmp_path, monkeypatch, "0" * 16)
    value, source = bench.measured_traffic("scene", "exact")
    assert value is None and "other kernel sources" in source
