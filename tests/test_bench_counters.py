"""The bench reports hardware counters of a profiled run only for the kernels
and the workload that they were taken of."""
import hashlib
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_counters_belong_to_the_sources_and_pairs(tmp_path, monkeypatch):
    import bench
    csrc = "starformationhistories.jl_amd/csrc"
    with open(os.path.join(ROOT, "profiles", "deposit_counters.json")) as f:
        c = json.load(f)
    (tmp_path / "profiles").mkdir()
    (tmp_path / csrc).mkdir(parents=True)
    for name in ("sfh_psf.h", "sfh_deposit.hip"):
        (tmp_path / csrc / name).write_text(name)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.deposit_counters(c["kernel_points"], c["pairs"]) is None         # no file
    c["sources_sha256"] = hashlib.sha256(b"sfh_psf.hsfh_deposit.hip").hexdigest()
    (tmp_path / "profiles" / "deposit_counters.json").write_text(json.dumps(c))
    assert bench.deposit_counters(c["kernel_points"], c["pairs"]) == c["kernels"]
    assert bench.deposit_counters(c["kernel_points"], c["pairs"] + 1) is None     # other templates
    (tmp_path / csrc / "sfh_psf.h").write_text("changed")
    assert bench.deposit_counters(c["kernel_points"], c["pairs"]) is None         # other kernels
