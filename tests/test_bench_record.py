"""bench.py's record, as far as it can be checked without a GPU."""
import os

import bench


def test_a_missing_cpu_baseline_says_why(tmp_path, monkeypatch):
    """A run that cannot time the reference CPU solver is told apart from one that
    was asked not to (null)."""
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    r = bench.cpu_baseline(2406)
    assert r["value"] is None and "ref_solver_sample" in r["skipped"]
    exe = tmp_path / "oracle" / "_ref" / "ref_solver_sample"
    os.makedirs(exe.parent)
    exe.touch()
    monkeypatch.setattr(bench.shutil, "which", lambda name: str(tmp_path / "no" / name))
    r = bench.cpu_baseline(2406)
    assert r["value"] is None and r["skipped"] == "missing: mpirun"
