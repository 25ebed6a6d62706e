"""What bench.py says about figures that it reads from files instead of measuring them."""
import shutil

import pytest

import bench


@pytest.mark.parametrize("changed", [None, "gemm_large_kernel.hpp", "gemm_tiles.hpp"])
def test_recorded_traffic_is_called_stale_once_a_source_of_the_kernel_has_changed(changed, tmp_path, monkeypatch):
    """The traffic of the probe's launch is set by its kernel and by the operand loads that the kernel includes."""
    for name in ("gemm_large_kernel.hpp", "gemm_tiles.hpp"):
        shutil.copy(f"{bench.CSRC}/{name}", tmp_path)
    monkeypatch.setattr(bench, "CSRC", str(tmp_path))
    summary = tmp_path / "summary.txt"
    summary.write_text(f"traffic_bytes_per_launch = 470067610\ngemm_hip_sha256 = {bench.source_digest()}\n")
    monkeypatch.setattr(bench, "TRAFFIC_FILE", str(summary))
    if changed:
        with open(tmp_path / changed, "a") as handle:
            handle.write("\n")
    value, note = bench.measured_traffic()
    assert value == 470067610
    assert note.startswith("STALE") == (changed is not None)
