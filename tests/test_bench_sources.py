"""bench.py tells measured traffic of another build by the sources of the kernel, wherever in them a change is."""
import shutil
from pathlib import Path

import bench

CSRC = Path(bench.ROOT) / "wgml_amd" / "csrc"


def test_a_changed_kernel_is_noticed(tmp_path):
    for name in ("gemv.hip", "gemv_kernels.h", "device_utils.h"):
        shutil.copytree(CSRC, tmp_path / name, ignore=shutil.ignore_patterns("build"))
        assert bench.gemv_sources_sha256(str(tmp_path / name)) == bench.gemv_sources_sha256()
        with open(tmp_path / name / name, "a") as f:
            f.write("//\n")
        assert bench.gemv_sources_sha256(str(tmp_path / name)) != bench.gemv_sources_sha256()
