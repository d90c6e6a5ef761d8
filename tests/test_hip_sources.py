"""Both extensions' sources compile for gfx950 as they are now: the libraries that the
GPU tests load may be older than the sources."""

from __future__ import annotations

import shutil
import subprocess
import sysconfig

import pytest

from llmq_amd.ops.build import GROUPS, HIPCC_FLAGS

HIPCC = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not HIPCC, reason="no hipcc")
@pytest.mark.parametrize("group", GROUPS)
def test_umbrella_unit_compiles(group):
    from torch.utils import cpp_extension as ext

    includes = [*ext.include_paths("cuda"), sysconfig.get_path("include")]
    done = subprocess.run(
        [HIPCC, *ext.COMMON_HIP_FLAGS, *ext.COMMON_HIPCC_FLAGS, *HIPCC_FLAGS,
         "--offload-arch=gfx950", "--cuda-device-only", "-fsyntax-only",
         *[f"-I{path}" for path in includes], str(GROUPS[group][0])],
        capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr[-4000:]
