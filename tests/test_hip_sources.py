"""Both extensions' sources compile for gfx950 as they are now: the libraries that the
GPU tests load may be older than the sources."""

from __future__ import annotations

import shutil
import subprocess
import sysconfig

import pytest

from llmq_amd.ops import build
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


class TestBuildErrors:
    """What torch's extension loader raises: a RuntimeError where compiling fails, an OSError
    where the library does not load; a name that it has built once is not built again."""

    @pytest.fixture
    def loads(self, tmp_path, monkeypatch):
        (tmp_path / "x.hip").write_text("")
        monkeypatch.setitem(build.GROUPS, "x", (tmp_path / "x.hip", tmp_path / "x.so",
                                                tmp_path / "b", "ext"))
        calls, errors = [], []

        def load(name, build_directory, **_):
            again = name in calls
            calls.append(name)
            if again:
                raise OSError("cannot open shared object file")
            if errors:
                raise errors.pop()
            with open(f"{build_directory}/{name}.so", "w") as f:
                f.write(name)

        monkeypatch.setattr("torch.utils.cpp_extension.load", load)
        return calls, errors

    def test_compile_error_is_raised(self, loads):
        calls, errors = loads
        errors.append(RuntimeError("error: call to 'f' is ambiguous"))
        with pytest.raises(RuntimeError, match="ambiguous"):
            build.build(force=True, group="x")
        assert calls == ["ext"]

    def test_library_that_does_not_load_is_built_anew(self, loads):
        calls, errors = loads
        errors.append(OSError("undefined symbol"))
        assert build.build(force=True, group="x").read_text() == "ext_clean"
        assert calls == ["ext", "ext_clean"]
