"""slab_gemm_kernel waits for its staged tokens by counting loads (vmcnt): the last
four before each counted barrier must be the next step's weights. Device code compiled
here, no GPU: the order in the compiled kernels, and that the weights' pointer passes
through an opaque asm (a plain kernel argument that nothing aliases may be read across
the barriers' memory clobbers)."""

from __future__ import annotations

import re
import shutil
import subprocess

import pytest

from llmq_amd.ops.build import HERE, HIPCC_FLAGS

HIPCC = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")
VARIANTS = [(tm, 1, 0) for tm in (1, 2, 3, 4, 6, 8)] + [       # TM, WK, EPI
    (tm, 2, epi) for tm in (1, 2, 3, 4) for epi in (1, 2)]
SOURCE = '#include "flash_prefill.hip"\n#include "slab_gemm.hip"\n' + "".join(
    f"template __global__ void slab_gemm_kernel<{tm}, {wk}, {epi}>(float*, __hip_bfloat16*, long, "
    "const __hip_bfloat16*, long, const __hip_bfloat16*, int, int, int, int);\n"
    for tm, wk, epi in VARIANTS)


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    if not HIPCC:
        pytest.skip("no hipcc")
    at = tmp_path_factory.mktemp("slab")
    (at / "slab.hip").write_text(SOURCE)

    def emit(name, *flags):
        subprocess.run([HIPCC, *HIPCC_FLAGS, "--offload-arch=gfx950", "--cuda-device-only",
                        f"-I{HERE / 'hip'}", "-S", *flags, str(at / "slab.hip"),
                        "-o", str(at / name)], check=True, capture_output=True, timeout=300)
        return (at / name).read_text()

    return emit("slab.s"), emit("slab.ll", "-emit-llvm")


def loads_and_waits(asm: str):
    """Per kernel its staging loads (L), weight loads (W) and counted barriers (B)."""
    out = {}
    for name, body in re.findall(r"^(_Z16slab_gemm_kernel\w+):.*?\n(.*?)\.Lfunc_end", asm,
                                 re.S | re.M):
        ops = ""
        for line in map(str.strip, body.splitlines()):
            if line.startswith("global_load_lds"):
                ops += "L"
            elif line.startswith("global_load_dwordx4") and line.endswith(" nt"):
                ops += "W"
            elif line.startswith("s_waitcnt vmcnt(4) lgkmcnt(0)"):
                ops += "B"
        out[tuple(map(int, re.findall(r"Li(\d+)E", name)))] = ops
    return out


def test_weights_are_the_last_four_loads(compiled):
    found = loads_and_waits(compiled[0])
    assert set(found) == set(VARIANTS)
    for (tm, _wk, _epi), ops in found.items():
        stage = "L" * tm
        # both weight sets, then two steps a round: barrier, staging, weights
        assert ops == stage + "WWWWWWWW" + 2 * ("B" + stage + "WWWW"), ops


def test_weights_pointer_is_opaque(compiled):
    kernels = re.findall(r"define .*?slab_gemm_kernel.*?\n}", compiled[1], re.S)
    assert len(kernels) == len(VARIANTS)
    for ir in kernels:
        assert 'ptr addrspace(1) asm sideeffect "", "=v,0,~{memory}"' in ir
