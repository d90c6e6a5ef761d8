"""Decode attention's host side, compiled from the kernel's own source and run here without a
GPU: what its workgroups take of a CU."""

from __future__ import annotations

import shutil
import subprocess

import pytest

from llmq_amd.ops.build import HERE, HIPCC_FLAGS

HIPCC = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")
SOURCE = r"""
#include "paged_decode.hip"
#include <cstdio>

template <int D, typename TC>
void variant() {
  constexpr bool fp8 = sizeof(TC) == 1;
  constexpr PdVariant v = pd_variant(D, fp8);
  for (int G = 1; G <= (D == 64 ? 8 : 16); ++G)
    printf("%d %d %d %d %d\n", D, fp8, G, v.resident, 4 * PdShape<D, TC, v.groups>::wave_lds(G));
}

int main() {
  variant<64, __hip_bfloat16>();
  variant<128, __hip_bfloat16>();
  variant<256, __hip_bfloat16>();
  variant<128, __hip_fp8_e4m3>();
  variant<256, __hip_fp8_e4m3>();
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not HIPCC:
        pytest.skip("no hipcc")
    at = tmp_path_factory.mktemp("deal")
    (at / "deal.hip").write_text(SOURCE)
    subprocess.run([HIPCC, *HIPCC_FLAGS, "--offload-arch=gfx950", "--cuda-host-only",
                    f"-I{HERE / 'hip'}", str(at / "deal.hip"), "-o", str(at / "deal")],
                   check=True, capture_output=True, timeout=300)

    def run(*args):
        out = subprocess.run([str(at / "deal"), *map(str, args)], check=True,
                             capture_output=True, text=True, timeout=60).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def test_workgroups_of_a_cu_fit_its_lds(program):
    """The launch counts them by registers alone: a batch dealt to more workgroups than run at a
    time takes a second round."""
    granule, cu, fixed = 1280, 160 * 1024, 1024              # fixed: the kernel's own arrays
    for D, fp8, G, resident, lds in program():
        of_one = -(-(lds + fixed) // granule) * granule
        assert resident * of_one <= cu, (D, fp8, G)
