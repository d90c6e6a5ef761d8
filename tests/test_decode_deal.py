"""Decode attention's rules, compiled from the kernel's own source and run here without a GPU: what
its workgroups take of a CU and how they cut a sequence."""

from __future__ import annotations

import shutil
import subprocess

import pytest

from decode_batches import BATCHES, VARIANTS
from llmq_amd.ops.build import HERE, HIPCC_FLAGS

HIPCC = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")
SOURCE = r"""
#include "paged_decode.hip"
#include <algorithm>
#include <cstdio>
#include <cstring>

// Pieces of the size that the kernel makes of their count: none empty, none over its size.
void pieces(int least, int c, float thick) {
  int most = 0;
  for (int nt = 1; nt <= 70000; nt += nt < 3000 ? 1 : 97) {
    const int of = pd_pieces(nt, c, least, thick);
    const int size = pd_quotient(nt + of - 1, pd_rcp((float)of));
    if (of < 1 || size != (nt + of - 1) / of || (long)(of - 1) * size >= nt ||
        of > (nt + c - 1) / c || (nt <= 2 * least && of != 1) || pd_pieces(0, c, least, thick))
      printf("%d %d %d %d\n", nt, c, of, size);
    most = of > most ? of : most;
  }
  printf("%d\n", most);
}

// The deal of a batch on 256 CUs, after its least pieces' count and a piece's tiles; then the tiles
// of a kv head of every sequence.
template <int D, typename TC>
void deal(int G, int KVH, int width, int window, char** from, char** to) {
  constexpr PdVariant v = pd_variant(D, sizeof(TC) == 1);
  using Shape = PdShape<D, TC, v.groups>;
  constexpr int kLeast = Shape::kLeastPiece;
  const float thick = G * (2.f / (Shape::kKeys * (int)sizeof(TC)));
  const int pairs = (int)(to - from) * KVH, resident = 256 * v.resident;
  const int wgs = (int)pd_workgroups(pairs, width / Shape::kKeys + 1, kLeast, resident);
  int total = 0, n0 = 0, most = 0;
  for (char** at = from; at < to; ++at) {
    const int n = pd_tiles<Shape::kTileShift>(atoi(*at), window);
    total += n * KVH;
    n0 += pd_pieces(n, kLeast, kLeast, thick) * KVH;
    most = std::max(most, n);
  }
  PdDeal d{kLeast, 1, n0};
  if (n0 > wgs)
    d = pd_choose(total, most, pairs, wgs, std::min(resident, wgs), kLeast,
                  D == 256 && sizeof(TC) == 2);
  printf("%d %d %d %d %d\n", n0 <= wgs, d.piece, most, d.share, d.total);
  for (char** at = from; at < to; ++at)
    printf("%d ", pd_tiles<Shape::kTileShift>(atoi(*at), window));
}

template <int D, typename TC>
void variant() {
  constexpr bool fp8 = sizeof(TC) == 1;
  constexpr PdVariant v = pd_variant(D, fp8);
  for (int G = 1; G <= (D == 64 ? 8 : 16); ++G)
    printf("%d %d %d %d %d\n", D, fp8, G, v.resident, 4 * PdShape<D, TC, v.groups>::wave_lds(G));
}

int main(int argc, char** argv) {
  if (argc > 1 && !strcmp(argv[1], "pieces")) {
    pieces(atoi(argv[2]), atoi(argv[3]), atof(argv[4]));
    return 0;
  }
  if (argc > 1) {
    const int D = atoi(argv[2]), fp8 = atoi(argv[3]);
    auto go = [&]<int HD, typename TC>() {
      if (D == HD && fp8 == (sizeof(TC) == 1))
        deal<HD, TC>(atoi(argv[4]), atoi(argv[5]), atoi(argv[6]), atoi(argv[7]), argv + 8,
                     argv + argc);
    };
    go.template operator()<64, __hip_bfloat16>();
    go.template operator()<128, __hip_bfloat16>();
    go.template operator()<256, __hip_bfloat16>();
    go.template operator()<128, __hip_fp8_e4m3>();
    go.template operator()<256, __hip_fp8_e4m3>();
    return 0;
  }
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


@pytest.mark.parametrize("least", [4, 8])
@pytest.mark.parametrize("longer", [0, 1, 3, 60, 1001])
@pytest.mark.parametrize("thick", [1 / 32, 0.125, 0.375, 1.0, 2.0])
def test_no_piece_is_empty(program, least, longer, thick):
    out = program("pieces", least, least + longer, thick)
    assert len(out) == 1, out[:5]                            # the largest count, no exceptions
    # the floor: sqrt(1.5 thick nt) tiles, no more than rounded up by four
    assert out[0][0] <= 70000 / max(least + longer, (1.5 * thick * 70000) ** 0.5 - 1) + 1


@pytest.mark.parametrize("batch", range(len(BATCHES)))
@pytest.mark.parametrize("variant", range(len(VARIANTS)))
def test_batches_take_their_ways(program, batch, variant):
    """The GPU tests' batches are dealt as they are meant to be. Equal ranges hold the end of a
    pair, whole ones and the start of another, and step over empty sequences."""
    D, G, fp8 = VARIANTS[variant]
    ways, lens, KVH, BS, window, _ = BATCHES[batch]
    (least, piece, most, share, total), tiles = program(
        "deal", D, int(fp8), G, KVH, -(-max(lens) // BS) * BS, window, *lens)
    way = "L" if least else "R" if piece == 0 else "W" if piece == most else "P"
    assert way == ways[variant]
    if way == "P":
        assert piece < most
    if way != "R":
        return
    assert total == sum(tiles) * KVH
    ends, segments = [0], []
    for b, n in enumerate(tiles):
        for _ in range(KVH if n else 0):
            ends.append(ends[-1] + n)
            segments.append(b)
    kinds = set()
    for lo in range(0, total, share):
        hi = min(total, lo + share)
        mine = [i for i, b in enumerate(segments) if ends[i] < hi and ends[i + 1] > lo]
        cut = ends[mine[0]] < lo, ends[mine[-1] + 1] > hi
        kinds.add((cut, len(mine) > 2))
        seen = [segments[i] for i in mine]
        if any(d > c + 1 for c, d in zip(seen, seen[1:])):
            kinds.add("empty")
    assert ((True, True), True) in kinds and "empty" in kinds
