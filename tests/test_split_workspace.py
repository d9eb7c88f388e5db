"""The key-range split's geometry and workspace (csrc/kernels.h key_split), compiled for the CPU and
compared with a plain restatement: the workspace holds the partial sums of the rows that are split and
nothing for whole tiles or key streams, and every output row is either whole or split."""

from __future__ import annotations

import random
import shutil
import subprocess
from pathlib import Path

import pytest

from piper_kernels.attention.piper_attention._plan import COMPUTE_UNITS, MAX_KEY_PARTS, split_parts

CSRC = Path(__file__).resolve().parents[1] / "piper-kernels_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include "kernels.h"
int main() {
  long bh, sq; int nkb, d, parts, cus;
  while (std::scanf("%ld %ld %d %d %d %d", &bh, &sq, &nkb, &d, &parts, &cus) == 6) {
    const piper::KeySplit k = piper::key_split(bh, sq, nkb, d, parts, cus);
    std::printf("%d %d %d %ld %ld %ld\n", k.parts, k.streams, k.part_tiles, k.whole_tiles, k.row0, k.bytes);
  }
}
"""


@pytest.fixture(scope="module")
def key_split(tmp_path_factory):
    folder = tmp_path_factory.mktemp("key_split")
    source, program = folder / "key_split.cpp", folder / "key_split"
    source.write_text(PROGRAM)
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", f"-I{CSRC}", "-I/opt/rocm/include",
                    "-w", "-o", str(program), str(source)], check=True)

    def run(cases):
        lines = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(program)], input=lines, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def test_partial_sums_cover_the_split_rows_and_no_others(key_split) -> None:
    rng = random.Random(7)
    cases = [(bh, sq, nkb, d, parts, cus) for bh in (1, 3, 24) for sq in (1, 128, 129, 5000) for nkb in (1, 2, 7, 256)
             for d in (64, 128) for parts in range(1, 9) for cus in (32, 256)]
    cases += [(rng.randint(1, 200), rng.randint(1, 40000), rng.randint(1, 700), rng.choice((64, 128)), rng.randint(1, 8), 256)
              for _ in range(2000)]
    for case, (got_parts, streams, part_tiles, whole, row0, size) in zip(cases, key_split(cases), strict=True):
        bh, sq, nkb, d, parts, cus = case
        per_head = -(-sq // 128)
        tiles = per_head * bh
        if streams > 1:
            assert streams == parts and got_parts == 1 and size == 0, case
        elif got_parts == 1:
            assert size == 0, case
        else:
            slots = cus * (4 if d == 64 else 3)
            rows = sum(min(128, sq - t % per_head * 128) for t in range(tiles // slots * slots, tiles))
            assert whole == tiles // slots * slots and row0 == bh * sq - rows, case
            assert size == got_parts * rows * (d + 2) * 4 and 0 < rows <= slots * 128, case
            assert (got_parts - 1) * part_tiles < nkb <= got_parts * part_tiles, case  # no empty part


@pytest.mark.parametrize("shape", [(1, 4, 100000, 100000), (1, 20, 20000, 20000), (2, 37, 6542, 6542), (1, 25, 27764, 4893)])
def test_a_chosen_split_needs_less_than_one_round_of_partial_sums(key_split, shape) -> None:
    """Grids of several rounds, which the plan splits into up to eight parts: at most a round of query rows
    times the parts, where counting every row of the call asked 1.0 to 2.9 GB."""
    b, h, sq, sk = shape
    parts = split_parts(b, h, sq, sk, 128)
    assert 1 < parts <= MAX_KEY_PARTS
    (_, _, _, _, _, size), = key_split([(b * h, sq, -(-sk // 64), 128, parts, COMPUTE_UNITS)])
    assert size <= 32 << 20
