"""The staged f16 kernel's reads (libosmos_amd/csrc/mmstage.h's index rule, which the kernel uses), every thread, round and row on
the host: none ends past the matrix, whatever the width leaves of the last round. An earlier rule did for threads past a round's
words, which the same check finds: bits cannot, since those words are never stored."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
# block values, bytes, slab, waves (mm.hip's tuned, short and odd shapes of the types that are staged)
SHAPES = {"Q4_0": (32, 18, 64, 4), "Q8_0": (32, 34, 128, 8), "Q8_0 odd": (32, 34, 64, 2), "Q2_K": (256, 84, 64, 8),
          "Q5_K": (256, 176, 32, 8), "Q6_K": (256, 210, 128, 8), "Q6_K short": (256, 210, 64, 8), "IQ2_XS": (256, 74, 128, 4),
          "IQ2_S": (256, 82, 128, 4), "IQ4_NL": (32, 18, 64, 4), "IQ4_XS": (256, 136, 64, 4)}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("mm_stage") / "driver")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", os.path.join(HERE, "mm_stage_driver.cpp"), "-o", exe],
                   check=True)
    return exe


def test_reads_end_inside(driver):
    lines = []
    for values, bytes_, slab, waves in SHAPES.values():
        step = max(values, slab)
        for cols in range(step, 2 * slab * waves + step + 1, step):
            for rows in (16, 80):
                for tiles in (1, 4):
                    lines.append((rows, cols, values, bytes_, slab, waves, tiles))
    text = "\n".join(" ".join(map(str, v)) for v in lines)
    out = subprocess.run([driver], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
    got = [tuple(map(int, v.split())) for v in out if v]
    assert len(got) == len(lines)
    for case, (total, end, _) in zip(lines, got):
        assert end <= total, case
    past = [case for case, (total, _, old_end) in zip(lines, got) if old_end > total]
    assert past and all(case[1] % (case[4] * case[5]) for case in past)  # (short last rounds only)
