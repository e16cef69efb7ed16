"""Tile width and occupancy cap of the step kernels (csrc/launch_rules.hpp), compiled for the host."""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "launch_rules"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(HERE.parent / "cfd_solvers_amd" / "csrc"),
                    str(HERE / "host" / "launch_rules.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_width_covers_the_row(rules):
    """Blocks of at most kStepThreads threads that launch few wavefronts beyond the row's end."""
    assert len(rules) == 3 * 2 * 80
    for elem, flagged, segments, width, *_ in rules:
        tile = width // 64
        assert width % 64 == 0 and 1 <= tile <= (4 if elem == 8 else 8)
        launched = -(-segments // tile) * tile
        assert launched <= max(1.125 * segments + (2 if elem == 8 else 1), 4), (elem, segments, width)


def test_caps_survive_the_width(rules):
    """The blocks that fit 160 KiB hold the waves asked for to half a wave a SIMD, whatever the width (FP16S
    is capped in plain planes alone, at 5, where 512-thread blocks give 6)."""
    for elem, flagged, segments, width, *lds in rules:
        if elem == 2:
            continue
        threads = max(width, 256)
        for waves, bytes_ in zip((3, 4, 5), lds):
            got = 163840 // (bytes_ + 1024) * threads / 256
            assert abs(got - waves) <= 0.5, (elem, segments, width, waves, got)
