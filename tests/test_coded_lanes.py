"""The reads of the kernels over entry codes stay inside their vectors: tests/coded_lanes.cpp replays every lane of the
grid with the functions that the kernels use (coded_lane.h)."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    exe = tmp_path_factory.mktemp("coded") / "coded_lanes"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'hazmath_amd' / 'csrc'}", "-o", str(exe),
                    str(ROOT / "tests" / "coded_lanes.cpp")], check=True)
    return exe


# wavefronts past the last slice: none (1,024 rows: 16 slices), one, two and three, with a last slice of 1, 40 and 64
# rows; one slice alone; words: one, and five (a second round)
@pytest.mark.parametrize("n", [64, 65, 104, 1024, 1025, 1064, 1088, 1128, 1152, 1192, 1216])
@pytest.mark.parametrize("words,offsets", [(1, (-1, 0, 1)), (2, (-63, -1, 0, 1, 63)), (5, tuple(range(-9, 10)))])
@pytest.mark.parametrize("bytes_", [4, 8])
def test_every_lane_reads_inside_the_vector(replay, n, words, offsets, bytes_):
    r = subprocess.run([str(replay), str(n), str(words), str(bytes_), *map(str, offsets)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
