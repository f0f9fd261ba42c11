"""Which calls in 256x128 tiles let the XCDs begin at eight places of K (turn_panels, fo_plan.h), in a CPU build: the edges of the
rule, and shapes on both sides of it against measured times."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

# plain GEMM with its bulk copy in 256x128 tiles, bf16, operands from HBM, MI355X, us: all XCDs at panel 0, and apart
MEASURED = {
    (2048, 3328, 4160): (57.7, 52.4), (2048, 2560, 6144): (105.1, 85.8), (512, 13312, 4160): (61.1, 57.1), (1536, 4352, 4160): (58.1, 55.3),
    (2176, 2304, 4160): (56.9, 51.0), (3072, 2176, 4160): (58.1, 53.7), (2816, 1920, 6272): (83.3, 76.2), (3200, 2048, 4160): (58.6, 53.7),
    (4224, 1152, 4160): (57.9, 53.3), (4864, 1024, 6272): (86.5, 81.2), (5120, 1280, 4160): (58.8, 56.5), (6144, 768, 4160): (58.8, 55.6),
    (6272, 1024, 4160): (59.8, 57.6),
    # rows of tiles that one XCD has to itself: a last band of one or two rows, bands of few columns
    (2304, 2304, 4160): (57.6, 60.6), (3328, 2048, 4160): (58.3, 61.8), (4352, 1536, 4160): (58.3, 60.8), (4608, 1408, 4160): (58.5, 61.0),
    (5376, 1152, 4160): (58.3, 60.7), (5632, 1152, 4160): (58.9, 61.8), (6656, 1024, 4160): (59.4, 62.9), (7168, 896, 4160): (59.7, 63.5),
    (7680, 1024, 4160): (63.2, 66.6), (9216, 896, 4160): (64.0, 68.3), (10240, 640, 4160): (61.0, 64.5),
    # 200 rows and 232 in the last row of tiles
    (2248, 3072, 6272): (87.2, 81.5), (2280, 3072, 6272): (86.4, 89.0),
    # a last band of three rows, 70 and 128 rows in the last of them
    (5702, 1280, 4288): (64.8, 62.8), (5760, 1152, 4160): (60.1, 56.6), (5760, 896, 4160): (58.9, 60.3),
    # 8, 16 and 32 columns in the last column of tiles, 40 and more
    (3755, 1320, 8128): (106.8, 96.4), (2663, 2220, 7616): (101.6, 95.9),
    (1024, 5768, 6272): (77.8, 80.0), (1024, 5792, 6272): (77.3, 79.5), (1024, 5840, 6272): (82.3, 80.1), (768, 8096, 6272): (78.5, 80.5),
    (768, 8160, 6272): (84.7, 81.2), (2432, 2960, 6272): (79.2, 83.0), (3584, 2064, 6272): (80.9, 83.1), (3584, 2144, 6272): (89.2, 82.7),
}


@pytest.fixture(scope="module")
def turn(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("turn") / "turn_choice")
    csrc = os.path.join(HERE, "..", "flashoverlap_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", csrc, os.path.join(HERE, "turn_choice.cpp"), "-o", exe], check=True)

    def ask(shapes):
        out = subprocess.run([exe], input="".join("%d %d %d\n" % s for s in shapes), capture_output=True, text=True, check=True).stdout
        tall, square = zip(*(map(int, line.split()) for line in out.splitlines()))
        assert not any(square)
        return tall
    return ask


def test_the_faster_way_is_taken(turn):
    slow = [(shape, t) for (shape, t), panels in zip(MEASURED.items(), turn(MEASURED)) if t[panels > 0] > 1.01 * min(t)]
    assert not slow


def test_edges_of_the_rule(turn):
    # 47 panels, 48, 49, 63, 64, a partial last panel, a full round of 256 tiles, one tile more
    assert turn([(2048, 2560, k) for k in (3008, 3072, 3136, 4032, 4096, 4104)]) == (0, 6, 6, 7, 8, 0)
    assert turn([(2048, 4096, 4096), (2048, 4224, 4096), (256, 32768, 4096), (1, 1, 4096), (1, 65472, 4096)]) == (8, 0, 8, 0, 0)
