"""The choice of macro tile and split (fo_plan.h), in a CPU build, against measured times: shapes in which the plans
that come near differ by more than the noise of a measurement."""
import math
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))

# plain GEMM with its bulk copy on an MI355X: (tile rows, tile columns, parts) -> us with operands from HBM, and from the memory-side cache
MEASURED = {
    (2041, 4096, 7168): {(256, 128, 1): (104.2, 101.5), (256, 256, 2): (113.0, 111.2), (128, 128, 1): (121.5, 107.0)},
    (2048, 4096, 7168): {(256, 128, 1): (105.0, 90.1), (256, 256, 2): (104.1, 102.0), (128, 128, 1): (117.5, 97.8)},
    (8192, 1024, 7040): {(256, 128, 1): (102.0, 94.7), (256, 256, 2): (106.8, 104.9), (128, 128, 1): (126.7, 103.6)},
    (4608, 1536, 6528): {(256, 128, 1): (90.3, 80.6), (256, 256, 2): (91.8, 88.8), (128, 128, 1): (101.0, 87.9)},
    (1664, 4608, 8000): {(256, 128, 1): (106.2, 100.9), (256, 256, 2): (111.6, 108.6), (128, 128, 1): (119.6, 105.0)},
    (77, 7680, 7936): {(128, 128, 4): (29.8, 24.9), (128, 128, 3): (33.9, 25.7), (64, 64, 1): (39.3, 26.9),
                       (64, 64, 2): (35.6, 31.7), (128, 128, 2): (42.4, 29.9)},
    (4608, 1152, 4544): {(256, 128, 1): (61.6, 50.0), (128, 128, 2): (67.0, 53.5), (128, 128, 3): (68.2, 53.6),
                         (128, 128, 1): (67.3, 54.4), (256, 256, 2): (61.4, 59.8)},
    (2688, 2816, 576): {(128, 128, 1): (12.6, 12.4), (256, 128, 1): (13.6, 13.4)},
    (6683, 1336, 1600): {(256, 256, 1): (38.6, 37.0), (128, 128, 3): (45.2, 36.9), (128, 128, 2): (46.8, 37.6),
                         (128, 128, 1): (51.6, 38.9), (256, 128, 1): (53.5, 44.4)},
    (640, 3840, 7872): {(256, 256, 5): (52.1, 52.4), (256, 256, 4): (54.5, 52.7), (256, 256, 3): (61.7, 58.5),
                        (128, 128, 1): (74.3, 51.0)},
    (1152, 3200, 7512): {(256, 256, 3): (76.7, 67.0), (128, 128, 1): (101.3, 74.6), (256, 256, 2): (95.3, 81.1)},
    (2688, 1920, 4944): {(256, 256, 2): (71.0, 64.2), (128, 128, 4): (78.8, 67.2), (128, 128, 3): (82.2, 65.6),
                         (128, 128, 2): (87.4, 70.1), (256, 128, 1): (92.4, 67.5)},
    (128, 4096, 7168): {(64, 64, 2): (23.2, 16.6), (128, 128, 8): (21.4, 18.5), (128, 128, 7): (22.0, 18.5),
                        (64, 64, 4): (24.2, 17.3), (128, 128, 6): (23.0, 18.2)},
    (1024, 8192, 3584): {(256, 128, 1): (54.3, 49.1), (128, 128, 1): (62.1, 52.4), (256, 256, 2): (67.7, 64.8),
                         (256, 256, 1): (71.8, 66.8)},
}


def test_the_plan_is_among_the_fastest_measured(tmp_path):
    exe = str(tmp_path / "plan_choice")
    csrc = os.path.join(HERE, "..", "flashoverlap_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", csrc, os.path.join(HERE, "plan_choice.cpp"), "-o", exe], check=True)
    asked = "".join("%d %d %d\n" % s for s in MEASURED)
    said = subprocess.run([exe], input=asked, capture_output=True, text=True, check=True).stdout.splitlines()
    slow = []
    for (shape, times), line in zip(MEASURED.items(), said):
        plan = tuple(int(v) for v in line.split())
        best = min(math.prod(t) for t in times.values())
        # two runs of one plan differ by up to 3 %
        if plan not in times or math.sqrt(math.prod(times[plan]) / best) > 1.03:
            slow.append((shape, plan))
    assert not slow
