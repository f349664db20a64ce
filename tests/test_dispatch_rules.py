"""The dispatch rules that csrc/kernels.hpp states, at calls whose both sides were timed on one card: the side that a
call takes is the faster one wherever they differ by more than 15%."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "qwen3-local-test_amd", "csrc")

# (pos, n, cr, budget, heads, dims), us of the whole call in the few-token and the many-token launches
QSA = [((16384, 16, 4, 2048, 4, 128), 31, 28), ((16384, 512, 4, 2048, 4, 128), 634, 67),
       ((16384, 16, 4, 2048, 16, 128), 39, 65), ((16384, 40, 4, 2048, 16, 128), 80, 65),
       ((16384, 16, 4, 2048, 8, 256), 51, 66), ((4096, 512, 64, 2048, 16, 128), 65, 86),
       ((131072, 40, 64, 2048, 16, 128), 51, 64), ((65536, 512, 64, 2048, 16, 128), 344, 107),
       ((4096, 60, 4, 2048, 64, 128), 82, 214), ((16384, 512, 4, 2048, 16, 128), 871, 162),
       ((2000, 100, 4, 2048, 4, 128), 24.2, 29.4), ((2000, 100, 4, 2048, 16, 128), 27.5, 64.9),
       ((2000, 512, 4, 2048, 16, 128), 175, 71), ((0, 1024, 64, 2048, 4, 128), 4.5, 5.4),
       ((0, 2048, 4, 2048, 4, 128), 30.8, 7.0), ((0, 2200, 4, 2048, 16, 128), 86, 64),
       ((131072, 512, 64, 2048, 16, 128), 555, 142), ((32768, 1, 4, 2048, 4, 128), 11.7, 27)]


def test_block_selection(tmp_path):
    exe = str(tmp_path / "qsa_rule")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", CSRC, os.path.join(ROOT, "tests", "cxx", "qsa_rule.cpp"), "-o", exe], check=True)
    calls = "\n".join(" ".join(map(str, call)) for call, _, _ in QSA)
    r = subprocess.run([exe], input=calls, capture_output=True, text=True, check=True)
    took = [many if w == "1" else few for w, (_, few, many) in zip(r.stdout.split(), QSA)]
    assert len(took) == len(QSA)
    assert [(call, t) for t, (call, few, many) in zip(took, QSA) if t > 1.15 * min(few, many)] == []
