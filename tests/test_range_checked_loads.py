"""The projection kernels' loads stay within their operands by the buffer resources' range check, which covers the
per-lane offset only: no load may keep a part of its offset in the scalar operand, and the per-lane offsets of partial
tiles have to fall on the right side of the resources' ends."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "qwen3-local-test_amd", "csrc")


def _arguments(text, at):
    """The argument texts of the call whose opening bracket is at text[at]."""
    args, depth, start = [], 0, at + 1
    for i in range(at, len(text)):
        depth += text[i] in "([{"
        depth -= text[i] in ")]}"
        if (depth == 1 and text[i] == ",") or depth == 0:
            args.append(text[start:i].strip())
            start = i + 1
        if depth == 0:
            return args


def test_whole_offset_is_checked():
    text = re.sub(r"//.*", "", open(os.path.join(CSRC, "mat.hip")).read())
    calls = [_arguments(text, m.end() - 1) for m in re.finditer(r"__builtin_amdgcn_raw_buffer_load_b\d+\(", text)]
    assert len(calls) >= 6
    assert [c for c in calls if c[2] != "0"] == []  # (resource, per-lane offset, scalar offset, cache bits)


def test_gemm_offsets(tmp_path):
    exe = str(tmp_path / "gemm_offsets")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", CSRC, os.path.join(ROOT, "tests", "cxx", "gemm_offsets.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
