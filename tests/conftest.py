import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
TESTS = os.path.dirname(os.path.abspath(__file__))
if TESTS not in sys.path:
    sys.path.insert(0, TESTS)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built libqwattn.so")
    config.addinivalue_line("markers", "slow: long-running case")


@pytest.fixture(scope="session")
def oracle():
    import oracle as orc
    return orc.Oracle()


@pytest.fixture(scope="session")
def qw():
    import common
    return common.load_package()


@pytest.fixture(scope="session")
def walk(tmp_path_factory):
    """Walks prefill launches' partial regions with the kernel's own index functions (cxx/prefill_regions.cpp) and
    fails on any fault: walk([(heads, KV heads, pos, n, max_tokens, visible key tiles), ...], CUs) -> the launches
    of the split schedule, those whose query tiles differ in parts, the most parts."""
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    exe = str(tmp_path_factory.mktemp("cxx") / "prefill_regions")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(ROOT, "qwen3-local-test_amd", "csrc"),
                    os.path.join(TESTS, "cxx", "prefill_regions.cpp"), "-o", exe], check=True)

    def run(launches, n_cu=256):
        text = "\n".join(" ".join(map(str, [*call, len(see), *see])) for *call, see in launches)
        r = subprocess.run([exe, str(n_cu)], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.stdout[:2000] + r.stderr[:2000]
        w = r.stdout.split()
        assert int(w[1]) == len(launches)
        return {"split": int(w[3]), "mixed": int(w[5]), "worst": int(w[7])}

    return run
