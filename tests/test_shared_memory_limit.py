"""The limit of dynamic shared memory is the runtime's for each kernel and device: it is raised on every device that a kernel is
launched on, from whatever thread."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "qwen-engine_amd" / "csrc"
PROGRAM = r"""
#include "shared_limit.h"
#include <cstdio>
#include <thread>
#include <vector>

// the runtime's two calls: which device a thread is on, and how often each device's limit was raised
static thread_local int on = 0;
static std::atomic<int> calls[128], fail{0};
extern "C" hipError_t hipGetDevice(int* d) { *d = on; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int bytes) {
    if (bytes != 70000) return hipErrorInvalidValue;
    if (fail) return hipErrorUnknown;
    calls[on]++;
    return hipSuccess;
}
#define EXPECT(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }

int main() {
    static std::atomic<unsigned long> raised{0};
    const auto launch = [&](int device) { on = device; return qe_raise_shared_limit((const void*)&raised, 70000, raised); };
    EXPECT(launch(0) == hipSuccess && launch(0) == hipSuccess && calls[0] == 1)
    EXPECT(launch(1) == hipSuccess && launch(1) == hipSuccess && calls[1] == 1 && calls[0] == 1)
    fail = 1;
    EXPECT(launch(2) == hipErrorUnknown)                                  // (told, and not taken for done)
    fail = 0;
    EXPECT(launch(2) == hipSuccess && calls[2] == 1)
    EXPECT(launch(63) == hipSuccess && launch(63) == hipSuccess && calls[63] == 1)
    EXPECT(launch(70) == hipSuccess && launch(70) == hipSuccess && calls[70] == 2 && launch(6) == hipSuccess && calls[6] == 1)
    std::vector<std::thread> threads;
    std::atomic<int> bad{0};
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&, t] {
            for (int d = 8; d < 40; ++d) if (launch(8 + (d + 5 * t) % 32) != hipSuccess || calls[on] < 1) bad++;
        });
    for (auto& t : threads) t.join();
    EXPECT(bad == 0)
    for (int d = 8; d < 40; ++d) EXPECT(calls[d] >= 1 && launch(d) == hipSuccess && calls[d] <= 8)
    return 0;
}
"""


def test_limit_is_raised_on_every_device(tmp_path):
    cxx = shutil.which("g++")
    headers = next((p for p in ("/opt/rocm/include",) if (Path(p) / "hip" / "hip_runtime_api.h").exists()), None)
    if not cxx or not headers:
        pytest.skip("no host compiler or no HIP headers")
    src = tmp_path / "limit.cpp"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", f"-I{headers}", str(src), "-o",
                    str(tmp_path / "limit")], check=True)
    got = subprocess.run([str(tmp_path / "limit")], capture_output=True, text=True, timeout=60)
    assert got.returncode == 0, got.stdout


def test_no_launch_keeps_a_flag_of_its_own():
    """Launches that raise the limit once do it by the function that knows the devices; the others do it each time."""
    for path in sorted(CSRC.glob("*.hip")):
        assert not re.search(r"static (bool|unsigned long|size_t|int) \w+ = ", path.read_text()), path.name
