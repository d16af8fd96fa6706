"""What is set once per device (the kernels' dynamic LDS limits): done again
for another device, not remembered when it failed, and complete before any
thread goes on."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pascal_tcs_amd", "csrc")
PROGRAM = r"""
#include "device_once.h"
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    using namespace tcs;
    DeviceSet d;
    int n = 0;
    auto ok = [&] { n++; return 0; };
    auto bad = [&] { n++; return -3; };
    CHECK(once_per_device(d, 0, bad) == -3 && n == 1);  // a failure is not remembered
    CHECK(once_per_device(d, 0, ok) == 0 && n == 2);
    CHECK(once_per_device(d, 0, bad) == 0 && n == 2);   // done
    for (int dev : {1, 7, 63}) {                         // every device has its own
        const int before = n;
        CHECK(once_per_device(d, dev, ok) == 0 && n == before + 1);
        CHECK(once_per_device(d, dev, ok) == 0 && n == before + 1);
    }
    for (int dev : {64, 200, -1}) {                      // not remembered: done each time
        const int before = n;
        CHECK(once_per_device(d, dev, ok) == 0 && once_per_device(d, dev, ok) == 0 && n == before + 2);
    }
    DeviceSet e;                                         // and every set of its own
    CHECK(once_per_device(e, 0, ok) == 0);
    for (int round = 0; round < 50; round++) {
        DeviceSet t;
        std::atomic<int> done{0}, early{0};
        std::vector<std::thread> threads;
        for (int q = 0; q < 8; q++)
            threads.emplace_back([&] {
                once_per_device(t, 5, [&] {
                    std::this_thread::sleep_for(std::chrono::microseconds(200));
                    done++;
                    return 0;
                });
                if (done == 0) early++;
            });
        for (auto &x : threads) x.join();
        CHECK(early == 0);
    }
    puts("ok");
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_once_per_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def test_no_kernel_attribute_is_set_behind_a_flag_of_the_process():
    """Every attribute goes through the one function that knows the device."""
    found = []
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as f:
            found += [name for line in f if "hipFuncSetAttribute(" in line]
    assert found == ["runtime.hip"], found
