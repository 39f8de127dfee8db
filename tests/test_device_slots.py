"""The per-device turns of the open-boundary sum (csrc/device_slots.hpp), on the host: callers on one device exclude
each other, callers on different devices do not wait for each other."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "device_slots.hpp"
#include <cstdio>
#include <thread>
int main()
{
    chmc::DeviceSlots<int, 4> slots;
    if (slots.of(-1) || slots.of(4) || !slots.of(0) || slots.of(0)->value != 0) return 1;
    std::lock_guard<std::mutex> lk(slots.of(1)->mu);             // a caller in its turn on device 1
    bool other[4] = {};
    for (int d = 0; d < 4; d++)
        std::thread([&] { if (slots.of(d)->mu.try_lock()) { other[d] = true; slots.of(d)->mu.unlock(); } }).join();
    return other[0] && !other[1] && other[2] && other[3] ? 0 : 2;
}
"""


def test_turns_are_per_device(tmp_path):
    (tmp_path / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "chemhmc_amd", "csrc"),
                    str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    assert subprocess.run([str(tmp_path / "t")], timeout=60).returncode == 0


def test_open_sum_takes_its_turn_on_its_device():
    # the only lock held over a call of the sum is the current device's; the lookup's ends with the lookup
    src = open(os.path.join(ROOT, "chemhmc_amd", "csrc", "capi.hip")).read()
    call = src[src.index('extern "C" int chmc_potential_energy_open('):]
    call = call[:call.index("\n}\n")]
    assert re.findall(r"lock_guard<std::mutex> \w+\((.*?)\)", call) == ["*turn"]
    lookup = src[src.index("static hipError_t open_memory("):]
    assert "*turn = &slot->mu" in lookup[:lookup.index("\n}\n")]
