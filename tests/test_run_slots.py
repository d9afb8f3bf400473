"""Slots of Widom runs near the largest insertion count (2^32 - 1).

The kernels walk the insertions of a bin, or of a group of bins, a workgroup or a
round at a time and compare each slot with the run's end.  The walk is compiled
here for the host: it must end and visit each slot of the run once, also where
the slots past the end exceed 32 bits.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "er_common.h"
#include <cstdio>
using namespace er;

// slots of [begin, end) that lane `tid` of a walk by `step` visits, first to last
static bool walk(uint32_t begin, uint32_t end, uint32_t step) {
    uint64_t seen = 0;
    for (uint32_t tid = 0; tid < step; ++tid) {
        long rounds = 0;
        for (uint64_t e = run_slot(begin, tid); e < end; e += step) {
            if (e < begin || ++rounds > 1000) return false;
            ++seen;
        }
    }
    return seen == (uint64_t)end - begin;
}

int main() {
    const uint32_t last = 0xffffffffu;
    // a workgroup's loop over a group, and a wave's rounds of 512 over a bin
    for (uint32_t step : {(uint32_t)kBinWG, 512u})
        for (uint32_t length : {0u, 1u, 63u, 511u, 512u, 1023u, 1024u, 20479u, 20481u, 70000u})
            for (uint32_t gap : {0u, 1u, 500u, 1023u, 1024u, 20480u, 100000u})
                if (!walk(last - gap - length, last - gap, step)) {
                    std::printf("step %u length %u gap %u\n", step, length, gap);
                    return 1;
                }
    // the slots a thread of the second binning step keeps in registers
    for (int q = 0; q < 20; ++q)
        for (uint32_t tid = 0; tid < (uint32_t)kBinWG; ++tid)
            if ((run_slot(last - 300, q * kBinWG + tid) < last) != (q == 0 && tid < 300)) return 2;
    return 0;
}
"""


def test_slots_do_not_wrap(tmp_path):
    src, exe = tmp_path / "slots.cpp", tmp_path / "slots"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "emptyroom_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
