"""The threads behind the library's large host copies (CopyPool), compiled alone for the CPU.

Copies of every size and alignment arrive whole and touch nothing beside them, with no helper, one
and several; faulting pages in leaves their contents; and helpers that get no CPU of their own hold
nobody up: three pools of five on one CPU, called in turn, take a few times what the same copies take
one thread (without the owner's share of the work and with unlimited spinning, each job waited out
time slices of the scheduler: about 60 times)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "sh_copypool.hpp"
#include <sched.h>
#include <stdio.h>
#include <stdlib.h>
using clk = std::chrono::steady_clock;
static double ms_since(clk::time_point t) { return std::chrono::duration<double, std::milli>(clk::now() - t).count(); }

static bool whole(int helpers) {
    sh::CopyPool pool(helpers);
    const size_t sizes[] = {0, 1, 4095, 131072, 131073, 1000003, 2u << 20, (9u << 20) + 5};
    std::vector<uint8_t> src((9u << 20) + 64), dst(src.size());
    for (size_t i = 0; i < src.size(); i++) src[i] = (uint8_t)(i * 2654435761u >> 13);
    for (int round = 0; round < 20; round++)
        for (size_t n : sizes)
            for (size_t off : {(size_t)0, (size_t)7}) {
                memset(dst.data(), 0xa5, n + 32);
                pool.start(dst.data() + off, src.data() + 3 * off, n);
                if (round % 2) pool.finish();
                if (round % 4 == 0) {   // the next job finishes this one; its pages keep what they hold
                    pool.start(dst.data() + off, nullptr, n);
                }
                pool.finish();
                if (memcmp(dst.data() + off, src.data() + 3 * off, n)) return false;
                for (size_t i = 0; i < off; i++) if (dst[i] != 0xa5) return false;
                for (size_t i = off + n; i < n + 32; i++) if (dst[i] != 0xa5) return false;
            }
    return true;
}

int main(int argc, char **argv) {
    if (argc > 1) {
        printf("%d\n", whole(atoi(argv[1])));
        return 0;
    }
    cpu_set_t one;
    sched_getaffinity(0, sizeof(one), &one);
    int cpu = 0;
    while (!CPU_ISSET(cpu, &one)) cpu++;
    CPU_ZERO(&one);
    CPU_SET(cpu, &one);
    sched_setaffinity(0, sizeof(one), &one);   // helpers inherit it
    const size_t n = 1u << 20;
    const int jobs = 60;
    std::vector<uint8_t> src(n, 1), dst(n, 2);
    auto t = clk::now();
    for (int i = 0; i < jobs; i++) memcpy(dst.data(), src.data(), n), src[i]++;
    const double alone = ms_since(t);
    {
        sh::CopyPool a(5), b(5), c(5);
        t = clk::now();
        for (int i = 0; i < jobs; i++) {
            sh::CopyPool &p = i % 3 == 0 ? a : i % 3 == 1 ? b : c;
            p.start(dst.data(), src.data(), n);
            p.finish();
            src[i]++;
        }
    }
    printf("%.3f %.3f\n", alone / jobs, ms_since(t) / jobs);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("copypool")
    (d / "main.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-pthread",
                           "-I" + os.path.join(ROOT, "ane-training-experiments_amd", "csrc"),
                           str(d / "main.cpp"), "-o", str(d / "main")])
    return str(d / "main")


@pytest.mark.parametrize("helpers", [0, 1, 5])
def test_copies_arrive_whole(program, helpers):
    assert subprocess.check_output([program, str(helpers)], timeout=120).split() == [b"1"]


def test_helpers_without_cpu_hold_nobody_up(program):
    alone, pooled = (float(x) for x in subprocess.check_output([program], timeout=120).split())
    print(f"1 MiB: {alone:.3f} ms on one thread, {pooled:.3f} ms through pools on the same CPU")
    assert pooled <= 10 * alone + 1.0
