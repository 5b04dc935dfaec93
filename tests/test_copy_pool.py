"""The threads that copy between a caller's arrays and the staging slots of the host-pointer path (accera_amd/csrc/copy_pool.h), built with the host
compiler and run on the CPU: the bytes are right from several callers at once, and the threads take no cores that they have no use for."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "accera_amd", "csrc")

PROGRAM = r'''
#include "copy_pool.h"
#include <cstdio>
#include <cstdlib>
#include <ctime>
#include <vector>
#include <sys/resource.h>
using namespace acc950;
static double cpu_ms() { timespec t; clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t); return t.tv_sec * 1e3 + t.tv_nsec * 1e-6; }
static void sleep_ms(int ms) { timespec t{ms / 1000, (ms % 1000) * 1000000L}; nanosleep(&t, nullptr); }
static bool good(CopyPool& pool, size_t bytes, size_t src_off, size_t dst_off, bool past)
{
    std::vector<unsigned char> a(bytes + 128), b(bytes + 128, 7);
    for (size_t i = 0; i < a.size(); ++i) a[i] = (unsigned char)(i * 2654435761u >> 13);
    pool.copy((char*)b.data() + dst_off, (char*)a.data() + src_off, bytes, past);
    for (size_t i = 0; i < dst_off; ++i) if (b[i] != 7) return false;
    for (size_t i = dst_off + bytes; i < b.size(); ++i) if (b[i] != 7) return false;
    return std::memcmp(b.data() + dst_off, a.data() + src_off, bytes) == 0;
}
int main(int argc, char** argv)
{
    CopyPool& pool = *new CopyPool;
    if (argc > 1) { // as many cores as the argument says
        cpu_set_t all, some;
        CPU_ZERO(&some);
        sched_getaffinity(0, sizeof all, &all);
        for (int i = 0, n = atoi(argv[1]); i < CPU_SETSIZE && n; ++i) if (CPU_ISSET(i, &all)) { CPU_SET(i, &some); --n; }
        sched_setaffinity(0, sizeof some, &some);
    }
    // bytes: sizes around the limits of the copy in pieces, every alignment of either side, several callers at once
    std::atomic<int> bad{0};
    std::vector<std::thread> callers;
    for (int t = 0; t < 3; ++t) callers.emplace_back([&, t] {
        CopyPool::Busy large(pool, t != 1);
        const size_t sizes[] = {1, 4095, 4096, 262143, 262144, 262145, 300001, 1048576 + 33, 5 * 1048576 + 7};
        for (size_t i = 0; i < sizeof sizes / sizeof *sizes; ++i) if (!good(pool, sizes[i], (i * 5 + t) % 64, (i * 11 + 3 * t) % 64, (i + t) % 2)) ++bad;
    });
    for (auto& c : callers) c.join();
    // a large call with a long pause between its copies, and the time after it
    double in_pause, after;
    {
        CopyPool::Busy large(pool, true);
        if (!good(pool, 4 << 20, 0, 0, true)) ++bad;
        const double t0 = cpu_ms();
        sleep_ms(400);
        in_pause = cpu_ms() - t0;
        if (!good(pool, 4 << 20, 1, 2, false)) ++bad; // (the threads are asleep: this copy wakes them)
    }
    const double t0 = cpu_ms();
    sleep_ms(200);
    after = cpu_ms() - t0;
    printf("bad %d threads %d in_pause %.1f after %.1f\n", bad.load(), pool.started(), in_pause, after);
    return bad ? 1 : 0;
}
'''


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    where = tmp_path_factory.mktemp("copy_pool")
    (where / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", CSRC, str(where / "t.cpp"), "-o", str(where / "t")], check=True)
    return str(where / "t")


@pytest.mark.parametrize("cores", [None, 1, 2, 4])
def test_copies_are_right_and_waiting_costs_no_cores(program, cores):
    """A pause of 400 ms inside a large call: threads that waited awake would take 400 ms each; ours look for 150 us and sleep."""
    have = len(os.sched_getaffinity(0))
    if cores and cores > have:
        pytest.skip("fewer cores here")
    out = subprocess.run([program] + ([str(cores)] if cores else []), check=True, capture_output=True, text=True, timeout=60).stdout
    bad, threads, in_pause, after = re.fullmatch(r"bad (\d+) threads (\d+) in_pause ([\d.]+) after ([\d.]+)\n", out).groups()
    assert int(bad) == 0
    assert int(threads) == min(6, (cores or have) - 1)     # one core is the caller's
    assert float(in_pause) < 40 and float(after) < 20, out  # (six threads' 150 us, and what the program itself takes)
