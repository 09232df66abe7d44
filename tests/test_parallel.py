"""The host set-up's threads (memphys_amd/csrc/parallel.hpp): an exception on any of
them, a failed allocation for instance, reaches the caller, whose C entry turns
it into a status; without it the process would end.  So do ranges for which no
thread can be started."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "memphys_amd",
                    "csrc")
MAIN = r"""
#include "parallel.hpp"
#include <sys/resource.h>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>

int main(int argc, char** argv) {
    const std::string what = argv[1];
    const int n = 5000;
    std::vector<int> seen(n, 0);
    if (what == "throw") {  // one index throws: first, middle and last range
        for (int bad : {0, 2500, n - 1}) {
            std::atomic<int> calls{0};
            bool caught = false;
            try {
                mp::parallel_for(n, [&](int i) {
                    ++calls;
                    if (i == bad) throw std::bad_alloc();
                });
            } catch (const std::bad_alloc&) {
                caught = true;
            }
            if (!caught || calls > n) return 1;
        }
    } else if (what == "throw_all") {
        try {
            mp::parallel_ranges(n, 7, [&](int, int, int q) { throw q; });
            return 1;
        } catch (int q) {
            if (q < 0 || q > 6) return 1;
        }
    } else {
        if (what == "no_threads") {  // no room for a thread's stack
            rlimit r;
            getrlimit(RLIMIT_AS, &r);
            long pages = 0;
            if (FILE* f = fopen("/proc/self/statm", "r")) {
                if (fscanf(f, "%ld", &pages) != 1) return 2;
                fclose(f);
            }
            r.rlim_cur = (rlim_t)pages * 4096 + (4 << 20);
            if (setrlimit(RLIMIT_AS, &r)) return 2;
        }
        for (int t : {1, 3, 16}) {
            seen.assign(n, 0);
            mp::parallel_ranges(n, t, [&](int i0, int i1, int) {
                for (int i = i0; i < i1; ++i) ++seen[i];
            });
            for (int i = 0; i < n; ++i)
                if (seen[i] != 1) return 1;
        }
        seen.assign(n, 0);
        mp::parallel_for(n, [&](int i) { ++seen[i]; });
        for (int i = 0; i < n; ++i)
            if (seen[i] != 1) return 1;
        mp::parallel_for(0, [&](int) { exit(1); });
    }
    puts("ok");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("parallel")
    src = d / "main.cpp"
    src.write_text(MAIN)
    exe = d / "main"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe),
                    "-lpthread"], check=True)
    return str(exe)


@pytest.mark.parametrize("what", ["cover", "throw", "throw_all", "no_threads"])
def test_parallel_ranges(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
