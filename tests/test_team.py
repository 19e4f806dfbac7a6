"""The host threads that take large results over (csrc/sev_team.hpp), compiled
by itself: every element is taken once however many of the wanted threads can be
started, none included, and a team that is given up early ends.  CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "sev_team.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <system_error>

static int allowed;

// std::thread, of which only `allowed` can be started
struct Few {
    std::thread t;
    template <class F>
    explicit Few(F f) {
        if (allowed-- <= 0)
            throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
        t = std::thread(f);
    }
    Few(Few &&) = default;
    void join() { t.join(); }
};

int main(int, char **argv) {
    const int want = std::atoi(argv[1]), can = std::atoi(argv[2]), chunks = std::atoi(argv[3]);
    const int per = 101;
    std::vector<std::atomic<int>> taken((size_t)(chunks * per));
    for (int given_up = 0; given_up < 2; ++given_up) {
        for (auto &x : taken) x = 0;
        allowed = can;
        const int upto = given_up ? chunks / 2 : chunks;
        {
            sev::ChunkTeam<Few> team(want, chunks, [&](int64_t c, int t, int nt) {
                for (int i = per * t / nt; i < per * (t + 1) / nt; ++i) taken[(size_t)(c * per + i)]++;
            });
            if (team.size() != (can < want ? can : want)) return 1;
            for (int c = 0; c < upto; ++c) {
                team.publish(c);
                if (c > 0) team.wait(c - 1);
            }
            if (upto) team.wait(upto - 1);
        }
        for (int i = 0; i < chunks * per; ++i)
            if (taken[(size_t)i] != (i < upto * per ? 1 : 0)) return 2;
    }
    std::puts("ok");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("team")
    src, out = d / "team.cpp", d / "team"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "severo.jl_amd", "csrc"), str(src), "-o", str(out)],
                   check=True)
    return str(out)


@pytest.mark.parametrize("want,can", [(8, 8), (8, 3), (8, 1), (8, 0), (1, 1)])
@pytest.mark.parametrize("chunks", [1, 2, 50])
def test_every_element_is_taken_once(program, want, can, chunks):
    r = subprocess.run([program, str(want), str(can), str(chunks)], capture_output=True,
                       text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n"
