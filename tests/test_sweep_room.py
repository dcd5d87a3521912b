"""The room that solves at once share (sweep_room.h), on host threads: never
more compute units inside than the device has, a solve larger than the device
alone, arrivals served in order, and every thread ends."""
import os
import subprocess

from conftest import ROOT

SOURCE = r"""
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
#include "sweep_room.h"
int main() {
    astg::SweepRoom room;
    const int cap = 256, wants[] = {1, 27, 100, 180, 252, 256, 300, 0};
    std::atomic<int> inside{0}, holders{0}, bad{0}, turns{0};
    std::vector<std::thread> t;
    for (int k = 0; k < 8; ++k)
        t.emplace_back([&, k] {
            for (int i = 0; i < 2000; ++i) {
                const astg::SweepLease lease(room, wants[k], cap);
                const int in = inside.fetch_add(wants[k]) + wants[k], h = holders.fetch_add(wants[k] > 0) + (wants[k] > 0);
                if (in > cap && h > 1) ++bad;
                ++turns;
                if (i % 64 == 0) std::this_thread::yield();
                inside -= wants[k];
                holders -= wants[k] > 0;
            }
        });
    for (auto& x : t) x.join();
    std::printf("%d turns, %d over the device\n", turns.load(), bad.load());
    return bad || turns != 16000;
}
"""


def test_room_is_never_overdrawn(tmp_path):
    src, exe = tmp_path / "room.cpp", tmp_path / "room"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I" + os.path.join(ROOT, "ast-grid_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(p.stdout)
    assert p.returncode == 0, p.stdout
