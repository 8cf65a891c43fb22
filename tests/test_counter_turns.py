"""The turns in which persistent launches take their tile counters (neraulgraphics_amd/csrc/ngx_turns.h), without a GPU: a
model of the two sets is driven through frames that end well, that an error ends half launched, and that take no counters,
in every order, and each launch must find its set zero."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "ngx_turns.h"
using ngx::CounterTurns;
// kinds of frames: 0 ends well, 1 fails after one of its two launches, 2 fails before any, 3 takes no counters
int main() {
    int bad = 0, launches = 0;
    for (int order = 0; order < 4096; ++order) {
        CounterTurns turns;
        bool used[2] = {false, false};
        for (int f = 0, o = order; f < 6; ++f, o /= 4) {
            const int kind = o % 4;
            if (kind != 3 && turns.dirty) {
                used[0] = used[1] = false;
                turns.dirty = false;
            }
            CounterTurns::Frame frame(kind == 3 ? nullptr : &turns);
            for (int launch = 0; kind != 3 && launch < 2; ++launch) {
                if (kind == 2) break;
                const int now = turns.set, next = turns.set ^= 1;
                if (kind == 1 && launch == 1) break;  // the set is taken, and the launch that would zero the next fails
                bad += used[now];
                ++launches;
                used[now] = true;
                used[next] = false;
            }
            if (kind == 0 || kind == 3) frame.close();
        }
    }
    std::printf("%d launches, %d on counters that were not zero\n", launches, bad);
    return bad != 0;
}
"""


def test_every_launch_finds_its_counters_zero(tmp_path):
    src, exe = tmp_path / "turns.cpp", tmp_path / "turns"
    src.write_text(PROGRAM)
    build = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "neraulgraphics_amd", "csrc"),
                            str(src), "-o", str(exe)], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and "launches" in run.stdout, run.stdout
