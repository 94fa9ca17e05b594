"""The rule by which a launch of a CG loop passes a scene over (sofa_amd/csrc/stop_mark.h), compiled on the CPU: the
waves of a launch decide alike whether or not they see the stop that this launch itself records, and every
later launch sees it."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sofa_amd", "csrc")

PROGRAM = r"""
#include "stop_mark.h"
#include <cstdio>
using namespace sofa_amd;
int main() {
    for (int it = 1; it <= 3000; it++)
        for (int phase = 0; phase < 2; phase++) {
            const int own = stop_mark(it, phase);
            if (own == 0 || stopped_before(0, own) || stopped_before(own, own)) return std::printf("own launch %d %d\n", it, phase), 1;
            if (!stopped_before(1, own)) return std::printf("before the loop: %d %d\n", it, phase), 1;
            for (int k = 1; k <= it; k++)
                for (int f = 0; f < 2; f++)
                    if (stop_mark(k, f) < own && !stopped_before(stop_mark(k, f), own))
                        return std::printf("%d %d after %d %d\n", it, phase, k, f), 1;
            if (!stopped_before(own, 0)) return std::printf("recording nothing: %d %d\n", it, phase), 1;
        }
    return stopped_before(0, 0) ? 1 : 0;
}
"""


def test_a_launch_passes_over_its_own_stop(tmp_path):
    src = tmp_path / "marks.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "marks"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)])
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
