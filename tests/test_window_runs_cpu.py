"""The cut of a window's rows into runs (csrc/window_runs.h): the one that a search over every count of runs finds, without
looking at every count, since the host makes it in every call."""
import os
import subprocess

from singe_amd import build

CSRC = os.path.join(os.path.dirname(build.__file__), "csrc")

SEARCH = """
#include "window_runs.h"
#include <cstdio>
#include <initializer_list>
static uint64_t exhaustive(uint64_t steps, uint64_t pairs, uint64_t places) {
    uint64_t best = ~0ull, best_steps = steps;
    for (uint64_t runs = 1; runs <= steps && (runs - 1) * pairs <= 4 * places; ++runs) {
        const uint64_t run_steps = (steps + runs - 1) / runs;
        const uint64_t cost = (pairs * ((steps + run_steps - 1) / run_steps) + places - 1) / places * (run_steps + 1);
        if (cost < best) best = cost, best_steps = run_steps;
    }
    return best_steps;
}
int main() {
    for (uint64_t places : {1, 38, 256, 512})
        for (uint64_t pairs : {1, 2, 3, 7, 8, 28, 64, 300})
            for (uint64_t steps = 1; steps < 3000; steps += 1 + steps / 40)
                if (singe_hip::window_run_steps(steps, pairs, places) != exhaustive(steps, pairs, places)) {
                    std::printf("steps %llu pairs %llu places %llu\\n", (unsigned long long)steps, (unsigned long long)pairs, (unsigned long long)places);
                    return 1;
                }
}
"""
# (89 candidates take some 10000 operations, all 2048 of them twenty times as many)
BOUNDED = '#include "window_runs.h"\nconstexpr uint64_t steps = singe_hip::window_run_steps(2048, 1, 512);\nstatic_assert(steps != 0);\n'


def test_runs_are_those_that_an_exhaustive_search_finds(tmp_path):
    source, program = tmp_path / "search.cpp", tmp_path / "search"
    source.write_text(SEARCH)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(source), "-o", str(program)], check=True)
    found = subprocess.run([str(program)], capture_output=True, text=True)
    assert found.returncode == 0, found.stdout


def test_runs_are_found_without_looking_at_every_count(tmp_path):
    source = tmp_path / "bounded.cpp"
    source.write_text(BOUNDED)
    subprocess.run(["g++", "-std=c++17", "-fconstexpr-ops-limit=20000", "-I", CSRC, "-c", str(source), "-o", str(tmp_path / "bounded.o")], check=True)
