"""The panels' scratch layout (host side, no device): a level of many fronts, beyond 2^31 entries in all, has offsets
that the 32-bit task fields hold and fronts that do not overlap; beyond the given limit the level is told to do
without."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparsedirectsolver.jl_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "panel_plan.h"
int main() {
    std::vector<int64_t> entries;
    for (int q = 0; q < 3000000; ++q) entries.push_back(900 + q % 777);
    std::vector<int32_t> off;
    int64_t total = 0, end = 0;
    if (!sds::panel_offsets(entries, INT64_MAX, off, total)) return 1;
    if (total <= ((int64_t)1 << 31) || off.size() != entries.size()) return 2;
    for (size_t q = 0; q < off.size(); ++q) {
        const int64_t at = (int64_t)off[q] * sds::PANEL_SCR_UNIT;
        if (at < end) return 3;
        end = at + entries[q];
    }
    if (end > total) return 4;
    if (!sds::panel_offsets(entries, total, off, total)) return 5;
    if (sds::panel_offsets(entries, total - 1, off, total)) return 6;
    if (!sds::panel_offsets({}, 0, off, total) || total != 0) return 7;
    // the most that 32 bits hold: the last front may reach past it, the next one is refused
    const int64_t unit = (int64_t)INT32_MAX * sds::PANEL_SCR_UNIT;
    if (!sds::panel_offsets({unit, 5}, INT64_MAX, off, total) || off[1] != INT32_MAX) return 8;
    if (sds::panel_offsets({unit, 5, 5}, INT64_MAX, off, total)) return 9;
    return 0;
}
"""


def test_panel_scratch_offsets(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
