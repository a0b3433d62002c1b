"""Tile ids of the work queues, on the host: whatever the tiles, the CUs and the cap, every tile is handed out once."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "open-instruct_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "oi_queue.h"
// A launch of `workgroups` over `items`: the ids that they begin with, then every queue drawn until it is empty.
static bool once(uint32_t workgroups, uint32_t items, bool begins) {
    const uint32_t locals = locals_for_items(items);
    std::vector<int> taken(items, 0);
    auto hand_out = [&](uint32_t pid) {
        const uint32_t item = item_of_pid(pid, items);
        if (item < items) ++taken[item];
    };
    if (begins)
        for (uint32_t b = 0; b < workgroups; ++b) hand_out(b);
    for (uint32_t q = 0; q < 8; ++q)
        for (uint32_t local = begins ? ids_begun(workgroups) : 0; local < locals; ++local) hand_out(local * 8 + q);
    for (uint32_t i = 0; i < items; ++i)
        if (taken[i] != 1) {
            printf("%u workgroups, %u items, begins %d: item %u taken %d times\n", workgroups, items, (int)begins, i, taken[i]);
            return false;
        }
    return true;
}
int main() {
    for (uint32_t items = 0; items <= 1100; items = items < 300 ? items + 1 : items + 37)
        for (uint32_t cus = 1; cus <= 310; cus = cus < 40 || cus >= 240 ? cus + 1 : cus + 24)
            for (uint32_t per_xcd : {0u, 1u, 4u, 64u}) {
                const uint32_t workgroups = resident_workgroups(items, cus, per_xcd);
                if ((workgroups == 0) != (items == 0) || (per_xcd && workgroups > per_xcd * 8)) return 2;
                if (!once(workgroups, items, true) || !once(workgroups, items, false)) return 1;
            }
    return 0;
}
"""


def test_every_tile_is_handed_out_once(tmp_path):
    source, program = tmp_path / "ids.cpp", tmp_path / "ids"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(source), "-o", str(program)], check=True)
    res = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
