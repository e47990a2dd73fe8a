"""The order of the token groups of the row-parallel kernels and the XCDs' shares of it, compiled for the CPU: every group has one place, and no XCD is handed
many more groups than another."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include "group_order.h"
#include <algorithm>
#include <cstdio>
#include <set>
#include <tuple>
using namespace order;
int main() {
    const int sizes[] = {1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 35, 36, 50, 63, 64, 65, 69, 82, 85, 113, 127, 128, 130, 255, 256, 257, 300, 511, 513, 1024, 2001, 4095, 4097};
    for (int batch : {1, 2, 3, 5, 7, 20, 50, 128}) for (int heads : {1, 2, 3, 4, 5, 8}) for (int groups : sizes) for (bool in_parts : {false, true}) {
        if (batch * heads * groups > 20000) continue;
        const GroupOrder o = group_order(batch, heads, groups, in_parts);
        const int total = static_cast<int>(o.places()), round = 8 << o.share_log2, grid = (total + round - 1) / round * round;
        std::set<std::tuple<int, int, int>> seen;
        int held[8] = {};
        bool once = true;
        for (int id = 0; id < grid; ++id) {
            const int place = place_from_end(o, id & 7, id >> 3);
            int grp, h, b;
            if (place >= total || !group_at(o, total - 1 - place, grp, h, b)) continue;
            once = once && grp >= 0 && grp < groups && h >= 0 && h < heads && b >= 0 && b < batch && seen.insert({grp, h, b}).second;
            ++held[id & 7];
        }
        std::printf("%d %d %d %d %d %d %d\n", batch, heads, groups, in_parts, once && static_cast<int>(seen.size()) == batch * heads * groups,
                    *std::max_element(held, held + 8), total);
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_one_place_each_and_even_shares(tmp_path):
    (tmp_path / "order.cpp").write_text(PROGRAM)
    program = str(tmp_path / "order")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__device__=", "-D__forceinline__=inline", "-DIV2_NS=order", "-I", os.path.join(ROOT, "infllmv2_cuda_impl_amd", "csrc"),
                    str(tmp_path / "order.cpp"), "-o", program], check=True)
    lines = [[int(x) for x in line.split()] for line in subprocess.run([program], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(lines) > 300
    for batch, heads, groups, in_parts, once, most, places in lines:
        case, all_groups = (batch, heads, groups, in_parts), batch * heads * groups
        assert once, case
        if in_parts:
            continue
        if all_groups <= 256:                                  # a group to each CU: 32 to an XCD
            assert most <= 32, case
        share = 16 if all_groups <= 256 or all_groups > 4096 else 4 if all_groups <= 2048 else 8
        # a share more than its part of the places, of which those at a head's last chunk may be nobody's
        assert most <= places / 8 + share and (places <= 256 or places <= 1.12 * all_groups), case
