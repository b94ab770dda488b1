"""Line indexes of the reverse volume kernel, evaluated on the host at compile
time over every block, grid and lane column of a workgroup, idle ones among
them: blocks of the grid meet their own lines, the rest stay inside the face
buffer."""
import os
import subprocess

import pytest

from dsem_amd import build as B

SOURCE = """
#include "dsem_hip.hip"

namespace {
template <int P>
constexpr bool lines_in_range()
{
    using S = Sz<P>;
    using V = Vol<P>;
    constexpr int BLK = AdjVol<P>::BLK, NFV = NEQ * S::NF;
    for (int bk = 0; bk < Passes<P, BLK>::N * (BLK / 16); ++bk)
        for (int D = 0; D < 3; ++D)
            for (int c4 = 0; c4 < 4; ++c4) {
                const int line = grid_line<P>(bk, D, c4), own = (bk - D * V::NG) * 4 + c4;
                // last field of the high face, the largest offset that meets the line
                if (line < 0 || D * 2 * NFV + NFV + 4 * S::NF + line >= 6 * NFV) return false;
                if (own >= 0 && own < V::NL && line != own) return false;
            }
    return true;
}
static_assert(lines_in_range<5>() && lines_in_range<6>(), "p = 5, 6");
static_assert(lines_in_range<7>(), "p = 7");
static_assert(lines_in_range<8>(), "p = 8");
}
"""


def test_reverse_volume_lines_stay_in_their_buffers(tmp_path):
    try:
        hipcc = B.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    src = tmp_path / "lines.hip"
    src.write_text(SOURCE)
    out = subprocess.run([hipcc, "-fsyntax-only", "--cuda-host-only", f"--offload-arch={B.ARCH}", "-std=c++17", "-w",
                          "-I", B.CSRC, "-I", os.path.join(B.ROOT, "include"), str(src)],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
