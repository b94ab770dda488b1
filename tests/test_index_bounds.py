"""Index functions of the volume kernels, evaluated on the host at compile time
over everything a workgroup can ask of them.

Lines of the reverse kernel, over every block, grid and lane column, idle ones
among them: blocks of the grid meet their own lines, the rest stay inside the
face buffer.

Face averages of the mixed-precision kernel, over every row of a line: a face
row loads its own face's, an interior row never those of a face whose place is
written in the same pass."""
import os
import subprocess

import pytest

from dsem_amd import build as B

LINES = """
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


AVERAGES = """
#include "dsem_hip.hip"

namespace {
template <int P, int D>
constexpr bool averages_apart()
{
    constexpr int lo = face_of<P>(D, 0), hi = face_of<P>(D, Sz<P>::NC - 1);
    if (average_face<P, D>(0) != lo || average_face<P, D>(Sz<P>::NC - 1) != hi) return false;
    for (int j = 1; j < Sz<P>::NC - 1; ++j) {
        const int f = average_face<P, D>(j);
        if (f < 1 || f > 6 || f == lo || f == hi) return false;
    }
    return true;
}
template <int P>
constexpr bool all_grids() { return averages_apart<P, 0>() && averages_apart<P, 1>() && averages_apart<P, 2>(); }
static_assert(all_grids<1>() && all_grids<2>() && all_grids<3>() && all_grids<4>(), "p = 1 to 4");
static_assert(all_grids<5>() && all_grids<6>() && all_grids<7>() && all_grids<8>(), "p = 5 to 8");
}
"""


def _compiles(tmp_path, source):
    try:
        hipcc = B.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    src = tmp_path / "check.hip"
    src.write_text(source)
    out = subprocess.run([hipcc, "-fsyntax-only", "--cuda-host-only", f"--offload-arch={B.ARCH}", "-std=c++17", "-w",
                          "-I", B.CSRC, "-I", os.path.join(B.ROOT, "include"), str(src)],
                         capture_output=True, text=True)
    assert out.returncode == 0, out.stderr


def test_reverse_volume_lines_stay_in_their_buffers(tmp_path):
    _compiles(tmp_path, LINES)


def test_mixed_volume_interior_rows_leave_the_written_faces_alone(tmp_path):
    _compiles(tmp_path, AVERAGES)
