"""Which calls the matrix-core gate and gate + up kernels take, asked of the built library's own rule by a host program.  Needs no GPU."""
import subprocess

import pytest

from cats_amd.build import CSRC, HIPCC, KERNEL_LIB, ROOT

SOURCE = r"""
#include <cstdio>
#include <cstring>
#include "cats_launch.h"
using namespace cats;
template <class DT>
static void ask(const char* dtype) {
  for (int rows : {4, 7, 12})
    for (int up = 0; up < 2; up++)
      for (int norm = 0; norm < 2; norm++) {
        RowsArgs a;
        memset(&a, 0, sizeof(a));
        a.K = 1024; a.N = 3000; a.nb = rows; a.row_vecs = a.K / DT::VEC; a.nch = (a.row_vecs + kWave - 1) / kWave; a.mma = 1;
        a.x = a.w = (const u32x4*)4096;
        if (up) a.w2 = a.w;
        if (norm) a.norm_w = a.w;
        const bool takes = rows > 8 ? rows_mma16_supported<DT>(a) : rows_takes_mma<DT>(up ? kGateUp : kGate, rows > 4 ? 8 : 4, a);
        printf("%s %d %d %d %d\n", dtype, rows, up, norm, (int)takes);
      }
}
int main() { ask<F16>("F16"); ask<BF16>("BF16"); ask<F32>("F32"); }
"""


@pytest.fixture(scope="module")
def answers(tmp_path_factory):
    if not KERNEL_LIB.exists():
        import __graft_entry__

        __graft_entry__.build()
    d = tmp_path_factory.mktemp("rules")
    (d / "ask.hip").write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", f"-I{ROOT / 'include'}", f"-I{CSRC}", str(d / "ask.hip"), "-o", str(d / "ask"),
                    f"-L{KERNEL_LIB.parent}", "-lcats_gemv", f"-Wl,-rpath,{KERNEL_LIB.parent}"], check=True, capture_output=True)
    lines = subprocess.run([str(d / "ask")], check=True, capture_output=True, text=True).stdout.split("\n")
    return {(f[0], int(f[1]), int(f[2]), int(f[3])): int(f[4]) for f in (line.split() for line in lines if line)}


def test_gate_pass_alone_is_not_given_a_norm(answers):
    """The matrix-core gate pass has no norm: a call with one is left to the kernels that apply it.  Without, and gate + up, as ever."""
    assert len(answers) == 36
    for (dtype, rows, up, norm), takes in answers.items():
        fp32_pair = dtype == "F32" and rows == 4  # the wave-per-row kernel's
        assert takes == int(not fp32_pair and (up or not norm)), (dtype, rows, up, norm)
