"""CPU test of the plan's choice for waves whose rows all lie past N (all_rows:
they compute like the others; otherwise they only stage tiles).  It is internal
to a launch and leaves the results as they are, so a small program reads it
from fa::plan_split itself.

Only staging made D = 64 non-causal grids of 2.375 to 3 workgroups per CU up to
11 % slower: CUs whose workgroups ended early took two of the remaining ones."""
from __future__ import annotations

import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "flash-attention_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "fa_fwd_kernel.h"
int main(int, char** v) {  // heads seq_len head_dim causal bf16 compute_units
  fa::KernelArgs a{};
  a.batch = 1;
  a.heads = std::atoi(v[1]);
  a.seq_len = std::atoi(v[2]);
  a.head_dim = std::atoi(v[3]);
  a.causal = std::atoi(v[4]);
  a.bf16 = std::atoi(v[5]);
  a.split.all_rows = -1;
  fa::plan_split(a, std::atoi(v[6]), true, &a.split);
  std::printf("%d", a.split.all_rows);
}
"""


@pytest.fixture(scope="module")
def all_rows(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("plan")
    src, exe = str(tmp / "rows.cpp"), str(tmp / "rows")
    with open(src, "w") as f:
        f.write(PROGRAM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    proc = subprocess.run(
        ["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-I", os.path.join(rocm, "include"),
         "-I", CSRC, src, os.path.join(CSRC, "fa_plan.cpp"), "-o", exe],
        stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-3000:]
    return lambda *args: int(subprocess.check_output([exe, *map(str, args)]))


@pytest.mark.parametrize("H,N,D,causal,cus,want", [
    (48, 2016, 64, 0, 256, 1),    # 768 workgroups: the end of the range
    (48, 2017, 64, 0, 304, 1),    # 2.53 per CU
    (64, 1472, 64, 0, 256, 1),
    (87, 800, 64, 0, 256, 1),     # 609: the first above 2.375 per CU
    (76, 1000, 64, 0, 256, 0),    # 608
    (97, 1000, 64, 0, 256, 0),    # 776
    (96, 799, 64, 0, 256, 0),     # short rows
    (48, 2016, 128, 0, 256, 0),   # D = 128
    (48, 2016, 64, 1, 256, 0),    # causal
    (77, 2048, 64, 0, 256, 0),    # 8-wave workgroups
    (1, 100, 64, 0, 256, 0),
])
@pytest.mark.parametrize("bf16", [0, 1])
def test_grids_where_every_wave_computes(all_rows, H, N, D, causal, cus, want, bf16):
    assert all_rows(H, N, D, causal, bf16, cus) == want
