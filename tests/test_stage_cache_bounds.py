"""The decode's scalar stage path reads the page cache only at entries that exist
(CPU): full_stage_in_cache (dvattention_amd/csrc/dv_stream.h), compiled for the
host, against the definition, for positions below 0, at both ends of the cache and
at the ends of the 32-bit range.  Fragment lengths are device data, so no host
check keeps such positions from the kernel."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dvattention_amd", "csrc")
KPC = 512  # entries of a wave's page cache

MAIN = r"""
#include <stdio.h>
#include "dv_stream.h"
int main(int, char**) {
    static_assert(dv::stream::kPc == %d, "entries");
    int pos, shift, lp0;
    while (scanf("%%d %%d %%d", &pos, &shift, &lp0) == 3) printf("%%d\n", (int)dv::stream::full_stage_in_cache(pos, shift, lp0));
}
""" % KPC


def expected(pos, shift, lp0):
    pages = [(pos >> shift) - lp0, ((pos + 16) >> shift) - lp0]
    return int(pos >= 0 and pos % 16 == 0 and all(0 <= i < KPC for i in pages))


def test_full_stage_in_cache(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "bounds.cpp", tmp_path / "bounds"
    src.write_text(MAIN)
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    cases = []
    for shift in (4, 5, 7, 20):
        for lp0 in (0, 3, 1000):
            first = lp0 << shift
            for page in (-1, 0, 1, KPC - 2, KPC - 1, KPC):
                cases += [(first + (page << shift) + o, shift, lp0) for o in (0, 1, 8, 16, (1 << shift) - 16)]
            cases += [(p, shift, lp0) for p in (-16, -32, -64, -1 << 20, -1 << 31, (1 << 31) - 16, (1 << 31) - 32)]
    cases = [c for c in cases if -1 << 31 <= c[0] < 1 << 31]
    out = subprocess.run([str(exe)], input="\n".join("%d %d %d" % c for c in cases), capture_output=True, text=True,
                         check=True).stdout.split()
    assert [int(x) for x in out] == [expected(*c) for c in cases]
