"""The check of a transform launch's jobs (spec_launch_ok in spectral.hpp), which
every launch passes before either kernel family sees it.  Compiled for the host."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

CASES = r"""
#include <cstdio>
#include <cstring>
#include "spectral.hpp"
using namespace mhd;
static double f[3];
// a launch as the step makes it: three jobs with an auxiliary line, one without
static SpecLaunch good(int f32)
{
    SpecLaunch L;
    memset((void*)&L, 0, sizeof L);
    L.mode = SM_DERIV2;
    L.njobs = 4;
    for (int q = 0; q < 3; ++q) {
        L.bf[q] = f;
        SpecJob& J = L.job[q];
        J.out[0] = J.out[1] = f;
        J.aux = q == 0 ? AUX_MAXW : AUX_PROD;
        J.ai = q;
        J.aj = 0;
        if (f32) J.out[2] = f;
        else if (q < 2) J.xin = f;
    }
    L.job[3].out[0] = f;
    return L;
}
int main()
{
    for (int f32 = 0; f32 < 2; ++f32) {
        auto say = [&](const char* n, const SpecLaunch& L) { printf("%s%d %d\n", n, f32, (int)spec_launch_ok(L, f32)); };
        SpecLaunch L = good(f32);
        say("good", L);
        L = good(f32); L.job[1].aj = L.job[1].ai; say("same", L);
        L = good(f32); L.job[1].ai = 3; say("ai", L);
        L = good(f32); L.job[1].aj = -1; say("aj", L);
        L = good(f32); L.job[1].aux = 3; say("op", L);
        L = good(f32); L.bf[2] = nullptr; say("field", L);
        L = good(f32); L.job[2].out[1] = nullptr; say("out", L);
        L = good(f32); L.job[4] = L.job[2]; L.njobs = 5; say("order", L);
        L = good(f32); L.mode = SM_DERIV1; say("mode", L);
        L = good(f32); L.njobs = SPEC_MAX_JOBS + 1; say("count", L);
        L = good(f32); L.job[0].out[2] = nullptr; say("third", L);
        L = good(f32); L.job[0].xin = f; say("term", L);
        memset((void*)&L, 0, sizeof L);
        L.mode = SM_HC2R; L.njobs = 1; L.job[0].out[0] = L.job[0].out[1] = f; say("inverse", L);
    }
}
"""
# refused in both precisions but for these
ACCEPTED = {"good0", "good1", "third0", "term0", "inverse0"}


def test_launch_check(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(CASES)
    subprocess.check_call([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-w",
                           "-I", os.path.join(ROOT, "fug30v0kxc_amd", "csrc"), str(src), "-o", str(exe)])
    got = dict(line.split() for line in subprocess.check_output([str(exe)], text=True).splitlines())
    assert len(got) == 26
    for name, ok in got.items():
        assert (ok == "1") == (name in ACCEPTED), name
