"""The persistent CG where the HIP runtime refuses what it needs: it leaves the solve to the launches and reports no
error. Without a GPU every runtime call is refused, so this runs on the CPU alone."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "lpm-mac_amd", "liblpm_mi355x.so")

SOURCE = r"""
#include <cstdio>
#include "lpm_internal.h"
int main() {
    int n = 0;
    if (hipGetDeviceCount(&n) == hipSuccess && n > 0) return std::puts("has a GPU"), 0;
    (void)hipGetLastError();
    int bad = 0;
    for (int precond = 0; precond < 3; ++precond)
        for (int precision = 0; precision < 2; ++precision)
            for (int prepared = 0; prepared < 2; ++prepared) {
                // one aggregate of 64 particles; `prepared`: the lists are there and the launch is what fails
                lpm_ctx c;
                c.n = 64;
                c.nslice = 1;
                c.nslots = 64 * 8;
                c.dim = 3;
                c.precond = precond;
                c.precision = precision;
                c.nagg = c.ncgrp = 1;
                c.ncoarse = c.cgrp_nbmax = c.nmode = 6;
                PcgPlan &p = c.pcg_plan[precond == 2];
                if (prepared) p.state = p.spw = p.grid = 1;
                for (int again = 0; again < 2; ++again) {
                    bool ran = true;
                    const int rc = pcg_solve(&c, 10, &ran);
                    if (rc != LPM_OK || ran)
                        ++bad, std::printf("precond %d precision %d prepared %d: %d %s\n", precond, precision, prepared, rc, c.err.c_str());
                }
            }
    std::printf("%d wrong\n", bad);
    return bad != 0;
}
"""


def test_runtime_refuses(tmp_path):
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    src, exe = tmp_path / "fallback.cpp", tmp_path / "fallback"
    src.write_text(SOURCE)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-D__HIP_PLATFORM_AMD__", "-std=c++17", "-I", os.path.join(ROOT, "lpm-mac_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(rocm, "include"), str(src), "-o", str(exe), LIB,
                    "-L", os.path.join(rocm, "lib"), "-lamdhip64", "-Wl,-rpath," + os.path.dirname(LIB) + ":" + os.path.join(rocm, "lib")],
                   check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(r.stdout, r.stderr)
    assert r.returncode == 0, r.stdout
