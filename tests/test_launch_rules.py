"""The size rules of the launchers, asked on the host: a C++ program on the
library's internal headers, no device calls."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "amressif_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def _run(tmp_path, body):
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text('#include <cstdio>\n#include "internal.hpp"\n#include "iter_tile.hpp"\n'
                   "int main()\n{\n" + body + "\n}\n")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc"), str(src), "-o", str(exe),
                    "-L" + PKG, "-lamressif_hip", "-L" + ROCM + "/lib", "-lamdhip64",
                    f"-Wl,-rpath,{PKG}:{ROCM}/lib"], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()


def test_one_launch_pseudo_iteration_refuses_sizes_past_its_records(tmp_path):
    """A launch writes one record per workgroup, into a set of kMaxPartials of
    them: 256^2 workgroups at n = 10239, 257^2 at n = 10240, 410^2 at the
    largest context.  (Only the refused sizes reach the launcher here.)"""
    out = _run(tmp_path, """
    for (int n : {4, 1024, 10239, 10240, 14480, 16384}) {
        amr::Ctx c;
        c.g.n = n;
        c.iter_tile = 2;
        const int blocks = amr::iter_tile_blocks(n);
        const bool fits = amr::iteration_fits(c);
        amr::StageLaunch a{};
        a.unguarded = 1;
        const int rc = fits ? 0 : (int)amr::launch_iteration(c, a, nullptr);
        std::printf("%d:%d:%d:%d:%d ", n, blocks <= amr::kMaxPartials, (int)fits, (int)amr::iter_tile_wanted(c), rc);
    }""")
    hip_error_invalid_value = 1
    for line in out:
        n, small, fits, wanted, rc = (int(x) for x in line.split(":"))
        assert fits == small == wanted == (n <= 10239), line
        assert rc == (0 if fits else hip_error_invalid_value), line


@pytest.mark.gpu
def test_timing_the_one_launch_pseudo_iteration_and_its_refusal():
    """which = 11 of the timing entry: 48 B per cell where the launch's records
    fit, refused with the context's message where they do not."""
    from amressif_amd import api
    ms, nbytes = api.Context(api.cavity_inputs(256, 400.0)).time_kernel(11, reps=3)
    assert ms > 0 and nbytes == 48.0 * 256 * 256
    with pytest.raises(api.AmressifError, match="no one-launch pseudo-iteration at this size"):
        api.Context(api.cavity_inputs(10240, 400.0)).time_kernel(11, reps=3)
