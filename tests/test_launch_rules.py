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


def test_odd_bottoms_are_solved_by_the_faster_form(tmp_path):
    """Strips of a padded depth of 128 or four dense products: FP64 takes the
    products up to 63 cells a side, where they are faster, and both types past
    128."""
    out = _run(tmp_path, """
    for (int m : {33, 49, 63, 65, 81, 127, 129})
        std::printf("%d%d ", (int)amr::bottom_strips(m, m, false), (int)amr::bottom_strips(m, m, true));
    """)
    assert out == ["01", "01", "01", "11", "11", "11", "00"]


def test_overlapping_output_views_are_not_written_in_one_launch(tmp_path):
    """Items that share memory start a new launch, so the last one of the list
    stays, as with a launch each: two views of one array, a view into the end of
    another, the second component of a cell array over a face array.  Views that
    only touch, and the components of one array, stay together."""
    n = 8
    out = _run(tmp_path, """
    const int n = 8;
    static double mem[4096];
    amr::Ctx c;
    c.g.n = n;
    auto xface = [&](double *p) { return amr_array4{p, {0, 0, 0}, {n, n - 1, 0}, 1, 0}; };
    auto cells = [&](double *p, int g) { return amr_array4{p, {-g, -g, 0}, {n - 1 + g, n - 1 + g, 0}, 2, 0}; };
    const int size = (n + 1) * n;
    const amr_array4 a = xface(mem), b = xface(mem), tail = xface(mem + size - 1), next = xface(mem + size),
                     uc = cells(mem + 1000, 1), over = xface(mem + 1000 + 100 + 50), before = xface(mem + 1000 - size + 11);
    auto put = [&](std::initializer_list<const amr_array4 *> faces) {
        amr::Copies l;
        for (const amr_array4 *f : faces) l.face(c, *f, nullptr, 0);
        for (int q = 0; q < l.count; q = l.disjoint_end(q)) std::printf("%d", l.disjoint_end(q));
        std::printf(" ");
    };
    put({&a, &next});
    put({&a, &b, &next});
    put({&a, &tail});
    put({&tail, &a, &b, &next});
    amr::Copies l;
    l.cell(c, uc, 0, nullptr);
    l.cell(c, uc, 1, nullptr);
    std::printf("%d ", l.disjoint_end(0));
    l.face(c, over, nullptr, 0);
    std::printf("%d%d ", l.disjoint_end(0), l.disjoint_end(2));
    amr::Copies m;  // ends where the box's cells begin, in the view's ghosts
    m.face(c, before, nullptr, 0);
    m.cell(c, uc, 0, nullptr);
    std::printf("%d", m.disjoint_end(0));
    """)
    # the launches' ends; {tail, a, b, next}: tail alone (a reaches into it), a, then b and next
    assert out == ["2", "13", "12", "124", "2", "23", "2"], (n, out)


@pytest.mark.gpu
def test_one_array_for_two_outputs_keeps_the_last_one():
    """One array as scratch for both half-node fluxes, and for the state and the
    one before: it ends with the output written last."""
    import torch
    from amressif_amd import api
    from amressif_amd import workloads as W
    n = 200
    ctx = api.Context(api.cavity_inputs(n, 400.0))
    g = torch.Generator("cuda").manual_seed(3)
    rnd = lambda *s: torch.rand(s, dtype=torch.float64, device="cuda", generator=g) - 0.5  # noqa: E731
    u, v = rnd(n, n + 1), rnd(n + 1, n)
    _, _, half = ctx.fluxes(u, v)
    for _ in range(20):
        x, y = torch.zeros_like(u), torch.zeros_like(v)
        one = api.faces_view(x, y, n)
        ctx._check(api._lib.amressif_fluxes(ctx._h, api.faces_view(u, v, n), None, None, one, one))
        assert torch.equal(x, half[2]) and torch.equal(y, half[3])
    ctx.load_faces([u, v], [2 * u, 2 * v], None)
    x, y = torch.zeros_like(u), torch.zeros_like(v)
    ctx.store_faces([x, y], [x, y], None)
    assert torch.equal(x, 2 * u) and torch.equal(y, 2 * v)
