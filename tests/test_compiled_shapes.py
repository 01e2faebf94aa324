"""What the kernel headers promise at compile time, checked by compiling small sources against them (no device)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skirt7_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")


def compiles(tmp_path, body):
    src = tmp_path / "t.hip"
    src.write_text('#include <hip/hip_runtime.h>\n#include "../../include/skirt7_amd.h"\n#include "sg_host.hpp"\n'
                   '#include "sg_mc.hpp"\n#include "sg_split.hpp"\nusing namespace sg;\n' + body)
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "-I" + CSRC, str(src)],
                       capture_output=True, text=True)
    return r.returncode == 0, r.stdout + r.stderr


def test_parking_area_holds_the_parked_state(tmp_path):
    """The LDS words set aside per lane are the words that a walk's state moves when it is parked."""
    ok, text = compiles(tmp_path, """
struct Words {
    int n = 0;
    template <typename T> __host__ __device__ constexpr void io(T&) { n += sizeof(T) == 8 ? 2 : 1; }
};
template <class W> constexpr int moved() { Hot<W> h{}; Words w; h.park(w); return w.n; }
#define SAME(W) static_assert(moved<W>() == hot_words<W>(), "parked words")
SAME(CartW64); SAME(CartW32); SAME(TreeW64); SAME(TreeW64Book); SAME(TreeW32); SAME(TreeW32TopDown);
SAME(VoroW<double>); SAME(VoroW<float>);
static_assert(hot_words<CartW64>() == 2 * (9 + 3 + 1 + 3) + 5 + 3 + 2 * 7 + 4, "exact Cartesian walk");
""")
    assert ok, text


def test_voronoi_groups_look_for_walls_where_they_are(tmp_path):
    """Of a list whose walls are among its first eight entries, dealt out to L lanes, a step looks for walls in every
    round of L entries that can hold one; group sizes the reductions cannot take are refused."""
    ok, text = compiles(tmp_path, """
template <class W> constexpr bool covers()
{
    for (int entry = 0; entry < kVoroWalls; entry++)
        if (!W::holds_walls(entry / W::kLanes)) return false;
    return true;
}
static_assert(covers<VoroC<float, 2, 12>>() && covers<VoroC<float, 4, 6>>() && covers<VoroC<float, 8, 3>>() &&
              covers<VoroC<double, 16, 2>>(), "walls beyond the entries looked at");
static_assert(!VoroC<float, 8, 3>::holds_walls(1), "eight lanes take the walls in one round");
""")
    assert ok, text
    for lanes in (3, 32):
        assert not compiles(tmp_path, "static_assert(sizeof(VoroC<float, %d, 2>) > 0, \"\");\n" % lanes)[0]


def test_run_errors_name_their_cause(tmp_path):
    """Every kind of run reports its error bits by the same texts: 1 the optical depth, 2 the walk order, 4 the walk
    queue, the library's own checks first; no entry point words them by itself."""
    ok, text = compiles(tmp_path, """
constexpr bool starts(const char* s, const char* w) { return !*w || (*s == *w && starts(s + 1, w + 1)); }
static_assert(starts(run_error(1), "The optical depth"), "");
static_assert(starts(run_error(2), "walk order") && starts(run_error(3), "walk order") && starts(run_error(6), "walk order"), "");
static_assert(starts(run_error(4), "walk queue") && starts(run_error(5), "walk queue"), "");
""")
    assert ok, text
    with open(os.path.join(CSRC, "sg_kernels.hip")) as f:
        source = f.read()
    for words in ("The optical depth along", "walk order: a request", "walk queue: a request"):
        assert words not in source
