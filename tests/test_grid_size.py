"""The sizes of the photon grid's buffers at the largest build that is accepted (host only)."""
import os
import subprocess

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "imbatracer_amd", "csrc", "hip",
                      "grid_size.h")


def test_sizes_at_the_limit(tmp_path):
    """Evaluated by the compiler, which rejects an arithmetic overflow in a constant."""
    src = tmp_path / "sizes.cpp"
    src.write_text("""#include "%s"
using namespace imba;
static_assert(grid_table_size(0, 0) == 0 && grid_table_size(100, 7) == 100 && grid_table_size(100, 51) == 102, "");
static_assert(grid_table_size(0, kGridMaxPhotons) == 1 << 30, "");
static_assert(grid_box_words(1) == 6 && grid_box_words(357913942) == 2147483652u, "");
static_assert(grid_box_words(grid_table_size(0, kGridMaxPhotons)) == 6442450944u, "");
""" % HEADER)
    p = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", str(src)], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
