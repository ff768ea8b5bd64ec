"""The footprint of one RK stage that decides about non-temporal marks, counted
array by array: 3D FP32 gradients read one word more per entry (a packed slot or
the cell the entry leads to), not the 120 B of unpacked slots that are read only
past the line."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lfm_public_amd", "csrc")

MAIN = """
#include <cstdio>
#include <cstdlib>
#include "mesh_builder.hpp"
int main(int, char **v) {
    lfm::StageShape s;
    s.D = atoi(v[1]); s.word = atoi(v[2]); s.nc = atol(v[3]); s.nf = atol(v[4]);
    s.one_launch = atoi(v[5]); s.packed = atoi(v[6]); s.grad_values = atoi(v[7]);
    const size_t b = lfm::stage_footprint(s);
    printf("%zu %d\\n", b, (int)lfm::outgrows_cache(b));
}
"""


@pytest.fixture(scope="module")
def footprint(tmp_path_factory):
    d = tmp_path_factory.mktemp("footprint")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "footprint")
    subprocess.check_call(["g++", "-std=c++17", "-I", CSRC, "-I", os.path.join(ROOT, "include"), str(d / "main.cpp"),
                           "-o", exe])

    def run(*args):
        b, nt = subprocess.check_output([exe, *(str(int(a)) for a in args)], text=True).split()
        return int(b), bool(int(nt))
    return run


def _expected(D, w, nc, nf, one, packed, g):
    state, reg, other = (D + 2) * w, (D + 2) * w, 2 * w  # 1/V, sponge
    slots = 4 if D == 2 else 6
    if one:
        return nc * (2 * state + reg + other + slots * (4 if packed else 4 + (D + 1) * w))
    face = (D + 2) * w + D * w + D * w + w + 2 * 4  # flux, S, d, w, both cells
    return nc * (state + reg + other + slots * 4 + (g * w + slots * 4 if g else 0)) + nf * face


@pytest.mark.parametrize("args", [
    (3, 4, 1048576, 3178496, 0, 0, 12), (3, 4, 1000000, 3030000, 0, 1, 12), (3, 8, 193161, 585000, 0, 0, 24),
    (2, 4, 1048576, 1835008, 0, 0, 10), (2, 8, 262144, 458752, 0, 0, 10), (3, 4, 4096000, 12364800, 1, 1, 0),
    (3, 4, 4096000, 12364800, 1, 0, 0), (2, 8, 65536, 131584, 1, 1, 0), (2, 4, 65536, 131584, 0, 0, 0)])
def test_footprint_counts_each_array_once(footprint, args):
    b, nt = footprint(*args)
    assert b == _expected(*args)
    assert nt == (b > 330_000_000)


def test_packed_slots_and_entries_count_alike(footprint):
    """A uniform viscous box of 313 MB stays below the line, packed or not."""
    n = 1_000_000
    a, b = footprint(3, 4, n, 3 * n, 0, 1, 12), footprint(3, 4, n, 3 * n, 0, 0, 12)
    assert a == b and not a[1]
