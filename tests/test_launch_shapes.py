"""Launch shapes that the host code chooses, on the CPU (a program linked with the library; the rules
take a chip of 256 CUs where there is no GPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "stokesflow.jl_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "sf_host.h"

using namespace sf;

int main(int argc, char** argv)
{
    char what[32];
    int a, b, c;
    while (std::scanf("%31s %d %d %d", what, &a, &b, &c) == 4) {
        if (!std::strcmp(what, "persistent")) std::printf("%d\n", persistent_rows(a, b, c));
        if (!std::strcmp(what, "plan")) std::printf("%d\n", pt_plan(a, b).kind);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    d = tmp_path_factory.mktemp("shapes")
    (d / "shapes.cpp").write_text(PROGRAM)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"), str(d / "shapes.cpp"),
                    "-o", str(d / "shapes"), "-L", PKG, "-lsfhip", "-Wl,-rpath," + PKG], check=True, timeout=300)

    def ask(lines):
        r = subprocess.run([str(d / "shapes")], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        return [[int(v) for v in line.split()] for line in r.stdout.splitlines()]

    return ask


def wave_rounds_rows(k, nx, ny, copies):
    """Tile height of k-iteration passes over `copies` grids: least rounds x steps of 1,024 SIMDs with two waves
    each, a launch of at most one wave per SIMD being 1.38 times faster."""
    strips = -(-(nx - 1) // (64 - 2 * k))

    def cost(rows):
        waves = copies * strips * -(-ny // rows)
        return (rows + 2 * k - 1) * (1.0 if waves <= 1024 else 1.38 * -(-waves // 2048))

    return min(ny, min([2, 4, 6, 8, 10, 12, *range(16, 65, 4)], key=cost))


def test_persistent_rows(shapes):
    """The heights of the persistent kernel's passes: by the number of instances up to 63, then 8 and 16
    rows; never more than the grid has."""
    many = {(128, 128, 70): 8, (257, 40, 64): 16, (512, 512, 200): 16, (64, 5, 100): 5}
    few = [(64, 3, 2), (20, 3000, 8), (256, 256, 4), (256, 256, 63), (64, 64, 1), (455, 400, 24)]
    got = shapes([f"persistent {nx} {ny} {n}" for nx, ny, n in [*many, *few]])
    assert [r[0] for r in got] == [*many.values(), *(wave_rounds_rows(3, *c) for c in few)]


def test_flat_grids_keep_one_wave_passes(shapes):
    """pt_plan's kinds (0 one-wave, 1 resident, 2 pipelined): one-wave only on flat grids of many strips."""
    one_wave = [(50000, 4), (100000, 3), (100000, 8), (250000, 6)]
    others = [(64, 64), (700, 700), (1024, 1024), (4096, 4096), (20000, 3), (20000, 8), (50000, 11), (8, 100000), (250000, 24),
              (16384, 16384), (53, 400000)]
    kinds = [r[0] for r in shapes([f"plan {nx} {ny} 0" for nx, ny in one_wave + others])]
    assert kinds[:len(one_wave)] == [0] * len(one_wave)
    assert 0 not in kinds[len(one_wave):]
