"""What the 16x16x32 MLP kernels stage in LDS (csrc/mlp32_lds.h, built for the host), walked over every shape they
take: widths, outputs narrower and wider than the hidden layers, depths."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WALK = r"""
#include <cstdio>
#include <initializer_list>
#include "mlp32_lds.h"
using namespace graft;

int main()
{
    int shapes = 0;
    for (int hid : {32, 64, 128})
        for (int in = 8; in <= 128; in += 8)
            for (int out = 4; out <= 128; out += 4)
                for (int layers = 2; layers <= 16; layers++) {
                    shapes++;
                    // what is staged: every row behind layer 0 has a layer, and goes where that layer is read
                    const int last = up32(out);
                    for (int R = 0; R < (layers - 2) * hid + last; R++) {
                        const int l = staged_layer(R, hid, layers), row = staged_row(R, hid, l);
                        if (l < 1 || l >= layers || row < 0 || row >= (l < layers - 1 ? hid : last) ||
                            rows0_halves(hid, in) + R * (hid + 8) != row_base(hid, in, l) + row * (hid + 8))
                            return printf("row %d of %d-%d-%d x %d: layer %d row %d\n", R, in, hid, out, layers, l, row), 1;
                    }
                }
    printf("%d shapes\n", shapes);
    return shapes > 3000 ? 0 : 1;
}
"""


def walk(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "3dmaker_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


def test_every_staged_row_belongs_to_a_layer(tmp_path):
    r = walk(tmp_path)
    assert r.returncode == 0, r.stdout
