"""What the 16x16x32 MLP kernels stage in LDS, and every address that the forward's layers read, against what is
staged: csrc/mlp32_lds.h built for the host and walked over every shape (widths, outputs narrower and wider than the
hidden layers, depths) the forward takes."""
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
                    if (fwd32_lds(in, hid, out, layers) > 160 * 1024) continue;
                    shapes++;
                    // what is staged: every chunk of every row once, from its place in W to where its layer is read
                    const int last = fwd32_last_rows(out);
                    int q = 0;
                    for (int l = 0; l < layers; l++) {
                        const int ld = l == 0 ? in : hid, width = l == 0 ? up32(in) : hid, end_l = l == layers - 1;
                        for (int row = 0; row < (end_l ? last : hid); row++)
                            for (int c = 0; c < width; c += 8, q++) {
                                const Staged s = staged_chunk(q, hid, in, out, layers);
                                const bool ok = c < ld && row < (end_l ? out : hid);
                                if (s.layer != l || s.ok != ok || (ok && s.at != row * ld + c) ||
                                    s.dst != row_base(hid, in, l) + row * (width + 8) + c)
                                    return printf("chunk %d of %d-%d-%d x %d: layer %d row %d column %d\n", q, in, hid,
                                                  out, layers, l, row, c), 1;
                            }
                    }
                    if (q != staged_chunks(hid, in, layers, last)) return printf("chunks %d\n", q), 1;
                    const int biases = fwd32_biases(hid, out, layers);
                    if (fwd32_bias_base(in, hid, out, layers) % 16) return printf("bias base unaligned\n"), 1;
                    for (int l = 0; l < layers; l++) {
                        const bool end_l = l == layers - 1, pairs = !end_l || fwd32_pairs(out);
                        const int pitch = (l == 0 ? up32(in) : hid) + 8, depth = l == 0 ? up32(in) : hid;
                        const int steps = end_l ? fwd32_last_steps(out) : hid / 32;
                        const int rows = end_l ? last : hid;  // staged for this layer
                        if (row_base(hid, in, l) + rows * pitch > rows_halves(hid, in, layers, fwd32_last_rows(out)))
                            return printf("rows of layer %d outside: %d-%d-%d x %d\n", l, in, hid, out, layers), 1;
                        for (int q = 0; q < steps; q++)
                            for (int m = 0; m < (pairs ? 2 : 1); m++)
                                for (int lane = 0; lane < 64; lane++) {
                                    const int r = lane & 15, g = lane >> 4;
                                    const int row = fwd32_lane_row(pairs, r) + 32 * q + 4 * m;
                                    const int end = 8 * g + depth - 32 + 8;  // behind the last 16-byte read of the row
                                    if (row >= rows || end > pitch)
                                        return printf("layer %d of %d-%d-%d x %d: row %d of %d, half %d of %d\n", l, in,
                                                      hid, out, layers, row, rows, end, pitch), 1;
                                    const int b = l * hid + fwd32_lane_col(pairs, q, m, g) + 4;
                                    if (b > biases || (!end_l && b > (l + 1) * hid))
                                        return printf("layer %d of %d-%d-%d x %d: bias %d of %d\n", l, in, hid, out,
                                                      layers, b, biases), 1;
                                }
                    }
                }
    printf("%d shapes\n", shapes);
    return shapes > 3000 ? 0 : 1;
}
"""


def test_forward_reads_only_staged_rows_and_biases(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "3dmaker_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
