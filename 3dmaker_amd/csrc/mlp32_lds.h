// Where the 16x16x32 MLP forward (mlp32.hip) keeps weights and biases in LDS,
// and which rows its layers read.  Plain C++, so that the reads can be walked
// against the sizes on the host.
#pragma once

#if defined(__HIPCC__)
#define GRAFT_HD __host__ __device__ __forceinline__
#else
#define GRAFT_HD inline
#endif

namespace graft {

GRAFT_HD int up16(int d) { return (d + 15) & ~15; }
GRAFT_HD int up32(int d) { return (d + 31) & ~31; }

// The weights in LDS: layer 0's HID rows of up32(in) halves, then the rows of
// all other layers, HID halves each, one after another (the last layer's
// padded to last_rows); every row is followed by 8 halves of padding
// against bank conflicts.
GRAFT_HD int rows0_halves(int hid, int in) { return hid * (up32(in) + 8); }
GRAFT_HD int rows_halves(int hid, int in, int layers, int last_rows)
{
    return rows0_halves(hid, in) + ((layers - 2) * hid + last_rows) * (hid + 8);
}
// First LDS half of layer l's rows.
GRAFT_HD int row_base(int hid, int in, int l)
{
    return l == 0 ? 0 : rows0_halves(hid, in) + (l - 1) * hid * (hid + 8);
}

// What is staged, in chunks of 8 halves: row by row, layer 0's rows first.
// Chunk q comes from half `at` of its layer's W (zeros where !ok: outside the
// matrix) and goes to half dst.  Every layer behind layer 0 has hid rows but
// the last, which may have more.  Rows of both kinds are 8 halves apart from
// each other, so that dst is q and the rows before it.  Written for few
// instructions and no branch, one chunk per thread: what a small batch waits
// for (1,003 samples of 8-128-128-128-8 11.3 to 11.8 us with rows and columns
// worked out apart, 10.8 with the two kinds of rows in branches, 10.2 so).
struct Staged {
    int layer, at, dst;
    bool ok;
};
GRAFT_HD int staged_chunks(int hid, int in, int layers, int last_rows)
{
    return (hid * up32(in) + ((layers - 2) * hid + last_rows) * hid) / 8;
}
GRAFT_HD Staged staged_chunk(int q, int hid, int in, int out, int layers)
{
    const int blocks = up32(in) / 32, first_end = hid * blocks * 4;  // a row of layer 0 has 4 * blocks chunks
    const int reciprocal = blocks == 1 ? 65536 : blocks == 2 ? 32768 : blocks == 3 ? 21846 : 16384;  // of blocks, 2^16
    const int first = q < first_end ? -1 : 0;  // all bits: both sides are worked out and selected, without a branch
    const int row0 = ((q >> 2) * reciprocal) >> 16;
    const int R = (q - first_end) >> (hid == 128 ? 4 : hid == 64 ? 3 : 2);  // row behind layer 0 (negative: layer 0)
    const int piece = R >> (hid == 128 ? 7 : hid == 64 ? 6 : 5);
    const int l = piece < -1 ? 0 : piece > layers - 2 ? layers - 1 : piece + 1;
    Staged s;
    s.layer = l;
    s.dst = 8 * (q + ((row0 & first) | ((hid + R) & ~first)));
    s.at = 8 * q + ((row0 * (in - 32 * blocks) & first) | ((-8 * first_end - (l - 1) * hid * hid) & ~first));
    s.ok = (((8 * q - row0 * 32 * blocks) & first) | (R & ~first)) < ((in & first) | (((layers - 2) * hid + out) & ~first));
    return s;
}

// The forward's last layer: one block of 16 rows, or pairs of blocks whose
// rows are dealt as the hidden layers' are (a block of a pair reaches into all
// 32 rows of it, so whole pairs are staged).
GRAFT_HD bool fwd32_pairs(int out) { return out > 16; }
GRAFT_HD int fwd32_last_rows(int out) { return fwd32_pairs(out) ? up32(out) : 16; }
GRAFT_HD int fwd32_last_steps(int out) { return fwd32_pairs(out) ? up32(out) / 32 : 1; }
// Row of a block that lane r reads: the first row of block m of pair q is 32 q + 4 m.
GRAFT_HD int fwd32_lane_row(bool pairs, int r) { return pairs ? 8 * (r >> 2) + (r & 3) : r; }
// First output of lane group g in block m of a pair, whose biases and results are 4 floats from there.
GRAFT_HD int fwd32_lane_col(bool pairs, int q, int m, int g) { return pairs ? 32 * q + 8 * g + 4 * m : 4 * g; }
// Biases behind the weights, HID floats apart: their byte offset, count, and the bytes of everything.
GRAFT_HD int fwd32_bias_base(int in, int hid, int out, int layers)
{
    return (rows_halves(hid, in, layers, fwd32_last_rows(out)) * 2 + 15) & ~15;
}
GRAFT_HD int fwd32_biases(int hid, int out, int layers) { return (layers - 1) * hid + fwd32_last_rows(out); }
GRAFT_HD int fwd32_lds(int in, int hid, int out, int layers)
{
    return fwd32_bias_base(in, hid, out, layers) + 4 * fwd32_biases(hid, out, layers);
}

}  // namespace graft
