// Where the 16x16x32 MLP kernels (mlp32.hip) keep weights in LDS.  Plain C++, so
// that what is staged can be walked on the host.
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

// Row R of the rows behind layer 0, counted through: its layer, and its row
// there.  Every layer has hid rows but the last, which may have more.
GRAFT_HD int staged_layer(int R, int hid, int layers)
{
    const int l = 1 + R / hid;
    return l < layers - 1 ? l : layers - 1;
}
GRAFT_HD int staged_row(int R, int hid, int l) { return R - (l - 1) * hid; }

}  // namespace graft
