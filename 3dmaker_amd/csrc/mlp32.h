// The 16x16x32 MFMA kernels of the fused MLP (mlp32.hip), behind mlp_forward
// and mlp_backward for the shapes they take.
#pragma once

#include "mlp.h"

namespace graft {

// Samples from which the hash-grid forward encodes in a launch of its own.
constexpr int kPlanarFrom = 1 << 15;

bool mlp32_forward_supported(const MlpShape& s);
void mlp32_forward(const MlpShape& s, const FwdInput& in, const __half* const* W, const float* const* B,
                   __half* const* acts, float* out, int N, int out_act, hipStream_t stream, const uint32_t* d_n);

// Block partials of dW (all layers, at wofs) and db (bofs), P floats each, and
// dx (nullable); returns how many are in ws.
struct Mlp32Backward {
    const __half* dy;
    const __half* const* acts;
    const __half* const* W;
    __half* dx;
    const uint32_t* d_n;
    const int *wofs, *bofs;
    int P;
    Workspace* ws;
};
bool mlp32_backward_supported(const MlpShape& s);
int mlp32_backward(const MlpShape& s, const Mlp32Backward& a, int N, hipStream_t stream);

}  // namespace graft
