// TinyMLP forward and backward on v_mfma_f32_16x16x32_f16 for nets of hidden
// width 32, 64 or 128 (every width the TinyMLP classes pad to, up to 128).
//
// Layout.  Activations are the B operand, samples along N: lane (r, g) holds
// features 8 g .. 8 g + 7 of 32-feature block kb of sample r.  Weights are the
// A operand, read from LDS where they lie as padded rows W[out][in].  The rows
// of a pair of 16-row blocks are dealt so that D puts output features
// 32 p + 8 g + 4 m + j into lane (r, g): eight consecutive features per lane,
// which is the next layer's B operand as it stands and one 16-byte store of
// the saved activation.
//
// Rounding points as in mlp.hip: hidden activations -> fp16 after bias + ReLU
// (the bias is where the accumulators start), the last layer stays fp32; each
// dX -> fp16, then masked where the saved activation is not positive.  dW and
// db are fp32 sums, reduced over blocks in a fixed order.
#include "mlp.h"
#include "mlp32.h"

#include "hash_encode.h"
#include "hashgrid.h"

#include <algorithm>

namespace graft {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f4 mfma32(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ h8 h8zero()
{
    const _Float16 z = (_Float16)0.f;
    return h8{z, z, z, z, z, z, z, z};
}

__host__ __device__ __forceinline__ int up16(int d) { return (d + 15) & ~15; }
__host__ __device__ __forceinline__ int up32(int d) { return (d + 31) & ~31; }

// The weights in LDS: layer 0's HID rows of up32(in) halves, then the rows of
// all other layers, HID halves each, one after another (the last layer's
// padded to a multiple of 16); every row is followed by 8 halves of padding
// against bank conflicts.
__host__ __device__ __forceinline__ int rows0_halves(int hid, int in) { return hid * (up32(in) + 8); }
__host__ __device__ __forceinline__ int rows_halves(int hid, int in, int out, int layers)
{
    return rows0_halves(hid, in) + ((layers - 2) * hid + up16(out)) * (hid + 8);
}
// First LDS half of layer l's rows, and their pitch.
template <int HID>
__device__ __forceinline__ int row_base(int l, int in)
{
    return l == 0 ? 0 : rows0_halves(HID, in) + (l - 1) * HID * (HID + 8);
}

// Copies every layer's W rows into LDS, zeros outside the matrix.  Each thread
// has kBatch 16-byte loads in flight; nothing branches around a load (a chunk
// outside the matrix reads its layer's first one): with a branch per chunk
// they came one after another, and 1,003 samples through 8-128-128-128-8 took
// 18.4 us instead of 11.4.  All threads call; ends with a barrier.
template <int HID>
__device__ __forceinline__ void stage_rows(_Float16* sw, const _Float16* const* W, int in, int out, int layers)
{
    constexpr int kBatch = 12;
    constexpr int C = HID / 8;  // chunks of a row behind layer 0
    __shared__ const _Float16* sW[kMaxLayers];
    const int tid = threadIdx.x;
    if (tid < layers) sW[tid] = W[tid];
    __syncthreads();
    uintptr_t low = 0;
    for (int l = 0; l < layers; l++) low |= reinterpret_cast<uintptr_t>(sW[l]);
    const bool vec = __builtin_amdgcn_readfirstlane((int)(low & 15u)) == 0;
    const int C0 = up32(in) >> 3, total0 = HID * C0;
    const int total = total0 + ((layers - 2) * HID + up16(out)) * C;
    for (int base = 0; base < total; base += kBatch * (int)blockDim.x) {
        h8 v[kBatch];
        int dst[kBatch];
        bool ok[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; k++) {
            const int q = min(base + k * (int)blockDim.x + tid, total - 1);
            const bool first = q < total0;
            const int row0 = (int)((unsigned)q / (unsigned)C0);
            const int e = q - total0, R = e / C;
            const int l = first ? 0 : 1 + R / HID;
            const int row = first ? row0 : R % HID;
            const int c = 8 * (first ? q - row0 * C0 : e % C);
            const int ld = first ? in : HID;
            dst[k] = first ? row * (8 * C0 + 8) + c : rows0_halves(HID, in) + R * (HID + 8) + c;
            ok[k] = c < ld && (l < layers - 1 || row < out);
            const _Float16* src = sW[l] + (ok[k] ? row * ld + c : 0);
            if (vec) {
                v[k] = *reinterpret_cast<const h8*>(src);
            } else {
#pragma unroll
                for (int j = 0; j < 8; j++) v[k][j] = src[j];
            }
        }
#pragma unroll
        for (int k = 0; k < kBatch; k++)
            if (base + k * (int)blockDim.x + tid < total) *reinterpret_cast<h8*>(sw + dst[k]) = ok[k] ? v[k] : h8zero();
    }
    __syncthreads();
}

__device__ __forceinline__ void st_row8(_Float16* dst, h8 v)
{
    if ((reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
        *reinterpret_cast<h8*>(dst) = v;
    } else {
#pragma unroll
        for (int j = 0; j < 8; j++) dst[j] = v[j];
    }
}

__device__ __forceinline__ h8 ld_row8(const _Float16* src)
{
    if ((reinterpret_cast<uintptr_t>(src) & 15u) == 0) return *reinterpret_cast<const h8*>(src);
    h8 v;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = src[j];
    return v;
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------

enum { kRows = 0, kFused = 1, kPlanar = 2 };  // layer 0's input: fp16 rows, positions, level-major encodings

struct Fwd32Params {
    const _Float16* x;         // kRows: [N x x_dim]
    const float* pos;          // kFused
    const _Float16* table;     // kFused
    const _Float16* enc;       // kPlanar: [L][plane] feature pairs
    _Float16* const* acts;     // SAVE
    const _Float16* const* W;
    const float* const* B;
    float* out;                // nullable [N x out_dim]
    float* user;               // nullable [N x user_dim]: the first user_dim outputs again
    const uint32_t* d_n;
    int N, in, out_dim, layers, pos_stride, plane, x_dim, user_dim;
    int save_x0, vec_x, vec_out, vec_user;
    int L, T, dense_start;
    int bias_base;  // bytes into LDS; layer l's biases HID floats apart
    float scale[kMaxLevels];
    int res[kMaxLevels];
};

// A wave takes NT tiles of 16 samples through every layer; each weight
// fragment read from LDS serves its NT tiles.  Bound by the bytes of input,
// saved activations and outputs for wide batches; the loads of the next tiles
// are issued before the current ones are computed.
// 2^18 samples through 64-64-64-64-64 with saved activations, 168 MB written and 34 read: 104 us and a 23 us copy to
// the caller's rows before, 65 us with that copy in it.
template <int HB, int NT, int MODE, bool SAVE, int OUT_ACT>
__global__ __launch_bounds__(256) void mlp32_fwd_kernel(const Fwd32Params p)
{
    constexpr int HID = 32 * HB;
    extern __shared__ __align__(16) unsigned char smem[];
    _Float16* sw = reinterpret_cast<_Float16*>(smem);
    float* sb = reinterpret_cast<float*>(smem + p.bias_base);
    // the first two biases of a thread are on their way while the weights are staged
    const int tid = threadIdx.x, nb = (p.layers - 1) * HID + up16(p.out_dim);
    auto bias = [&](int e) {
        const int l = min(e / HID, p.layers - 1), i = e - l * HID;
        const bool ok = e < nb && i < (l == p.layers - 1 ? p.out_dim : HID);
        const float v = p.B[l][ok ? i : 0];
        return ok ? v : 0.f;
    };
    const float b0 = bias(tid), b1 = bias(tid + 256);
    stage_rows<HID>(sw, p.W, p.in, p.out_dim, p.layers);
    if (tid < nb) sb[tid] = b0;
    if (tid + 256 < nb) sb[tid + 256] = b1;
    for (int e = tid + 512; e < nb; e += 256) sb[e] = bias(e);
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int N = p.d_n ? min((int)*p.d_n, p.N) : p.N;
    const int units = (N + 16 * NT - 1) / (16 * NT);
    const int KB0 = (p.in + 31) >> 5;
    constexpr int XB = 4;  // 32-feature blocks of the widest input
    _Float16* act0 = nullptr;
    if constexpr (SAVE) act0 = p.acts[0];

    auto load = [&](int u, h8 (&X)[NT][XB]) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int n = (u * NT + t) * 16 + r;
#pragma unroll
            for (int kb = 0; kb < XB; kb++) {
                X[t][kb] = h8zero();
                if (kb >= KB0) continue;
                const int col = 32 * kb + 8 * g;
                if (n >= N || col >= p.in) continue;
                if constexpr (MODE == kRows) {
                    const _Float16* src = p.x + (size_t)n * p.x_dim + col;
                    if (p.vec_x) {
                        X[t][kb] = *reinterpret_cast<const h8*>(src);
                    } else {
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            if (col + j < p.x_dim) X[t][kb][j] = src[j];
                    }
                } else {
                    const int l0 = col >> 1;
                    if constexpr (MODE == kPlanar) {
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            if (l0 + j < p.L) {
                                const h2 v = *reinterpret_cast<const h2*>(p.enc + ((size_t)(l0 + j) * p.plane + n) * 2);
                                X[t][kb][2 * j] = v.x;
                                X[t][kb][2 * j + 1] = v.y;
                            }
                    } else {
                        const float* pp = p.pos + (size_t)n * p.pos_stride;
                        const float px = pp[0], py = pp[1], pz = pp[2];
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            if (l0 + j < p.L) {
                                const int l = l0 + j;
                                const float2 e = encode_level(px, py, pz, p.scale[l], p.res[l], l < p.dense_start,
                                                              (uint32_t)p.T - 1u, p.table + (size_t)l * p.T * 2);
                                X[t][kb][2 * j] = to_h(e.x);
                                X[t][kb][2 * j + 1] = to_h(e.y);
                            }
                    }
                }
            }
        }
    };

    int u = blockIdx.x * 4 + wave;
    const int stride = gridDim.x * 4;
    h8 nxt[NT][XB];
    if (u < units) load(u, nxt);
    for (; u < units; u += stride) {
        h8 X[NT][XB];
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int kb = 0; kb < XB; kb++) X[t][kb] = nxt[t][kb];
        if (u + stride < units) load(u + stride, nxt);
        if (SAVE && (MODE != kRows || p.save_x0)) {
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int n = (u * NT + t) * 16 + r;
#pragma unroll
                for (int kb = 0; kb < XB; kb++) {
                    const int col = 32 * kb + 8 * g;
                    if (kb < KB0 && n < N && col < p.in) st_row8(act0 + (size_t)n * p.in + col, X[t][kb]);
                }
            }
        }
        for (int l = 0; l < p.layers - 1; l++) {
            const int KS = l == 0 ? KB0 : HB;
            const int pitch = l == 0 ? 32 * KB0 + 8 : HID + 8;
            const _Float16* w = sw + row_base<HID>(l, p.in) + (8 * (r >> 2) + (r & 3)) * pitch + 8 * g;
            const float* bl = sb + l * HID + 8 * g;
            h8 Y[NT][HB];
#pragma unroll
            for (int q = 0; q < HB; q++) {
                f4 acc[NT][2];
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int m = 0; m < 2; m++) acc[t][m] = *reinterpret_cast<const f4*>(bl + 32 * q + 4 * m);
#pragma unroll
                for (int kb = 0; kb < XB; kb++) {
                    if (kb >= KS) continue;
#pragma unroll
                    for (int m = 0; m < 2; m++) {
                        const h8 a = *reinterpret_cast<const h8*>(w + (32 * q + 4 * m) * pitch + 32 * kb);
#pragma unroll
                        for (int t = 0; t < NT; t++) acc[t][m] = mfma32(a, X[t][kb], acc[t][m]);
                    }
                }
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const float v = acc[t][j >> 2][j & 3];
                        Y[t][q][j] = to_h(v > 0.f ? v : 0.f);
                    }
            }
            _Float16* act = nullptr;
            if constexpr (SAVE) act = p.acts[l + 1];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const int n = (u * NT + t) * 16 + r;
#pragma unroll
                for (int q = 0; q < HB; q++) {
                    X[t][q] = Y[t][q];
                    if (SAVE && n < N) st_row8(act + (size_t)n * HID + 32 * q + 8 * g, Y[t][q]);
                }
            }
        }
        // last layer: blocks of 16 outputs when there are at most 16, else pairs
        const int l = p.layers - 1;
        const int pitch = HID + 8;
        const bool pairs = p.out_dim > 16;
        const _Float16* w = sw + row_base<HID>(l, p.in) + (pairs ? 8 * (r >> 2) + (r & 3) : r) * pitch + 8 * g;
        const float* bl = sb + l * HID;
        const int OQ = pairs ? (p.out_dim + 31) >> 5 : 1;
        for (int q = 0; q < OQ; q++) {
#pragma unroll
            for (int m = 0; m < 2; m++) {
                if (m == 1 && !pairs) continue;
                const int col = pairs ? 32 * q + 8 * g + 4 * m : 4 * g;
                f4 acc[NT];
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = *reinterpret_cast<const f4*>(bl + col);
#pragma unroll
                for (int kb = 0; kb < HB; kb++) {
                    const h8 a = *reinterpret_cast<const h8*>(w + (32 * q + 4 * m) * pitch + 32 * kb);
#pragma unroll
                    for (int t = 0; t < NT; t++) acc[t] = mfma32(a, X[t][kb], acc[t]);
                }
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const int n = (u * NT + t) * 16 + r;
                    if (n >= N || col >= p.out_dim) continue;
                    f4 y = acc[t];
                    if (OUT_ACT == 1) {
#pragma unroll
                        for (int j = 0; j < 4; j++) y[j] = 1.0f / (1.0f + expf(-y[j]));
                    }
                    if (p.out) {
                        float* dst = p.out + (size_t)n * p.out_dim + col;
                        if (p.vec_out) {
                            *reinterpret_cast<f4*>(dst) = y;
                        } else {
#pragma unroll
                            for (int j = 0; j < 4; j++) dst[j] = y[j];
                        }
                    }
                    if (p.user) {
                        float* dst = p.user + (size_t)n * p.user_dim + col;
                        if (p.vec_user) {
                            *reinterpret_cast<f4*>(dst) = y;
                        } else {
#pragma unroll
                            for (int j = 0; j < 4; j++)
                                if (col + j < p.user_dim) dst[j] = y[j];
                        }
                    }
                }
            }
        }
    }
}

constexpr int kStaticLds = kMaxLayers * 8 + 64;  // stage_rows' pointers, rounded up

template <int HB, int MODE, bool SAVE, int ACT>
void launch_fwd32(const Fwd32Params& p, int lds, int N, hipStream_t stream)
{
    // two tiles per wave once every SIMD has a wave that way
    const bool two = N >= 32 * 4 * num_cus();
    const int units = (N + (two ? 31 : 15)) / (two ? 32 : 16);
    const int per_cu = std::max(1, std::min(8, max_lds_per_block() / (lds + kStaticLds)));
    const int blocks = std::max(1, std::min((units + 3) / 4, num_cus() * per_cu));
    if (two)
        hipLaunchKernelGGL((mlp32_fwd_kernel<HB, 2, MODE, SAVE, ACT>), dim3(blocks), dim3(256), lds, stream, p);
    else
        hipLaunchKernelGGL((mlp32_fwd_kernel<HB, 1, MODE, SAVE, ACT>), dim3(blocks), dim3(256), lds, stream, p);
    GRAFT_LAUNCH_CHECK();
}

template <int HB>
void pick_fwd32(const Fwd32Params& p, int mode, bool save, int act, int lds, int N, hipStream_t stream)
{
    if (mode == kPlanar) {
        if (save) launch_fwd32<HB, kPlanar, true, 0>(p, lds, N, stream);
        else launch_fwd32<HB, kPlanar, false, 0>(p, lds, N, stream);
    } else if (mode == kFused) {
        if (save) launch_fwd32<HB, kFused, true, 0>(p, lds, N, stream);
        else launch_fwd32<HB, kFused, false, 0>(p, lds, N, stream);
    } else if (act == 1) {
        if (save) launch_fwd32<HB, kRows, true, 1>(p, lds, N, stream);
        else launch_fwd32<HB, kRows, false, 1>(p, lds, N, stream);
    } else {
        if (save) launch_fwd32<HB, kRows, true, 0>(p, lds, N, stream);
        else launch_fwd32<HB, kRows, false, 0>(p, lds, N, stream);
    }
}

int fwd32_bias_base(const MlpShape& s) { return (rows_halves(s.hid, s.in, s.out, s.layers) * 2 + 15) & ~15; }
int fwd32_lds(const MlpShape& s) { return fwd32_bias_base(s) + 4 * ((s.layers - 1) * s.hid + up16(s.out)); }
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

bool mlp32_forward_supported(const MlpShape& s)
{
    if (s.layers < 2 || (s.hid != 32 && s.hid != 64 && s.hid != 128)) return false;
    if (s.in % 8 || s.in > 128 || s.out % 4 || s.out > 128) return false;
    return fwd32_lds(s) + kStaticLds <= max_lds_per_block();
}

void mlp32_forward(const MlpShape& s, const FwdInput& in, const __half* const* W, const float* const* B,
                   __half* const* acts, float* out, int N, int out_act, hipStream_t stream, const uint32_t* d_n)
{
    Fwd32Params p{};
    p.W = reinterpret_cast<const _Float16* const*>(W);
    p.B = B;
    p.acts = reinterpret_cast<_Float16* const*>(acts);
    p.d_n = d_n;
    p.in = s.in;
    p.out_dim = s.out;
    p.layers = s.layers;
    p.bias_base = fwd32_bias_base(s);
    const int lds = fwd32_lds(s);
    p.x_dim = in.x_dim > 0 ? in.x_dim : s.in;
    p.save_x0 = in.save_x0 ? 1 : 0;
    p.user_dim = in.user_dim > 0 ? in.user_dim : s.out;
    const bool save = acts != nullptr;
    const int act = in.table ? 0 : out_act;  // the hash-grid net has no output activation
    auto run = [&](int mode, int n0, int n) {
        p.N = n;
        const int xs = p.x_dim;
        if (in.x) p.x = reinterpret_cast<const _Float16*>(in.x) + (size_t)n0 * xs;
        p.vec_x = xs == s.in && aligned16(p.x);
        p.out = out ? out + (size_t)n0 * s.out : nullptr;
        p.vec_out = aligned16(p.out);
        p.user = in.user ? in.user + (size_t)n0 * p.user_dim : nullptr;
        p.vec_user = p.user_dim == s.out && aligned16(p.user);
        switch (s.hid) {
            case 32: pick_fwd32<1>(p, mode, save, act, lds, n, stream); break;
            case 64: pick_fwd32<2>(p, mode, save, act, lds, n, stream); break;
            default: pick_fwd32<4>(p, mode, save, act, lds, n, stream); break;
        }
    };
    if (!in.table) {
        run(kRows, 0, N);
        return;
    }
    const GridMeta& m = *in.meta;
    if (2 * m.numLevels != s.in) throw std::runtime_error("TinyMLPHashGrid: inputDim must equal 2 * numLevels");
    p.L = m.numLevels;
    p.T = m.tableSize;
    p.dense_start = m.denseLevelStart;
    p.table = reinterpret_cast<const _Float16*>(in.table);
    p.pos_stride = in.pos_stride;
    for (int l = 0; l < m.numLevels; l++) {
        p.scale[l] = m.scale[l];
        p.res[l] = m.res[l];
    }
    // Encodings first, level-major into scratch, then the net on them: the
    // encode then works on one table at a time per XCD.  One launch for
    // everything below kPlanarFrom samples, where its shorter chain wins, and
    // where no scratch is to be had.  Saved activations hold one batch, so
    // only inference is cut into pieces that bound the scratch.
    if (in.scratch && !d_n && N >= kPlanarFrom) {
        const int piece = save ? N : std::min(N, kPlanarPiece);
        std::lock_guard<std::mutex> lk(in.scratch->mutex());
        if (void* enc = in.scratch->try_get((size_t)piece * m.numLevels * 2 * sizeof(__half), stream)) {
            p.enc = static_cast<const _Float16*>(enc);
            p.plane = piece;
            for (int n0 = 0; n0 < N; n0 += piece) {
                const int n = std::min(piece, N - n0);
                hash_encode_planar(m, in.table, in.pos + (size_t)n0 * in.pos_stride, in.pos_stride,
                                   static_cast<__half*>(enc), piece, n, stream, nullptr, /*scattered=*/true);
                run(kPlanar, n0, n);
            }
            return;
        }
    }
    p.pos = in.pos;
    run(kFused, 0, N);
}

}  // namespace graft
