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
#include "mlp32_lds.h"

#include "hash_encode.h"
#include "hashgrid.h"

#include <algorithm>
#include <type_traits>

namespace graft {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f4 mfma32(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ h8 h8zero()
{
    const _Float16 z = (_Float16)0.f;
    return h8{z, z, z, z, z, z, z, z};
}

// Copies every layer's W rows into LDS, zeros outside the matrix.  Each thread
// has up to 12 16-byte loads in flight; nothing branches around a load (a chunk
// outside the matrix reads its layer's first one): with a branch per chunk
// they came one after another, and 1,003 samples through 8-128-128-128-8 took
// 18.4 us instead of 11.4.  How many chunks a thread takes at a time follows the
// size of the nets, since a clamped chunk costs as much as one that is wanted:
// with 12 always, 200,000 samples through 16-32-8 took 12.7 us instead of 8.7 (9.3
// on 16x16x16 products), 65,537 forward and backward through 32-64-64-8 42.3
// instead of 40.2, 1,003 through 8-128-128-128-8 10.2 instead of 9.3.
// All threads call; ends with a barrier.
template <int HID, int BATCH>
__device__ __forceinline__ void stage_chunks(_Float16* sw, const _Float16* const* sW, bool vec, int base, int total,
                                             int in, int out, int layers)
{
    h8 v[BATCH];
    int dst[BATCH];
    bool ok[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; k++) {
        const Staged c = staged_chunk(min(base + k * 256 + (int)threadIdx.x, total - 1), HID, in, out, layers);
        dst[k] = c.dst;
        ok[k] = c.ok;
        const _Float16* src = sW[c.layer] + (c.ok ? c.at : 0);
        if (vec) {
            v[k] = *reinterpret_cast<const h8*>(src);
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) v[k][j] = src[j];
        }
    }
#pragma unroll
    for (int k = 0; k < BATCH; k++)
        if (base + k * 256 + (int)threadIdx.x < total)
            *reinterpret_cast<h8*>(sw + dst[k]) = ok[k] ? v[k] : h8zero();
}

template <int HID>
__device__ __forceinline__ void stage_rows(_Float16* sw, const _Float16* const* W, int in, int out, int layers,
                                           int last_rows)
{
    __shared__ const _Float16* sW[kMaxLayers];
    const int tid = threadIdx.x;
    if (tid < layers) sW[tid] = W[tid];
    __syncthreads();
    uintptr_t low = 0;
    for (int l = 0; l < layers; l++) low |= reinterpret_cast<uintptr_t>(sW[l]);
    const bool vec = __builtin_amdgcn_readfirstlane((int)(low & 15u)) == 0;
    const int total = staged_chunks(HID, in, layers, last_rows);
    for (int base = 0; base < total;) {
        const int left = (total - base + 255) >> 8;  // per thread
        if (left > 8) {
            stage_chunks<HID, 12>(sw, sW, vec, base, total, in, out, layers);
            base += 12 * 256;
        } else if (left > 4) {
            stage_chunks<HID, 8>(sw, sW, vec, base, total, in, out, layers);
            break;
        } else if (left > 2) {
            stage_chunks<HID, 4>(sw, sW, vec, base, total, in, out, layers);
            break;
        } else {
            stage_chunks<HID, 2>(sw, sW, vec, base, total, in, out, layers);
            break;
        }
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
    int row0;                  // the batch's first row in acts
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
// the caller's rows before, 58 us with that copy in it.
template <int HB, int NT, int MODE, bool SAVE, int OUT_ACT>
__global__ __launch_bounds__(256) void mlp32_fwd_kernel(const Fwd32Params p)
{
    constexpr int HID = 32 * HB;
    extern __shared__ __align__(16) unsigned char smem[];
    _Float16* sw = reinterpret_cast<_Float16*>(smem);
    float* sb = reinterpret_cast<float*>(smem + p.bias_base);
    // the first two biases of a thread are on their way while the weights are staged
    const int tid = threadIdx.x, nb = fwd32_biases(HID, p.out_dim, p.layers);
    auto bias = [&](int e) {
        const int l = min(e / HID, p.layers - 1), i = e - l * HID;
        const bool ok = e < nb && i < (l == p.layers - 1 ? p.out_dim : HID);
        const float v = p.B[l][ok ? i : 0];
        return ok ? v : 0.f;
    };
    const float b0 = bias(tid), b1 = bias(tid + 256);
    stage_rows<HID>(sw, p.W, p.in, p.out_dim, p.layers, fwd32_last_rows(p.out_dim));
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
    if constexpr (SAVE) act0 = p.acts[0] + (size_t)p.row0 * p.in;

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
            const _Float16* w = sw + row_base(HID, p.in, l) + fwd32_lane_row(true, r) * pitch + 8 * g;
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
            if constexpr (SAVE) act = p.acts[l + 1] + (size_t)p.row0 * HID;
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
        const bool pairs = fwd32_pairs(p.out_dim);
        const _Float16* w = sw + row_base(HID, p.in, l) + fwd32_lane_row(pairs, r) * pitch + 8 * g;
        const float* bl = sb + l * HID;
        const int OQ = fwd32_last_steps(p.out_dim);
        for (int q = 0; q < OQ; q++) {
#pragma unroll
            for (int m = 0; m < 2; m++) {
                if (m == 1 && !pairs) continue;
                const int col = fwd32_lane_col(pairs, q, m, g);
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

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------

constexpr int kBwdRows = 128;  // samples of a block's chunk: 32 per wave

struct Bwd32Params {
    const _Float16* dy;          // [N x out]
    const _Float16* const* acts; // device array: acts[0] = layer-0 input, acts[l] = H_l
    const _Float16* const* W;
    float* ws;                   // [gridDim.x][P] partial dW (all layers) then db
    _Float16* dx;                // nullable [N x in]
    const uint32_t* d_n;
    int N, in, out_dim, layers;
    int wofs[kMaxLayers], bofs[kMaxLayers];
    int P, pitch;                // pitch: halves of a row of the exchange buffers
    int g_base, x_base;          // their byte offsets in LDS
    int vec_dy;
};

// Transposing LDS read (16-bit): of the 4 x 16 halves that the 16 lanes of a
// group name (lane k: row k / 4, columns 4 (k % 4) ..), lane i gets column i.
typedef short s4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ h4 lds_tr(const _Float16* p)
{
    typedef __attribute__((address_space(3))) s4 lds_s4;
    return __builtin_bit_cast(h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p));
}
// Eight rows from p (this lane's row and column of lds_tr's 4 x 16) on: the
// lane's column of rows 0..7.
__device__ __forceinline__ h8 lds_tr8(const _Float16* p, int pitch)
{
    const h4 a = lds_tr(p), b = lds_tr(p + 4 * pitch);
    return h8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// A block takes 128 samples through all layers.  Per layer every wave puts the
// dL/dy and the input activations of its 32 samples into LDS as they lie (16
// bytes per lane); dW = dY^T X then takes its operands, samples along K, with
// the transposing LDS read, each wave owning a quarter of the layer's 16x16
// blocks over all 128 samples, and dX = dY W of the wave's own samples takes
// W^T from the weights' rows the same way.  db is one more column of ones.
// dW/db stay in registers until the block's last chunk; the next layer's (or
// chunk's) activations are loaded during the products.
// What is left is the bytes of dL/dy and activations (33 us for 2^18 samples
// of 64-64-64-64-64 at a large copy's rate) and two barriers per layer: 76 us,
// 150 with 2-byte transposing LDS writes and 16x16x16 products before; 65,537
// samples of 32-64-64-8 20 us, 37 before; 2^18 of 32-64-16 28 us, 33 before.
template <int HB, int LAYERS>
__global__ __launch_bounds__(256, HB == 1 ? 4 : HB == 2 ? 2 : 1) void mlp32_bwd_kernel(const Bwd32Params p)
{
    constexpr int HID = 32 * HB;
    constexpr int WO_H = HB == 1 ? 2 : 4, WI_H = 4 / WO_H;  // a hidden layer's waves along o and i
    constexpr int AH = 2 * HB / WO_H, BH = 2 * HB / WI_H;   // and the blocks of each
    constexpr int QW = AH * BH;
    extern __shared__ __align__(16) unsigned char smem[];
    _Float16* sw = reinterpret_cast<_Float16*>(smem);
    _Float16* sg = reinterpret_cast<_Float16*>(smem + p.g_base);
    _Float16* sx = reinterpret_cast<_Float16*>(smem + p.x_base);
    stage_rows<HID>(sw, p.W, p.in, p.out_dim, LAYERS, up32(p.out_dim));

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int N = p.d_n ? min((int)*p.d_n, p.N) : p.N;
    const int nchunks = (N + kBwdRows - 1) / kBwdRows;
    const int pitch = p.pitch;
    h8 ones;
#pragma unroll
    for (int j = 0; j < 8; j++) ones[j] = (_Float16)1.f;
    f4 dw[LAYERS][QW], db[LAYERS][AH];
#pragma unroll
    for (int l = 0; l < LAYERS; l++) {
#pragma unroll
        for (int k = 0; k < QW; k++) dw[l][k] = f4zero();
#pragma unroll
        for (int k = 0; k < AH; k++) db[l][k] = f4zero();
    }

    auto load = [&](const _Float16* src, int width, bool vec, int chunk, h8 (&V)[2][HB]) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int n = chunk * kBwdRows + (wave * 2 + t) * 16 + r;
#pragma unroll
            for (int b = 0; b < HB; b++) {
                V[t][b] = h8zero();
                const int col = 32 * b + 8 * g;
                if (n >= N || col >= width) continue;
                const _Float16* q = src + (size_t)n * width + col;
                if (vec) {
                    V[t][b] = *reinterpret_cast<const h8*>(q);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        if (col + j < width) V[t][b][j] = q[j];
                }
            }
        }
    };
    auto load_act = [&](int l, int chunk, h8 (&V)[2][HB]) {
        const _Float16* src = p.acts[l];
        load(src, l == 0 ? p.in : HID, (reinterpret_cast<uintptr_t>(src) & 15u) == 0, chunk, V);
    };

    h8 G[2][HB], X[2][HB];
    int chunk = blockIdx.x;
    if (chunk < nchunks) {
        load(p.dy, p.out_dim, p.vec_dy, chunk, G);
        load_act(LAYERS - 1, chunk, X);
    }
    for (; chunk < nchunks; chunk += gridDim.x) {
        const int next = chunk + gridDim.x;
        auto layer = [&](auto lc, f4 (&dwl)[QW], f4 (&dbl)[AH]) {
            constexpr int l = decltype(lc)::value;
            constexpr bool last = l == LAYERS - 1;
            const int KO = last ? (p.out_dim + 31) >> 5 : HB;  // 32-blocks of dL/dy
            const int KI = l == 0 ? (p.in + 31) >> 5 : HB;     // and of the input
            h8 Xn[2][HB], Gn[2][HB];
            if constexpr (l > 0) {
                load_act(l - 1, chunk, Xn);
            } else if (next < nchunks) {
                load_act(LAYERS - 1, next, Xn);
                load(p.dy, p.out_dim, p.vec_dy, next, Gn);
            }
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int row = ((wave * 2 + t) * 16 + r) * pitch + 8 * g;
#pragma unroll
                for (int b = 0; b < HB; b++) {
                    if (b < KO) *reinterpret_cast<h8*>(sg + row + 32 * b) = G[t][b];
                    if (b < KI) *reinterpret_cast<h8*>(sx + row + 32 * b) = X[t][b];
                }
            }
            __syncthreads();

            // dW, db: this wave's blocks (wo + WO a, wi + WI b) over the chunk's samples
            const int OB = last ? up16(p.out_dim) >> 4 : 2 * HB, IB = l == 0 ? up16(p.in) >> 4 : 2 * HB;
            const int WO = last ? min(OB, 4) : WO_H, WI = 4 / WO;
            const int wo = wave & (WO - 1), wi = wave / WO;
            const int NB = (IB + WI - 1) / WI;  // blocks of the wave along i
            const _Float16* tg = sg + (8 * g + (r >> 2)) * pitch + 4 * (r & 3);
            const _Float16* tx = sx + (8 * g + (r >> 2)) * pitch + 4 * (r & 3);
#pragma unroll 1
            for (int ks = 0; ks < kBwdRows / 32; ks++) {
                const int at = 32 * ks * pitch;
                if constexpr (!last) {
#pragma unroll
                    for (int a = 0; a < AH; a++) {
                        const h8 A = lds_tr8(tg + at + 16 * (wo + WO_H * a), pitch);
                        if (wi == 0) dbl[a] = mfma32(A, ones, dbl[a]);
#pragma unroll
                        for (int b = 0; b < BH; b++)
                            if (wi + WI_H * b < IB)
                                dwl[a * BH + b] = mfma32(A, lds_tr8(tx + at + 16 * (wi + WI_H * b), pitch), dwl[a * BH + b]);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < QW; k++) {
                        const int a = k / NB, b = k - a * NB;
                        if (wo + WO * a >= OB || wi + WI * b >= IB) continue;
                        const h8 A = lds_tr8(tg + at + 16 * (wo + WO * a), pitch);
                        dwl[k] = mfma32(A, lds_tr8(tx + at + 16 * (wi + WI * b), pitch), dwl[k]);
                    }
#pragma unroll
                    for (int a = 0; a < AH; a++)
                        if (wi == 0 && wo + WO * a < OB)
                            dbl[a] = mfma32(lds_tr8(tg + at + 16 * (wo + WO * a), pitch), ones, dbl[a]);
                }
            }
            // dX of this wave's 32 samples, rounded to fp16, masked by the input
            if (l > 0 || p.dx != nullptr) {
                const int wp = l == 0 ? 32 * KI + 8 : HID + 8;
                const _Float16* w = sw + row_base(HID, p.in, l) + (8 * g + (r >> 2)) * wp + 8 * (r & 3);
                h8 D[2][HB];
#pragma unroll
                for (int q = 0; q < HB; q++) {
                    if (q >= KI) continue;
                    f4 acc[2][2];
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int m = 0; m < 2; m++) acc[t][m] = f4zero();
#pragma unroll
                    for (int kb = 0; kb < HB; kb++) {
                        if (kb >= KO) continue;
#pragma unroll
                        for (int m = 0; m < 2; m++) {
                            const h8 A = lds_tr8(w + 32 * kb * wp + 32 * q + 4 * m, wp);
#pragma unroll
                            for (int t = 0; t < 2; t++) acc[t][m] = mfma32(A, G[t][kb], acc[t][m]);
                        }
                    }
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const _Float16 v = to_h(acc[t][j >> 2][j & 3]);
                            D[t][q][j] = l > 0 && !(X[t][q][j] > (_Float16)0.f) ? (_Float16)0.f : v;
                        }
                }
                if (l == 0) {
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        const int n = chunk * kBwdRows + (wave * 2 + t) * 16 + r;
#pragma unroll
                        for (int q = 0; q < HB; q++) {
                            const int col = 32 * q + 8 * g;
                            if (q < KI && n < N && col < p.in) st_row8(p.dx + (size_t)n * p.in + col, D[t][q]);
                        }
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int q = 0; q < HB; q++) Gn[t][q] = D[t][q];
                }
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int b = 0; b < HB; b++) {
                    G[t][b] = Gn[t][b];
                    X[t][b] = Xn[t][b];
                }
        };
        if constexpr (LAYERS > 3) layer(std::integral_constant<int, 3>{}, dw[3], db[3]);
        if constexpr (LAYERS > 2) layer(std::integral_constant<int, 2>{}, dw[2], db[2]);
        layer(std::integral_constant<int, 1>{}, dw[1], db[1]);
        layer(std::integral_constant<int, 0>{}, dw[0], db[0]);
    }

    float* dst = p.ws + (size_t)blockIdx.x * p.P;
#pragma unroll
    for (int l = 0; l < LAYERS; l++) {
        const bool last = l == LAYERS - 1;
        const int in_l = l == 0 ? p.in : HID, out_l = last ? p.out_dim : HID;
        const int OB = last ? up16(p.out_dim) >> 4 : 2 * HB, IB = l == 0 ? up16(p.in) >> 4 : 2 * HB;
        const int WO = last ? min(OB, 4) : WO_H, WI = 4 / WO;
        const int wo = wave & (WO - 1), wi = wave / WO;
        const int NB = last ? (IB + WI - 1) / WI : BH;
#pragma unroll
        for (int k = 0; k < QW; k++) {
            const int a = k / NB, b = k - a * NB;
            const int i = 16 * (wi + WI * b) + r;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int o = 16 * (wo + WO * a) + 4 * g + j;
                if (o < out_l && i < in_l) dst[p.wofs[l] + o * in_l + i] = dw[l][k][j];
            }
        }
#pragma unroll
        for (int a = 0; a < AH; a++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int o = 16 * (wo + WO * a) + 4 * g + j;
                if (wi == 0 && r == 0 && o < out_l) dst[p.bofs[l] + o] = db[l][a][j];
            }
        }
    }
}

// LDS of the backward: weights with the last layer's rows padded for the
// 32-wide products, then the two exchange buffers.
struct Bwd32Lds {
    int pitch, g_base, x_base, bytes;
};

Bwd32Lds bwd32_lds(const MlpShape& s)
{
    Bwd32Lds o{};
    o.pitch = s.hid + 8;
    o.g_base = (rows_halves(s.hid, s.in, s.layers, up32(s.out)) * 2 + 15) & ~15;
    o.x_base = o.g_base + kBwdRows * o.pitch * 2;
    o.bytes = o.x_base + kBwdRows * o.pitch * 2;
    return o;
}

template <int HB>
void launch_bwd32(const Bwd32Params& p, int lds, int blocks, hipStream_t stream)
{
    if (p.layers == 2) {
        hipLaunchKernelGGL((mlp32_bwd_kernel<HB, 2>), dim3(blocks), dim3(256), lds, stream, p);
    } else if constexpr (HB < 4) {
        if (p.layers == 3)
            hipLaunchKernelGGL((mlp32_bwd_kernel<HB, 3>), dim3(blocks), dim3(256), lds, stream, p);
        else
            hipLaunchKernelGGL((mlp32_bwd_kernel<HB, 4>), dim3(blocks), dim3(256), lds, stream, p);
    }
    GRAFT_LAUNCH_CHECK();
}

}  // namespace

bool mlp32_forward_supported(const MlpShape& s)
{
    if (s.layers < 2 || (s.hid != 32 && s.hid != 64 && s.hid != 128)) return false;
    if (s.in % 8 || s.in > 128 || s.out % 4 || s.out > 128) return false;
    return fwd32_lds(s.in, s.hid, s.out, s.layers) + kStaticLds <= max_lds_per_block();
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
    p.bias_base = fwd32_bias_base(s.in, s.hid, s.out, s.layers);
    const int lds = fwd32_lds(s.in, s.hid, s.out, s.layers);
    p.x_dim = in.x_dim > 0 ? in.x_dim : s.in;
    p.save_x0 = in.save_x0 ? 1 : 0;
    p.user_dim = in.user_dim > 0 ? in.user_dim : s.out;
    const bool save = acts != nullptr;
    const int act = in.table ? 0 : out_act;  // the hash-grid net has no output activation
    auto run = [&](int mode, int n0, int n) {
        p.N = n;
        p.row0 = n0;
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
    // where no scratch is to be had.  Pieces of kEncodePiece bound the scratch.
    const std::shared_ptr<Workspace> ws = in.scratch && !d_n && N >= kPlanarFrom ? in.scratch->of(stream) : nullptr;
    if (ws) {
        const int piece = std::min(N, kEncodePiece);
        std::lock_guard<std::mutex> lk(ws->mutex());
        if (void* enc = ws->try_get((size_t)piece * m.numLevels * 2 * sizeof(__half))) {
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

// Widths up to the hidden one (32 at least) at both ends, and layers whose
// dW fits the registers: four of width 64, two of 128.  What lies outside is
// mlp.hip's.
bool mlp32_backward_supported(const MlpShape& s)
{
    if (s.hid != 32 && s.hid != 64 && s.hid != 128) return false;
    if (s.layers < 2 || s.layers > (s.hid == 128 ? 2 : 4)) return false;
    if (s.in % 8 || up32(s.in) > s.hid || s.out % 4 || up32(s.out) > s.hid) return false;
    const int ob = up16(s.out) / 16;
    if (ob & (ob - 1)) return false;
    return bwd32_lds(s).bytes + kStaticLds <= max_lds_per_block();
}

int mlp32_backward(const MlpShape& s, const Mlp32Backward& a, int N, hipStream_t stream)
{
    const Bwd32Lds lds = bwd32_lds(s);
    const int nchunks = (N + kBwdRows - 1) / kBwdRows;
    const int per_cu = std::max(1, std::min(s.hid == 32 ? 4 : 2, max_lds_per_block() / (lds.bytes + kStaticLds)));
    const int blocks = std::max(1, std::min(nchunks, num_cus() * per_cu));
    Bwd32Params p{};
    p.dy = reinterpret_cast<const _Float16*>(a.dy);
    p.acts = reinterpret_cast<const _Float16* const*>(a.acts);
    p.W = reinterpret_cast<const _Float16* const*>(a.W);
    p.dx = reinterpret_cast<_Float16*>(a.dx);
    p.d_n = a.d_n;
    p.N = N;
    p.in = s.in;
    p.out_dim = s.out;
    p.layers = s.layers;
    for (int l = 0; l < s.layers; l++) {
        p.wofs[l] = a.wofs[l];
        p.bofs[l] = a.bofs[l];
    }
    p.P = a.P;
    p.pitch = lds.pitch;
    p.g_base = lds.g_base;
    p.x_base = lds.x_base;
    p.vec_dy = s.out % 8 == 0 && aligned16(a.dy);
    p.ws = static_cast<float*>(a.ws->get((size_t)blocks * a.P * sizeof(float)));
    switch (s.hid) {
        case 32: launch_bwd32<1>(p, lds.bytes, blocks, stream); break;
        case 64: launch_bwd32<2>(p, lds.bytes, blocks, stream); break;
        default: launch_bwd32<4>(p, lds.bytes, blocks, stream); break;
    }
    return blocks;
}

}  // namespace graft
