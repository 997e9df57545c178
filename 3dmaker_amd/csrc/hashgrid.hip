// Multiresolution hash grid on gfx950: standalone encode and the gradient
// scatter, plus the host-side level table shared with the fused forward.
//
//   encode   networkFusionHashtable.cu:441-551 (encode block of the fused kernel)
//   scatter  networkFusionBackwardHashtable.cu:783-910 (hashTableScatter_Backward)
//
// Thread mappings: the encode deals levels to XCDs (workgroup i runs on XCD
// i mod 8) and writes level-major encodings, from which rows are made where a
// caller wants them; the atomic scatter has one thread per (sample, group of 4
// levels), group fastest, and reads the gradient rows with 16-byte accesses.
#include "hashgrid.h"

#include "hash_encode.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <memory>
#include <mutex>

namespace graft {

int dense_level_start(int tableSize, int lowestSize, float b, int numLevels)
{
    // networkFusionHashtable.cu:367-377, host float arithmetic (libm).
    float inner = (std::cbrt(static_cast<float>(tableSize)) - 1.0f) / (float)lowestSize;
    float cont = std::log2(inner) / std::log2(b);
    int d = static_cast<int>(std::floor(cont)) + 1;
    return std::max(0, std::min(d, numLevels));
}

GridMeta make_grid_meta(int tableSize, int numLevels, float b, int lowestSize)
{
    if (numLevels < 1 || numLevels > kMaxLevels)
        throw std::runtime_error("TinyMLPHashGrid: numLevels must be in [1, 64]");
    if (tableSize < 2 || (tableSize & (tableSize - 1)))
        throw std::runtime_error("TinyMLPHashGrid: tableSize must be a power of two");
    GridMeta m{};
    m.numLevels = numLevels;
    m.tableSize = tableSize;
    m.denseLevelStart = dense_level_start(tableSize, lowestSize, b, numLevels);
    for (int l = 0; l < numLevels; l++) {
        m.scale[l] = (float)((double)lowestSize * std::pow((double)b, (double)l));
        m.res[l] = (int)std::floor(m.scale[l]);
        if (l < m.denseLevelStart) {
            const double cells = std::pow((double)m.res[l] + 1.0, 3.0);
            if (cells > (double)tableSize)
                throw std::runtime_error("TinyMLPHashGrid: dense level exceeds the table size");
        }
    }
    return m;
}

namespace {

struct GridKernelArgs {
    const uint32_t* d_n;   // nullable device-side sample count (<= N)
    int L, T, dense_start, pos_stride, N;
    float scale[kMaxLevels];
    int res[kMaxLevels];
};

__device__ __forceinline__ void stage_meta(const GridKernelArgs& a, float* ss, int* sr)
{
    for (int e = threadIdx.x; e < a.L; e += blockDim.x) {
        ss[e] = a.scale[e];
        sr[e] = a.res[e];
    }
    __syncthreads();
}

// gfx950 dispatches workgroup i to XCD i mod 8, and each XCD has its own 4 MB
// L2.  The encode gives each XCD its own levels, dealt in snake order, l -> l
// mod 8 for even l / 8 and 7 - l mod 8 for odd, which pairs level l with level
// 15 - l (a small dense level with a hashed one).
constexpr int kXcds = 8;
constexpr int kEncodeTile = 256;       // samples of one workgroup
constexpr int kEncodeTiles = 1 << 16;  // sample tiles of one launch: more are looped over

// Scattered points (SCATTERED): one workgroup encodes one level for one tile
// of 256 samples.  Workgroups of an XCD are ordered level by level, its finest
// first, so that the XCD works on one fp16 table at a time (2 MiB at T = 2^19,
// half of its L2).  What bounds it is the lines the corner gathers bring from
// the L2 into a CU's L1: a 128-byte line takes 1.8 to 2.4 cycles of a CU
// (measured with random gathers of 4, 8 and 16 bytes, which all cost the
// same), 64 lines per sample at 16 levels: 257 us for 2^20.
// Samples in ray or cell order (!SCATTERED) share most lines of the coarse
// levels with their neighbours; there a tile's workgroup takes the XCD's two
// levels of each 16 together, one position load and twice the gathers in
// flight.
// Measured at T = 2^19, b = 1.3819, level-major output, SCATTERED / not, and
// 2,048 looping workgroups with two levels per thread and 4-byte gathers
// before: 2^20 uniform points 285 / 350, before 354 us; 2^18 uniform 79 / 93,
// before 94 us; 2^18 ray-ordered 48.6 / 46.4, before 48.6 us; 2^20 ray-ordered
// 171 / 166, before 174 us.
// Output: PLANAR, enc[l][plane] feature pairs; else row-major enc[n][2L].
template <bool PLANAR, bool SCATTERED>
__global__ __launch_bounds__(kEncodeTile) void hash_encode_kernel(const GridKernelArgs a,
                                                                  const float* __restrict__ pos,
                                                                  const _Float16* __restrict__ table,
                                                                  _Float16* __restrict__ enc, int plane, int tiles)
{
    const int N = a.d_n ? min((int)*a.d_n, a.N) : a.N;
    const int x = blockIdx.x % kXcds, item = blockIdx.x / kXcds;
    const int groups = (a.L + kXcds - 1) / kXcds;
    const int k = SCATTERED ? item / tiles : 0;
    const uint32_t mask = (uint32_t)a.T - 1u;
    const int D = 2 * a.L;
    for (long long n = (long long)(item - k * tiles) * kEncodeTile + threadIdx.x; n < N;
         n += (long long)tiles * kEncodeTile) {
        const float* pp = pos + (size_t)n * a.pos_stride;
        const float px = pp[0], py = pp[1], pz = pp[2];
        auto level = [&](int g) {
            const int l = kXcds * g + ((g & 1) ? kXcds - 1 - x : x);
            if (l >= a.L) return;
            const float2 e = encode_level(px, py, pz, a.scale[l], a.res[l], l < a.dense_start, mask,
                                          table + (size_t)l * a.T * 2);
            const size_t at = PLANAR ? ((size_t)l * plane + n) * 2 : (size_t)n * D + 2 * l;
            *reinterpret_cast<h2*>(enc + at) = h2{to_h(e.x), to_h(e.y)};
        };
        if constexpr (SCATTERED) {
            level(groups - 1 - k);
        } else {
            for (int g = groups - 1; g >= 0; g -= 2) {
                level(g);
                if (g > 0) level(g - 1);
            }
        }
    }
}

// Level-major encodings to rows [n][2L]: four lanes per sample, four levels a
// lane at a time, so that a wave reads 64 contiguous bytes per level and
// stores whole rows (16 bytes per lane where rows allow it).  2^18 samples of
// 16 levels: 6 us.
__global__ __launch_bounds__(256) void encode_rows_kernel(const _Float16* __restrict__ planar, int plane, int L, int N,
                                                          _Float16* __restrict__ enc)
{
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    const int sub = threadIdx.x & 3;
    for (long long n = (long long)blockIdx.x * 64 + (threadIdx.x >> 2); n < N; n += (long long)gridDim.x * 64) {
        for (int l = 4 * sub; l < L; l += 16) {
            h2 v[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (l + j < L) v[j] = *reinterpret_cast<const h2*>(planar + ((size_t)(l + j) * plane + n) * 2);
            h2* dst = reinterpret_cast<h2*>(enc + (size_t)n * 2 * L + 2 * l);
            if (l + 4 <= L && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
                *reinterpret_cast<h8*>(dst) = h8{v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, v[3].x, v[3].y};
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (l + j < L) dst[j] = v[j];
            }
        }
    }
}

// grads[l][idx][f] += dL/denc[n][2l+f] * w_c for the 8 corners (scatter clamp).
//
// fp32 atomics on gfx950 are priced per cache-line request rather than per
// lane (measured: 4 atomics into one line cost about as much as one), so:
//  - a wave covers 16 consecutive samples at one level, four lanes per sample
//    for (x-corner xs, feature f).  The two x-neighbour corners of a level
//    differ only in the low bits of their index (dense: adjacent entries;
//    hashed: x0 ^ (x0 + 1) touches the low bits only, inside one 16-entry =
//    128-byte block 15 times in 16), so the quad's 4 atomics per y/z corner
//    usually share a line and each lane issues 4 atomics instead of 16;
//  - samples arrive ray by ray, closely spaced, so at coarse levels
//    consecutive samples share corners: a segmented sum over the 16 samples
//    merges equal addresses and only the last lane of each run issues the
//    atomic.  The products g_f * w_c are unchanged; only the order of the
//    fp32 additions differs (the reference's red.add order is unspecified).
__global__ __launch_bounds__(256) void hash_scatter_kernel(const GridKernelArgs a,
                                                           const float* __restrict__ pos,
                                                           const _Float16* __restrict__ denc,
                                                           float* __restrict__ grads)
{
    // This kernel's waves issue ahead of other kernels' waves on the same
    // SIMD (the side stream's work runs beside it): its atomic stream is the
    // step's critical path.
    __builtin_amdgcn_s_setprio(3);
    __shared__ float ss[kMaxLevels];
    __shared__ int sr[kMaxLevels];
    stage_meta(a, ss, sr);
    const uint32_t mask = (uint32_t)a.T - 1u;
    const int D = 2 * a.L;
    const int N = a.d_n ? min((int)*a.d_n, a.N) : a.N;
    const int lane = threadIdx.x & 63;
    const int s = lane >> 2, xs = (lane >> 1) & 1, f = lane & 1;
    const long long nwaves = (long long)((N + 15) / 16) * a.L;
    const long long wstride = ((long long)gridDim.x * blockDim.x) >> 6;
    for (long long w = ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 6; w < nwaves; w += wstride) {
        const int l = (int)(w % a.L);
        const int n = (int)((w / a.L) * 16 + s);
        const bool valid = n < N;
        Corners c;
        float gv = 0.0f;
        if (valid) {
            const float* pp = pos + (size_t)n * a.pos_stride;
            gv = (float)denc[(size_t)n * D + 2 * l + f];
            level_corners<true>(pp[0], pp[1], pp[2], ss[l], sr[l], l < a.dense_start, mask, c);
        }
        float* lvl = grads + (size_t)l * a.T * 2;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t A = valid ? c.idx[xs + 2 * q] + (uint32_t)f : 0xffffffffu;
            float v = valid ? gv * c.w[xs + 2 * q] : 0.0f;
            const uint32_t A_prev = __shfl_up(A, 4, 64);
            bool seen = (s == 0) || (A != A_prev);  // run head
            const bool head = seen;
#pragma unroll
            for (int d = 1; d < 16; d <<= 1) {
                const float vp = __shfl_up(v, 4 * d, 64);
                const int sp = __shfl_up((int)seen, 4 * d, 64);
                if (s >= d && !seen) {
                    v += vp;
                    seen = sp != 0;
                }
            }
            const int next_head = __shfl_down((int)head, 4, 64);
            const bool tail = (s == 15) || next_head;
            if (valid && tail) atomic_add_f32(lvl + A, v);
        }
    }
}

GridKernelArgs grid_args(const GridMeta& m, int N, int pos_stride)
{
    GridKernelArgs a{};
    a.L = m.numLevels;
    a.T = m.tableSize;
    a.dense_start = m.denseLevelStart;
    a.pos_stride = pos_stride;
    a.N = N;
    for (int l = 0; l < m.numLevels; l++) {
        a.scale[l] = m.scale[l];
        a.res[l] = m.res[l];
    }
    return a;
}

template <bool PLANAR, bool SCATTERED>
void launch_encode(const GridMeta& m, const __half* table, const float* pos, int pos_stride, __half* enc, int plane,
                   int N, hipStream_t stream, const uint32_t* d_n)
{
    GridKernelArgs a = grid_args(m, N, pos_stride);
    a.d_n = d_n;
    // With a count on the device N is only a bound, and each workgroup past the
    // count costs its dispatch (about 350 per us): ordered samples, where the
    // order of the levels does not matter, loop over at most 1,024 tiles then.
    const int tiles = std::min((N - 1) / kEncodeTile + 1, d_n && !SCATTERED ? 1024 : kEncodeTiles);
    const int groups = (m.numLevels + kXcds - 1) / kXcds;
    hipLaunchKernelGGL((hash_encode_kernel<PLANAR, SCATTERED>), dim3(kXcds * tiles * (SCATTERED ? groups : 1)),
                       dim3(kEncodeTile), 0, stream, a, pos, reinterpret_cast<const _Float16*>(table),
                       reinterpret_cast<_Float16*>(enc), plane, tiles);
    GRAFT_LAUNCH_CHECK();
}

}  // namespace

// Row-major output costs the encode a partial line per level and sample; from
// kRowsFromPlanar samples on, level-major encodings in the stream's scratch and
// a pass that turns them into rows are the faster way, kEncodePiece samples at
// a time so that what is kept has a bound.  The launches are enqueued under the
// scratch's lock, so that calls of several threads on one stream do not come
// between each other's.
void hash_encode(const GridMeta& m, const __half* table, const float* pos, int pos_stride,
                 __half* enc, int N, hipStream_t stream, const uint32_t* d_n, StreamScratch* scratch)
{
    if (N <= 0) return;
    if (pos_stride < 3) throw std::runtime_error("hash encode: position stride must be >= 3");
    constexpr int kRowsFromPlanar = 1 << 15;
    const std::shared_ptr<Workspace> ws = scratch && !d_n && N >= kRowsFromPlanar ? scratch->of(stream) : nullptr;
    if (ws) {
        const int D = 2 * m.numLevels, piece = std::min(N, kEncodePiece);
        std::lock_guard<std::mutex> lk(ws->mutex());
        if (void* planar = ws->try_get((size_t)piece * D * sizeof(__half))) {
            for (int n0 = 0; n0 < N; n0 += piece) {
                const int n = std::min(piece, N - n0);
                launch_encode<true, true>(m, table, pos + (size_t)n0 * pos_stride, pos_stride,
                                          static_cast<__half*>(planar), piece, n, stream, nullptr);
                hipLaunchKernelGGL(encode_rows_kernel, dim3((n + 63) / 64), dim3(256), 0, stream,
                                   static_cast<const _Float16*>(planar), piece, m.numLevels, n,
                                   reinterpret_cast<_Float16*>(enc) + (size_t)n0 * D);
                GRAFT_LAUNCH_CHECK();
            }
            return;
        }
    }
    launch_encode<false, true>(m, table, pos, pos_stride, enc, 0, N, stream, d_n);
}

void hash_encode_planar(const GridMeta& m, const __half* table, const float* pos, int pos_stride,
                        __half* enc, int plane, int N, hipStream_t stream, const uint32_t* d_n, bool scattered)
{
    if (N <= 0) return;
    if (pos_stride < 3) throw std::runtime_error("hash encode: position stride must be >= 3");
    if (plane < N) throw std::runtime_error("hash encode: plane stride below the sample count");
    if (scattered)
        launch_encode<true, true>(m, table, pos, pos_stride, enc, plane, N, stream, d_n);
    else
        launch_encode<true, false>(m, table, pos, pos_stride, enc, plane, N, stream, d_n);
}

void hash_scatter_atomic(const GridMeta& m, const __half* denc, const float* pos, int pos_stride,
                         float* grads, int N, hipStream_t stream, const uint32_t* d_n)
{
    if (N <= 0) return;
    if (pos_stride < 3) throw std::runtime_error("hash scatter: position stride must be >= 3");
    GridKernelArgs a = grid_args(m, N, pos_stride);
    a.d_n = d_n;
    // One workgroup per CU: the memory-side atomic rate, not the number of
    // waves issuing atomics, bounds this kernel (measured on a training step:
    // 1 block per CU is as fast as 16), and the idle CU slots then run the
    // side stream's work (next batch's compaction, occupancy refresh).
    const long long threads = (long long)((N + 15) / 16) * m.numLevels * 64;
    const int blocks = (int)std::max(1LL, std::min((threads + 255) / 256, (long long)num_cus()));
    hipLaunchKernelGGL(hash_scatter_kernel, dim3(blocks), dim3(256), 0, stream, a,
                       pos, reinterpret_cast<const _Float16*>(denc), grads);
    GRAFT_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// process-wide helpers
// ---------------------------------------------------------------------------

namespace {
std::mutex g_ws_mu;
int g_cus = 0;
int g_lds = 0;
}  // namespace

int max_lds_per_block()
{
    if (g_lds == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && n > 0)
            g_lds = n;
        else
            g_lds = 64 * 1024;
    }
    return g_lds;
}

Workspace::~Workspace()
{
    if (p_) (void)hipFree(p_);
}

void* Workspace::get(size_t bytes)
{
    if (bytes > bytes_) {
        if (p_) GRAFT_HIP_CHECK(hipFree(p_));
        p_ = nullptr;
        bytes_ = 0;
        const size_t nb = std::max(bytes, (size_t)1 << 16);
        GRAFT_HIP_CHECK(hipMalloc(&p_, nb));
        bytes_ = nb;
    }
    return p_;
}

void* Workspace::try_get(size_t bytes)
{
    if (bytes <= bytes_) return p_;
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (p_) (void)hipFree(p_);
    p_ = p;
    bytes_ = bytes;
    return p_;
}

std::shared_ptr<Workspace> StreamScratch::of(hipStream_t s)
{
    // hipStreamPerThread names another stream in every thread
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (s == hipStreamPerThread || hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return nullptr;
    }
    int dev = 0;
    GRAFT_HIP_CHECK(hipGetDevice(&dev));
    std::shared_ptr<Workspace> given_back;  // freed behind the lock
    std::lock_guard<std::mutex> lk(mu_);
    calls_++;
    auto at = held_.find({dev, s});
    if (at == held_.end()) {
        if (held_.size() >= kMost) {
            auto old = held_.begin();
            for (auto i = held_.begin(); i != held_.end(); ++i)
                if (i->second.used < old->second.used) old = i;
            if (calls_ - old->second.used <= kIdle) return nullptr;
            given_back = std::move(old->second.ws);
            held_.erase(old);
        }
        at = held_.emplace(std::make_pair(dev, s), Held{std::make_shared<Workspace>(), 0}).first;
    }
    at->second.used = calls_;
    return at->second.ws;
}

StreamScratch& launcher_encode_scratch()
{
    static StreamScratch* all = new StreamScratch();  // outlives static destructors
    return *all;
}

Workspace& stream_workspace(hipStream_t s)
{
    int dev = 0;
    GRAFT_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_ws_mu);
    static std::map<std::pair<int, hipStream_t>, std::unique_ptr<Workspace>>* cache =
        new std::map<std::pair<int, hipStream_t>, std::unique_ptr<Workspace>>();  // outlives static destructors
    auto& w = (*cache)[{dev, s}];
    if (!w) w.reset(new Workspace());
    return *w;
}

int num_cus()
{
    if (g_cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            g_cus = n;
        else
            g_cus = 256;
    }
    return g_cus;
}

}  // namespace graft
