// ops.hip -- the reference's per-op inference kernels
// (include/spbitnet/inference_kernels.h:14-87, src/kernels/inference_kernels.cu)
// as C-ABI entry points for fp16 and bf16 storage, for callers that keep the
// reference engine's op-by-op dataflow.  The fused decode engine (engine.hip)
// does not call these; they are the drop-in replacements of the individual
// wrappers.
//
// Semantics follow the reference kernels (formula, operation order, storage
// type of every output); arithmetic is float32.  Differences by design:
// 1/sqrt is correctly rounded where the reference uses rsqrtf, and reductions
// use wave-64 trees.  Shapes are validated on the host; every kernel bounds-
// checks its own indices.
#include <algorithm>

#include "common.hpp"
#include "spbitnet_amd.h"

namespace spb {
namespace {

constexpr int kOpBlock = 256;
constexpr int kNormBlock = 1024;

template <int kCtrl>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kCtrl, 0xF, 0xF, true));
}

__device__ __forceinline__ float lane_f(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Wave-64 sum (pairwise tree over adjacent lanes; every lane gets the result).
__device__ __forceinline__ float wsum(float v) {
    v += dpp_f<0xB1>(v);
    v += dpp_f<0x4E>(v);
    v += dpp_f<0x141>(v);
    v += dpp_f<0x140>(v);
    return (lane_f(v, 0) + lane_f(v, 16)) + (lane_f(v, 32) + lane_f(v, 48));
}

__device__ __forceinline__ float wmax(float v) {
    v = fmaxf(v, dpp_f<0xB1>(v));
    v = fmaxf(v, dpp_f<0x4E>(v));
    v = fmaxf(v, dpp_f<0x141>(v));
    v = fmaxf(v, dpp_f<0x140>(v));
    return fmaxf(fmaxf(lane_f(v, 0), lane_f(v, 16)), fmaxf(lane_f(v, 32), lane_f(v, 48)));
}

template <int kThreads, bool kMax>
__device__ __forceinline__ float block_reduce(float v, float* slot) {
    v = kMax ? wmax(v) : wsum(v);
    if ((threadIdx.x & (kWave - 1)) == 0) slot[threadIdx.x / kWave] = v;
    __syncthreads();
    float s = slot[0];
#pragma unroll
    for (int w = 1; w < kThreads / kWave; ++w) s = kMax ? fmaxf(s, slot[w]) : s + slot[w];
    return s;
}

struct F32 {
    static __device__ __forceinline__ float to_float(float v) { return v; }
};

// rms_norm_kernel / rms_norm_f32in_kernel (inference_kernels.cu:15-56, 418-455):
// y = T((x * inv) * w), inv = 1 / sqrt(mean(x^2) + eps).  One block; input
// and output may alias (each element is read before the thread that reads
// it writes it).
template <class T, class In, class InT>
__global__ __launch_bounds__(kNormBlock) void rms_norm_kernel(const InT* x, const float* w,
                                                              uint16_t* y, int n, float eps) {
    __shared__ float slot[kNormBlock / kWave];
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += kNormBlock) {
        const float v = In::to_float(x[i]);
        ss = fmaf(v, v, ss);
    }
    ss = block_reduce<kNormBlock, false>(ss, slot);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(n) + eps);
    __syncthreads();  // every thread has read its inputs before any output aliasing them
    for (int i = threadIdx.x; i < n; i += kNormBlock)
        y[i] = T::from_float((In::to_float(x[i]) * inv) * w[i]);
}

// rope_kernel (inference_kernels.cu:185-206): pair (2i, 2i+1) of each head
// rotated by angle pos * theta^(-2i/hd), in place.
template <class T>
__global__ __launch_bounds__(kOpBlock) void rope_kernel(uint16_t* v, int nheads, int hd, int pos,
                                                        float theta) {
    const int t = blockIdx.x * kOpBlock + threadIdx.x;
    const int half = hd / 2;
    if (t >= nheads * half) return;
    const int head = t / half, pair = t - head * half;
    const float freq =
        1.0f / powf(theta, static_cast<float>(2 * pair) / static_cast<float>(hd));
    const float angle = static_cast<float>(pos) * freq;
    float s, c;
    sincosf(angle, &s, &c);
    const int idx = head * hd + 2 * pair;
    const float x0 = T::to_float(v[idx]), x1 = T::to_float(v[idx + 1]);
    v[idx] = T::from_float(x0 * c - x1 * s);
    v[idx + 1] = T::from_float(x0 * s + x1 * c);
}

// scatter_kv_kernel (inference_kernels.cu:215-227)
__global__ __launch_bounds__(kOpBlock) void scatter_kv_kernel(const uint16_t* src, uint16_t* cache,
                                                              int nkv, int hd, int max_seq,
                                                              int pos) {
    const int t = blockIdx.x * kOpBlock + threadIdx.x;
    if (t >= nkv * hd) return;
    const int h = t / hd, d = t - h * hd;
    cache[(static_cast<long>(h) * max_seq + pos) * hd + d] = src[t];
}

// attention_scores_kernel (inference_kernels.cu:241-275): one wave per
// (position, head); lanes over head_dim; GQA kv = h * nkv / nh.
template <class T>
__global__ __launch_bounds__(kOpBlock) void attention_scores_kernel(
    const uint16_t* Q, const uint16_t* K, float* scores, int nh, int nkv, int hd, int max_seq,
    int seq_len, float scale) {
    const int lane = threadIdx.x & (kWave - 1);
    const int j = blockIdx.x * (kOpBlock / kWave) + threadIdx.x / kWave;
    const int h = blockIdx.y;
    if (j >= seq_len) return;
    const int kvh = h * nkv / nh;
    const uint16_t* q = Q + static_cast<long>(h) * hd;
    const uint16_t* k = K + (static_cast<long>(kvh) * max_seq + j) * hd;
    float acc = 0.0f;
    for (int d = lane; d < hd; d += kWave) acc = fmaf(T::to_float(q[d]), T::to_float(k[d]), acc);
    acc = wsum(acc);
    if (lane == 0) scores[static_cast<long>(h) * max_seq + j] = acc * scale;
}

// Eight 16-bit values of a 16-byte load.
template <class T>
__device__ __forceinline__ void unpack8(const uint4 r, float (&f)[8]) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[2 * k] = T::to_float(static_cast<uint16_t>(w[k] & 0xFFFFu));
        f[2 * k + 1] = T::to_float(static_cast<uint16_t>(w[k] >> 16));
    }
}

// The q heads of kv head k: [first_head(k), first_head(k + 1)), those with
// h * nkv / nh == k.
__device__ __forceinline__ int first_head(int k, int nh, int nkv) {
    return static_cast<int>((static_cast<long>(k) * nh + nkv - 1) / nkv);
}

// The same scores for head_dim 8 L, L = 4, 8, 16 or 32, and 16-byte aligned
// rows: L lanes take a K row, 16 bytes each, once for `per` q heads of its kv
// head (blockIdx.z: which).  A launch is one round trip per block: the kernel
// above reads 2 bytes per lane and every K row once per q head (20 heads on 5,
// head_dim 128, 2500 positions: 9.2 us, 3.5 us with this one).
template <class T, int L>
__global__ __launch_bounds__(kOpBlock) void attention_scores_rows_kernel(
    const uint16_t* Q, const uint16_t* K, float* scores, int nh, int nkv, int max_seq,
    int seq_len, float scale, int per) {
    const int c = threadIdx.x % L, kvh = blockIdx.y;
    const int j = blockIdx.x * (kOpBlock / L) + threadIdx.x / L;
    const int jr = j < seq_len ? j : seq_len - 1;
    float k[8];
    unpack8<T>(reinterpret_cast<const uint4*>(K)[(static_cast<long>(kvh) * max_seq + jr) * L + c],
               k);
    const int h0 = first_head(kvh, nh, nkv) + blockIdx.z * per;
    const int end = first_head(kvh + 1, nh, nkv), h1 = h0 + per < end ? h0 + per : end;
    for (int h = h0; h < h1; ++h) {
        float q[8], acc = 0.0f;
        unpack8<T>(reinterpret_cast<const uint4*>(Q)[static_cast<long>(h) * L + c], q);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = fmaf(q[e], k[e], acc);
        acc += dpp_f<0xB1>(acc);
        acc += dpp_f<0x4E>(acc);
        if (L >= 8) acc += dpp_f<0x141>(acc);
        if (L >= 16) acc += dpp_f<0x140>(acc);
        if (L >= 32) acc += __shfl_xor(acc, 16, kWave);
        if (c == 0 && j < seq_len) scores[static_cast<long>(h) * max_seq + j] = acc * scale;
    }
}

// softmax_kernel (inference_kernels.cu:283-339): per head, in place over the
// first seq_len entries: max, exp, sum, multiply by 1/sum.
__global__ __launch_bounds__(kNormBlock) void softmax_kernel(float* scores, int max_seq,
                                                             int seq_len) {
    __shared__ float slot[2][kNormBlock / kWave];
    float* hs = scores + static_cast<long>(blockIdx.x) * max_seq;
    float m = -INFINITY;
    for (int j = threadIdx.x; j < seq_len; j += kNormBlock) m = fmaxf(m, hs[j]);
    m = block_reduce<kNormBlock, true>(m, slot[0]);
    float s = 0.0f;
    for (int j = threadIdx.x; j < seq_len; j += kNormBlock) {
        const float e = expf(hs[j] - m);
        hs[j] = e;
        s += e;
    }
    s = block_reduce<kNormBlock, false>(s, slot[1]);
    const float inv = 1.0f / s;
    for (int j = threadIdx.x; j < seq_len; j += kNormBlock) hs[j] *= inv;
}

// The same, operation for operation, for up to E * 1024 entries, which stay in
// registers between one read and one write (20 heads, 2500 entries: 4.6 -> 3.3 us).
template <int E>
__global__ __launch_bounds__(kNormBlock) void softmax_regs_kernel(float* scores, int max_seq,
                                                                  int seq_len) {
    __shared__ float slot[2][kNormBlock / kWave];
    float* hs = scores + static_cast<long>(blockIdx.x) * max_seq;
    float v[E], m = -INFINITY;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        const int j = threadIdx.x + k * kNormBlock;
        v[k] = j < seq_len ? hs[j] : -INFINITY;
    }
#pragma unroll
    for (int k = 0; k < E; ++k) m = fmaxf(m, v[k]);
    m = block_reduce<kNormBlock, true>(m, slot[0]);
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        const int j = threadIdx.x + k * kNormBlock;
        v[k] = expf(v[k] - m);
        if (j < seq_len) s += v[k];
    }
    s = block_reduce<kNormBlock, false>(s, slot[1]);
    const float inv = 1.0f / s;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        const int j = threadIdx.x + k * kNormBlock;
        if (j < seq_len) hs[j] = v[k] * inv;
    }
}

// attention_output_kernel (inference_kernels.cu:350-371):
// out[h][d] = sum_j score[h][j] * V[kv_h][j][d].  One block per head; wave w
// takes positions w, w + 4, ...; lane d, d + 64, ...; wave partials summed
// in LDS (head_dim <= 256).
template <class T>
__global__ __launch_bounds__(kOpBlock) void attention_output_kernel(
    const float* scores, const uint16_t* V, uint16_t* out, int nh, int nkv, int hd, int max_seq,
    int seq_len) {
    __shared__ float part[kOpBlock / kWave][256];
    const int h = blockIdx.x, lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int kvh = h * nkv / nh;
    const float* p = scores + static_cast<long>(h) * max_seq;
    const uint16_t* v = V + static_cast<long>(kvh) * max_seq * hd;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int j = wave; j < seq_len; j += kOpBlock / kWave) {
        const float pj = p[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = lane + r * kWave;
            if (d < hd) acc[r] = fmaf(pj, T::to_float(v[static_cast<long>(j) * hd + d]), acc[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int d = lane + r * kWave;
        if (d < hd) part[wave][d] = acc[r];
    }
    __syncthreads();
    for (int d = threadIdx.x; d < hd; d += kOpBlock) {
        float s = part[0][d];
#pragma unroll
        for (int w = 1; w < kOpBlock / kWave; ++w) s += part[w][d];
        out[static_cast<long>(h) * hd + d] = T::from_float(s);
    }
}

// The same sums for head_dim a multiple of 8 and 16-byte aligned rows.  One
// block per 8 dims, kv head and up to NH of its q heads (blockIdx.z): thread t
// takes positions t, t + 512, ... with one 16-byte V read for all of the
// block's heads.  The caller has no room for partial sums, so positions cannot
// go to different blocks; dims can (head_dim 128 and 5 kv heads: 80 blocks of
// 8 waves instead of 20 of 4 that walked over the positions with 2-byte loads:
// 2500 positions 238 us -> 7.1 us, a chain of one V round trip and the sums).
constexpr int kOutBlock = 512;
template <class T, int NH>
__global__ __launch_bounds__(kOutBlock) void attention_output_cols_kernel(
    const float* scores, const uint16_t* V, uint16_t* out, int nh, int nkv, int hd, int max_seq,
    int seq_len) {
    constexpr int kRows = kOutBlock / 16;  // 16-lane rows, one partial sum each
    __shared__ float part[NH * 8][kRows + 1];
    const int tid = threadIdx.x, u = blockIdx.x, kvh = blockIdx.y;
    const int h0 = first_head(kvh, nh, nkv) + blockIdx.z * NH;
    const int h1 = first_head(kvh + 1, nh, nkv);
    if (h0 >= h1) return;  // uniform
    const uint4* v = reinterpret_cast<const uint4*>(V) + static_cast<long>(kvh) * max_seq * (hd / 8) + u;
    const float* p[NH];
#pragma unroll
    for (int g = 0; g < NH; ++g)
        p[g] = scores + static_cast<long>(h0 + g < h1 ? h0 + g : h0) * max_seq;
    float acc[NH][8];
#pragma unroll
    for (int g = 0; g < NH; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] = 0.0f;
    constexpr int kAhead = 4;  // positions of a thread in flight
    for (int j0 = tid; j0 < seq_len; j0 += kAhead * kOutBlock) {
        uint4 w[kAhead];
        float pj[kAhead][NH];
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const int j = j0 + a * kOutBlock;
            if (j < seq_len) {
                w[a] = v[static_cast<long>(j) * (hd / 8)];
#pragma unroll
                for (int g = 0; g < NH; ++g) pj[a][g] = p[g][j];
            }
        }
#pragma unroll
        for (int a = 0; a < kAhead; ++a)
            if (j0 + a * kOutBlock < seq_len) {
                float f[8];
                unpack8<T>(w[a], f);
#pragma unroll
                for (int g = 0; g < NH; ++g)
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[g][e] = fmaf(pj[a][g], f[e], acc[g][e]);
            }
    }
    // the 16 lanes of a row hold a value's row sum after four exchanges; lane
    // i of the row keeps values i and 16 + i
    constexpr int kKeep = (NH * 8 + 15) / 16;
    float keep[kKeep];
#pragma unroll
    for (int i = 0; i < NH * 8; ++i) {
        float s = acc[i / 8][i % 8];
        s += dpp_f<0xB1>(s);
        s += dpp_f<0x4E>(s);
        s += dpp_f<0x141>(s);
        s += dpp_f<0x140>(s);
        if (i % 16 == 0 || (tid & 15) == i % 16) keep[i / 16] = s;
    }
#pragma unroll
    for (int i = 0; i < kKeep; ++i) {
        const int val = 16 * i + (tid & 15);
        if (val < NH * 8) part[val][tid >> 4] = keep[i];
    }
    __syncthreads();
    // 16 lanes per value: 32 partial sums
    const int val = tid >> 4, i = tid & 15;
    if (val < NH * 8) {  // whole 16-lane rows
        float s = part[val][i] + part[val][16 + i];
        s += dpp_f<0xB1>(s);
        s += dpp_f<0x4E>(s);
        s += dpp_f<0x141>(s);
        s += dpp_f<0x140>(s);
        const int h = h0 + val / 8;
        if (i == 0 && h < h1) out[static_cast<long>(h) * hd + 8 * u + val % 8] = T::from_float(s);
    }
}

// relu2_mul_kernel / relu2_mul_f32_kernel (inference_kernels.cu:380-410)
template <class T, bool kF32Out>
__global__ __launch_bounds__(kOpBlock) void relu2_mul_kernel(const uint16_t* g, const uint16_t* u,
                                                             void* out, long n) {
    for (long i = static_cast<long>(blockIdx.x) * kOpBlock + threadIdx.x; i < n;
         i += static_cast<long>(gridDim.x) * kOpBlock) {
        const float r = fmaxf(0.0f, T::to_float(g[i]));
        const float v = (r * r) * T::to_float(u[i]);
        if (kF32Out)
            static_cast<float*>(out)[i] = v;
        else
            static_cast<uint16_t*>(out)[i] = T::from_float(v);
    }
}

// float_to_half_kernel (inference_kernels.cu:460-466)
template <class T>
__global__ __launch_bounds__(kOpBlock) void float_to_16_kernel(const float* x, uint16_t* y, long n) {
    for (long i = static_cast<long>(blockIdx.x) * kOpBlock + threadIdx.x; i < n;
         i += static_cast<long>(gridDim.x) * kOpBlock)
        y[i] = T::from_float(x[i]);
}

// residual_add_kernel (inference_kernels.cu:471-479): T(float(a) + float(b))
template <class T>
__global__ __launch_bounds__(kOpBlock) void residual_add_kernel(const uint16_t* a, const uint16_t* b,
                                                                uint16_t* y, long n) {
    for (long i = static_cast<long>(blockIdx.x) * kOpBlock + threadIdx.x; i < n;
         i += static_cast<long>(gridDim.x) * kOpBlock)
        y[i] = T::from_float(T::to_float(a[i]) + T::to_float(b[i]));
}

// half_gemv_kernel (inference_kernels.cu:488-531): y[r] = sum_c W[r][c] x[c]
// in float32, one wave per row; 16-byte chunks when rows are 16-byte aligned.
template <class T>
__global__ __launch_bounds__(kOpBlock) void gemv16_kernel(const uint16_t* W, const uint16_t* x,
                                                          float* y, int rows, int cols,
                                                          bool vec) {
    const int lane = threadIdx.x & (kWave - 1);
    const long r = static_cast<long>(blockIdx.x) * (kOpBlock / kWave) + threadIdx.x / kWave;
    if (r >= rows) return;
    const uint16_t* w = W + r * cols;
    float acc = 0.0f;
    int tail = 0;
    if (vec) {
        const int nch = cols >> 3;
        for (int c = lane; c < nch; c += kWave) {
            const uint4 a = reinterpret_cast<const uint4*>(w)[c];
            const uint4 b = reinterpret_cast<const uint4*>(x)[c];
            const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                acc = fmaf(T::to_float(static_cast<uint16_t>(aw[k] & 0xFFFFu)),
                           T::to_float(static_cast<uint16_t>(bw[k] & 0xFFFFu)), acc);
                acc = fmaf(T::to_float(static_cast<uint16_t>(aw[k] >> 16)),
                           T::to_float(static_cast<uint16_t>(bw[k] >> 16)), acc);
            }
        }
        tail = nch << 3;
    }
    for (int c = tail + lane; c < cols; c += kWave) acc = fmaf(T::to_float(w[c]), T::to_float(x[c]), acc);
    acc = wsum(acc);
    if (lane == 0) y[r] = acc;
}

// Greedy token pick: index of the maximum (lowest index among equal maxima,
// as std::max_element in src/main.cpp:194-200); NaN entries never win.
__global__ __launch_bounds__(kNormBlock) void argmax_kernel(const float* x, int n, int* out) {
    __shared__ float sv[kNormBlock / kWave];
    __shared__ int si[kNormBlock / kWave];
    float b = -INFINITY;
    int bi = 0x7FFFFFFF;
    for (int i = threadIdx.x; i < n; i += kNormBlock)
        if (x[i] > b) {  // ascending per thread: strict > keeps the first
            b = x[i];
            bi = i;
        }
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const float ov = __shfl_xor(b, off, kWave);
        const int oi = __shfl_xor(bi, off, kWave);
        if (ov > b || (ov == b && oi < bi)) {
            b = ov;
            bi = oi;
        }
    }
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    if (lane == 0) {
        sv[wave] = b;
        si[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kNormBlock / kWave; ++w)
            if (sv[w] > b || (sv[w] == b && si[w] < bi)) {
                b = sv[w];
                bi = si[w];
            }
        *out = bi == 0x7FFFFFFF ? 0 : bi;
    }
}

int grid_for(long n) {
    long g = (n + kOpBlock - 1) / kOpBlock;
    return static_cast<int>(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <class T, class In, class InT>
int rms_norm(const char* fn, const InT* x, const float* w, uint16_t* y, int n, float eps,
             spb_stream_t s) {
    clear_error();
    if (n < 0) return invalid("%s: negative size", fn);
    if (n == 0) return 0;
    if (!x || !w || !y) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL((rms_norm_kernel<T, In, InT>), dim3(1), dim3(kNormBlock), 0, as_stream(s),
                       x, w, y, n, eps);
    return launch_status(fn);
}

template <class T>
int rope(const char* fn, uint16_t* v, int nh, int hd, int pos, float theta, spb_stream_t s) {
    clear_error();
    if (nh < 0 || hd < 0 || pos < 0) return invalid("%s: negative argument", fn);
    if (hd % 2) return invalid("%s: head_dim must be even", fn);
    if (nh == 0 || hd == 0) return 0;
    if (!v) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL(rope_kernel<T>, dim3(grid_for(static_cast<long>(nh) * hd / 2)),
                       dim3(kOpBlock), 0, as_stream(s), v, nh, hd, pos, theta);
    return launch_status(fn);
}

int check_attn(const char* fn, int nh, int nkv, int hd, int max_seq, int seq_len) {
    if (nh <= 0 || nkv <= 0 || hd <= 0 || max_seq <= 0)
        return invalid("%s: non-positive dimension", fn);
    if (seq_len < 0 || seq_len > max_seq) return invalid("%s: seq_len outside [0, max_seq]", fn);
    if (nkv > nh) return invalid("%s: more kv heads than heads", fn);
    return 0;
}

// A block's q heads go one after the other, so they are spread over blocks (z)
// until there are 4 blocks per CU.  us, general kernel / all heads in a block /
// this: 64 heads on 1, head_dim 128, 1 / 200 / 1000 / 8192 positions 2.1 / 12.7 /
// 2.1, 3.2 / 15.1 / 2.5, 8.3 / 14.6 / 3.2, 52 / 15.6 / 9.2; 8 on 1, 1 / 1000 / 4096
// 2.0 / 3.0 / 2.1, 2.8 / 3.4 / 2.2, 5.2 / 3.5 / 2.8; 20 on 5, 1 / 200 / 2500 2.1 /
// 2.6 / 2.2, 2.4 / 2.7 / 2.2, 7.1 / 3.1 / 3.1.
dim3 scores_rows_grid(int row_blocks, int nh, int nkv, int* per) {
    const int group = (nh + nkv - 1) / nkv;  // the most q heads of a kv head
    const long blocks = static_cast<long>(row_blocks) * nkv;
    const long want = std::min<long>(group, std::max(1L, 4L * device_cu_count() / blocks));
    *per = static_cast<int>((group + want - 1) / want);
    return dim3(row_blocks, nkv, (group + *per - 1) / *per);
}

template <class T>
int attention_scores(const char* fn, const uint16_t* Q, const uint16_t* K, float* sc, int nh,
                     int nkv, int hd, int max_seq, int seq_len, float scale, spb_stream_t s) {
    clear_error();
    if (int e = check_attn(fn, nh, nkv, hd, max_seq, seq_len)) return e;
    if (seq_len == 0) return 0;
    if (!Q || !K || !sc) return invalid("%s: null pointer", fn);
    if (al16(Q) && al16(K) && (hd == 32 || hd == 64 || hd == 128 || hd == 256)) {
        const int rows = kOpBlock / (hd / 8);
        int per = 1;
        const dim3 grid = scores_rows_grid((seq_len + rows - 1) / rows, nh, nkv, &per);
        switch (hd) {
        case 32: hipLaunchKernelGGL((attention_scores_rows_kernel<T, 4>), grid, dim3(kOpBlock), 0, as_stream(s), Q, K, sc, nh, nkv, max_seq, seq_len, scale, per); break;
        case 64: hipLaunchKernelGGL((attention_scores_rows_kernel<T, 8>), grid, dim3(kOpBlock), 0, as_stream(s), Q, K, sc, nh, nkv, max_seq, seq_len, scale, per); break;
        case 128: hipLaunchKernelGGL((attention_scores_rows_kernel<T, 16>), grid, dim3(kOpBlock), 0, as_stream(s), Q, K, sc, nh, nkv, max_seq, seq_len, scale, per); break;
        default: hipLaunchKernelGGL((attention_scores_rows_kernel<T, 32>), grid, dim3(kOpBlock), 0, as_stream(s), Q, K, sc, nh, nkv, max_seq, seq_len, scale, per); break;
        }
        return launch_status(fn);
    }
    const dim3 grid((seq_len + kOpBlock / kWave - 1) / (kOpBlock / kWave), nh);
    hipLaunchKernelGGL(attention_scores_kernel<T>, grid, dim3(kOpBlock), 0, as_stream(s), Q, K, sc,
                       nh, nkv, hd, max_seq, seq_len, scale);
    return launch_status(fn);
}

template <class T>
int attention_output(const char* fn, const float* sc, const uint16_t* V, uint16_t* out, int nh,
                     int nkv, int hd, int max_seq, int seq_len, spb_stream_t s) {
    clear_error();
    if (int e = check_attn(fn, nh, nkv, hd, max_seq, seq_len)) return e;
    if (hd > 256) return invalid("%s: head_dim %d > 256", fn, hd);
    if (!sc || !V || !out) return invalid("%s: null pointer", fn);
    // A few positions are one round trip and short sums, which the general
    // kernel's four waves per head finish first.  us, general -> 8 dims per
    // block: 20 heads on 5, head_dim 128, 1 / 8 / 16 / 32 positions 2.2 -> 2.7, 2.4
    // -> 2.7, 2.8 -> 2.7, 3.8 -> 2.7; 64 on 64, 256, 1 / 16 / 32 2.3 -> 4.7, 3.6 ->
    // 4.7, 5.1 -> 4.6; 8 on 1, 64, 8 / 16 2.2 -> 2.4, 2.4 -> 2.3.
    if (al16(V) && hd % 8 == 0 && seq_len > std::min(8 + nh / 4, 24)) {
        const int group = (nh + nkv - 1) / nkv;  // the most q heads of a kv head
        // Up to a position per thread a block's time is its sums over the
        // threads, 8 for every head: one head, or as many as leave 2 blocks per
        // CU.  us with 1 / 2 / 4, 64 positions: 20 on 5, head_dim 128 2.7 / 2.7 /
        // 3.1; 64 on 1, 64 2.8 / 2.7 / 3.2, 128 3.3 / 3.1 / 3.2, 256 4.6 / 3.9 /
        // 3.9.  Past that, the reads of V that heads share (2500 positions: 20
        // on 5, 128 6.4 / 5.0 / 5.3, 256 21.4 / 13.3 / 11.4).
        int per = group >= 4 ? 4 : (group >= 2 ? 2 : 1);
        if (seq_len <= kOutBlock)
            for (int p = 1; p < per; p *= 2)
                if (static_cast<long>(hd / 8) * nkv * ((group + p - 1) / p) <=
                    2L * device_cu_count())
                    per = p;
        const dim3 grid(hd / 8, nkv, (group + per - 1) / per), block(kOutBlock);
        switch (per) {
        case 1: hipLaunchKernelGGL((attention_output_cols_kernel<T, 1>), grid, block, 0, as_stream(s), sc, V, out, nh, nkv, hd, max_seq, seq_len); break;
        case 2: hipLaunchKernelGGL((attention_output_cols_kernel<T, 2>), grid, block, 0, as_stream(s), sc, V, out, nh, nkv, hd, max_seq, seq_len); break;
        default: hipLaunchKernelGGL((attention_output_cols_kernel<T, 4>), grid, block, 0, as_stream(s), sc, V, out, nh, nkv, hd, max_seq, seq_len); break;
        }
        return launch_status(fn);
    }
    hipLaunchKernelGGL(attention_output_kernel<T>, dim3(nh), dim3(kOpBlock), 0, as_stream(s), sc, V,
                       out, nh, nkv, hd, max_seq, seq_len);
    return launch_status(fn);
}

template <class T, bool kF32>
int relu2_mul(const char* fn, const uint16_t* g, const uint16_t* u, void* out, int n,
              spb_stream_t s) {
    clear_error();
    if (n < 0) return invalid("%s: negative size", fn);
    if (n == 0) return 0;
    if (!g || !u || !out) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL((relu2_mul_kernel<T, kF32>), dim3(grid_for(n)), dim3(kOpBlock), 0,
                       as_stream(s), g, u, out, static_cast<long>(n));
    return launch_status(fn);
}

template <class T>
int float_to_16(const char* fn, const float* x, uint16_t* y, int n, spb_stream_t s) {
    clear_error();
    if (n < 0) return invalid("%s: negative size", fn);
    if (n == 0) return 0;
    if (!x || !y) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL(float_to_16_kernel<T>, dim3(grid_for(n)), dim3(kOpBlock), 0, as_stream(s), x,
                       y, static_cast<long>(n));
    return launch_status(fn);
}

template <class T>
int residual_add(const char* fn, const uint16_t* a, const uint16_t* b, uint16_t* y, int n,
                 spb_stream_t s) {
    clear_error();
    if (n < 0) return invalid("%s: negative size", fn);
    if (n == 0) return 0;
    if (!a || !b || !y) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL(residual_add_kernel<T>, dim3(grid_for(n)), dim3(kOpBlock), 0, as_stream(s),
                       a, b, y, static_cast<long>(n));
    return launch_status(fn);
}

template <class T>
int gemv16(const char* fn, const uint16_t* W, const uint16_t* x, float* y, int rows, int cols,
           spb_stream_t s) {
    clear_error();
    if (rows < 0 || cols < 0) return invalid("%s: negative shape", fn);
    if (rows == 0) return 0;
    if (!W || !x || !y) return invalid("%s: null pointer", fn);
    const bool vec = cols % 8 == 0 && al16(W) && al16(x);
    const long blocks = (static_cast<long>(rows) + kOpBlock / kWave - 1) / (kOpBlock / kWave);
    hipLaunchKernelGGL(gemv16_kernel<T>, dim3(blocks), dim3(kOpBlock), 0, as_stream(s), W, x, y,
                       rows, cols, vec);
    return launch_status(fn);
}

}  // namespace
}  // namespace spb

using namespace spb;

extern "C" {

int spb_rms_norm_f16(const uint16_t* x, const float* w, uint16_t* y, int size, float eps,
                     spb_stream_t s) {
    return rms_norm<F16, F16, uint16_t>("spb_rms_norm_f16", x, w, y, size, eps, s);
}
int spb_rms_norm_bf16(const uint16_t* x, const float* w, uint16_t* y, int size, float eps,
                      spb_stream_t s) {
    return rms_norm<BF16, BF16, uint16_t>("spb_rms_norm_bf16", x, w, y, size, eps, s);
}
int spb_rms_norm_f32in_f16(const float* x, const float* w, uint16_t* y, int size, float eps,
                           spb_stream_t s) {
    return rms_norm<F16, F32, float>("spb_rms_norm_f32in_f16", x, w, y, size, eps, s);
}
int spb_rms_norm_f32in_bf16(const float* x, const float* w, uint16_t* y, int size, float eps,
                            spb_stream_t s) {
    return rms_norm<BF16, F32, float>("spb_rms_norm_f32in_bf16", x, w, y, size, eps, s);
}
int spb_rope_f16(uint16_t* v, int nh, int hd, int pos, float theta, spb_stream_t s) {
    return rope<F16>("spb_rope_f16", v, nh, hd, pos, theta, s);
}
int spb_rope_bf16(uint16_t* v, int nh, int hd, int pos, float theta, spb_stream_t s) {
    return rope<BF16>("spb_rope_bf16", v, nh, hd, pos, theta, s);
}
int spb_scatter_kv(const uint16_t* src, uint16_t* cache, int nkv, int hd, int max_seq, int pos,
                   spb_stream_t s) {
    clear_error();
    const char* fn = "spb_scatter_kv";
    if (nkv < 0 || hd < 0 || max_seq < 0) return invalid("%s: negative argument", fn);
    if (pos < 0 || pos >= max_seq) return invalid("%s: pos %d outside [0, %d)", fn, pos, max_seq);
    if (nkv == 0 || hd == 0) return 0;
    if (!src || !cache) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL(scatter_kv_kernel, dim3(grid_for(static_cast<long>(nkv) * hd)),
                       dim3(kOpBlock), 0, as_stream(s), src, cache, nkv, hd, max_seq, pos);
    return launch_status(fn);
}
int spb_attention_scores_f16(const uint16_t* Q, const uint16_t* K, float* sc, int nh, int nkv,
                             int hd, int max_seq, int seq_len, float scale, spb_stream_t s) {
    return attention_scores<F16>("spb_attention_scores_f16", Q, K, sc, nh, nkv, hd, max_seq,
                                 seq_len, scale, s);
}
int spb_attention_scores_bf16(const uint16_t* Q, const uint16_t* K, float* sc, int nh, int nkv,
                              int hd, int max_seq, int seq_len, float scale, spb_stream_t s) {
    return attention_scores<BF16>("spb_attention_scores_bf16", Q, K, sc, nh, nkv, hd, max_seq,
                                  seq_len, scale, s);
}
int spb_softmax(float* sc, int nh, int max_seq, int seq_len, spb_stream_t s) {
    clear_error();
    const char* fn = "spb_softmax";
    if (nh < 0 || max_seq < 0 || seq_len < 0 || seq_len > max_seq)
        return invalid("%s: bad shape", fn);
    if (nh == 0 || seq_len == 0) return 0;
    if (!sc) return invalid("%s: null pointer", fn);
    const dim3 grid(nh), block(kNormBlock);
    if (seq_len <= kNormBlock)
        hipLaunchKernelGGL(softmax_regs_kernel<1>, grid, block, 0, as_stream(s), sc, max_seq, seq_len);
    else if (seq_len <= 4 * kNormBlock)
        hipLaunchKernelGGL(softmax_regs_kernel<4>, grid, block, 0, as_stream(s), sc, max_seq, seq_len);
    else if (seq_len <= 8 * kNormBlock)
        hipLaunchKernelGGL(softmax_regs_kernel<8>, grid, block, 0, as_stream(s), sc, max_seq, seq_len);
    else
        hipLaunchKernelGGL(softmax_kernel, grid, block, 0, as_stream(s), sc, max_seq, seq_len);
    return launch_status(fn);
}
int spb_attention_output_f16(const float* sc, const uint16_t* V, uint16_t* out, int nh, int nkv,
                             int hd, int max_seq, int seq_len, spb_stream_t s) {
    return attention_output<F16>("spb_attention_output_f16", sc, V, out, nh, nkv, hd, max_seq,
                                 seq_len, s);
}
int spb_attention_output_bf16(const float* sc, const uint16_t* V, uint16_t* out, int nh, int nkv,
                              int hd, int max_seq, int seq_len, spb_stream_t s) {
    return attention_output<BF16>("spb_attention_output_bf16", sc, V, out, nh, nkv, hd, max_seq,
                                  seq_len, s);
}
int spb_relu2_mul_f16(const uint16_t* g, const uint16_t* u, uint16_t* out, int n, spb_stream_t s) {
    return relu2_mul<F16, false>("spb_relu2_mul_f16", g, u, out, n, s);
}
int spb_relu2_mul_bf16(const uint16_t* g, const uint16_t* u, uint16_t* out, int n, spb_stream_t s) {
    return relu2_mul<BF16, false>("spb_relu2_mul_bf16", g, u, out, n, s);
}
int spb_relu2_mul_f32_f16(const uint16_t* g, const uint16_t* u, float* out, int n, spb_stream_t s) {
    return relu2_mul<F16, true>("spb_relu2_mul_f32_f16", g, u, out, n, s);
}
int spb_relu2_mul_f32_bf16(const uint16_t* g, const uint16_t* u, float* out, int n,
                           spb_stream_t s) {
    return relu2_mul<BF16, true>("spb_relu2_mul_f32_bf16", g, u, out, n, s);
}
int spb_float_to_f16(const float* x, uint16_t* y, int n, spb_stream_t s) {
    return float_to_16<F16>("spb_float_to_f16", x, y, n, s);
}
int spb_float_to_bf16(const float* x, uint16_t* y, int n, spb_stream_t s) {
    return float_to_16<BF16>("spb_float_to_bf16", x, y, n, s);
}
int spb_residual_add_f16(const uint16_t* a, const uint16_t* b, uint16_t* y, int n,
                         spb_stream_t s) {
    return residual_add<F16>("spb_residual_add_f16", a, b, y, n, s);
}
int spb_residual_add_bf16(const uint16_t* a, const uint16_t* b, uint16_t* y, int n,
                          spb_stream_t s) {
    return residual_add<BF16>("spb_residual_add_bf16", a, b, y, n, s);
}
int spb_gemv_f16(const uint16_t* W, const uint16_t* x, float* y, int rows, int cols,
                 spb_stream_t s) {
    return gemv16<F16>("spb_gemv_f16", W, x, y, rows, cols, s);
}
int spb_gemv_bf16(const uint16_t* W, const uint16_t* x, float* y, int rows, int cols,
                  spb_stream_t s) {
    return gemv16<BF16>("spb_gemv_bf16", W, x, y, rows, cols, s);
}
int spb_argmax_f32(const float* x, int n, int* out_index, spb_stream_t s) {
    clear_error();
    const char* fn = "spb_argmax_f32";
    if (n <= 0) return invalid("%s: need n > 0", fn);
    if (!x || !out_index) return invalid("%s: null pointer", fn);
    hipLaunchKernelGGL(argmax_kernel, dim3(1), dim3(kNormBlock), 0, as_stream(s), x, n, out_index);
    return launch_status(fn);
}

}  // extern "C"
