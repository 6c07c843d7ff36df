// sparse_i8.hip -- 2:4 structured-sparse int8 GEMM on the int8 sparse matrix
// cores of gfx950 (v_smfmac_i32_16x16x128_i8): the drop-in for the
// reference's cuSPARSELt backend, CuSparseLtGemm (include/spbitnet/
// cusparselt_backend.h:28-77, src/cusparselt_backend.cu:38-219), whose
// prepare() prunes a dense int8 weight matrix to 2:4 and compresses it and
// whose execute() computes D = A_pruned * B with int32 accumulation.
//
// Unlike spbitnet's ternary format, the weights here are any int8 values
// (the reference's tests feed {-1, 0, +1} with kept zeros,
// tests/test_cusparselt.cu:68-117), so the compressed operand keeps two int8
// values per group of four.
//
// Pruning rule (cuSPARSELt's STRIP selection is not specified by the
// reference and is not reproduced): in each group of four along k keep the
// two largest |a|, on equal magnitudes the higher index -- the rule of the
// stable argsort in python/convert_model.py:88-119 that the ternary
// converter uses.  A group with at most two non-zeros keeps all of them, so
// a matrix already in 2:4 form is unchanged.
//
// Compressed operand ("tile order"): the matrix is cut into tiles of 16 rows
// x 128 columns (rows padded to a multiple of 16, columns to 128, with
// zeros); tile (strip s, step j) sits at byte (s * steps + j) * 1280 and
// holds, for SMFMAC lane l = 16 a + i (row 16 s + i, columns 128 j + 32 a +
// [0, 32)), the lane's 16 compressed values at byte 16 l (value 2g, 2g + 1
// = the kept entries of group g, lower column first) and its index word at
// byte 1024 + 4 l (nibble g = p0 | p1 << 2, the kept positions inside
// group g).  That is exactly the A operand of v_smfmac_i32_16x16x128_i8, so
// a wave loads a tile's operand with one 16-byte and one 4-byte load per
// lane, both fully coalesced, and decodes nothing.  Empty groups hold zeros
// with positions (0, 1).
//
// B is int8 [k x n] column-major (= token-major [n][k]) and D int32 [m x n]
// column-major (= [n][m]), as the reference declares them
// (src/cusparselt_backend.cu:53-78).
#include "common.hpp"
#include "gemm_staged.hpp"
#include "spbitnet_amd.h"

namespace spb {
namespace {

constexpr int kI8TileBytes = 1280;  // 16 rows x 128 columns: values then index words
constexpr int kI8ValBytes = 1024;
constexpr uint32_t kI8EmptyNibble = 0x4u;  // positions (0, 1)
constexpr int kI8RawBufferFlags = 0x00020000;  // gfx9 raw buffer resource word 3

long i8_steps(int k) { return (k + 127) / 128; }
long i8_strips(int m) { return (m + 15) / 16; }

// Kept positions of a group (v[0..3]): nibble p0 | p1 << 2, p0 < p1.
__device__ __forceinline__ uint32_t i8_top2_nibble(int v0, int v1, int v2, int v3) {
    const int a[4] = {v0 < 0 ? -v0 : v0, v1 < 0 ? -v1 : v1, v2 < 0 ? -v2 : v2, v3 < 0 ? -v3 : v3};
    uint32_t keep = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int beaten = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j != i && (a[j] > a[i] || (a[j] == a[i] && j > i))) ++beaten;
        if (beaten < 2) keep |= 1u << i;
    }
    const uint32_t p0 = __builtin_ctz(keep), p1 = __builtin_ctz(keep & (keep - 1));
    return p0 | (p1 << 2);
}

// One wave per tile: lane (a, i) prunes row 16 s + i, columns 128 j + 32 a +
// [0, 32) and writes its compressed values, its index word and (optionally)
// the pruned dense row segment.
__global__ __launch_bounds__(256) void sparse_i8_prune_kernel(const int8_t* __restrict__ A,
                                                              int8_t* __restrict__ pruned,
                                                              uint8_t* __restrict__ comp, int m,
                                                              int k, int steps, long ntiles) {
    const long tile = static_cast<long>(blockIdx.x) * 4 + threadIdx.x / kWave;
    if (tile >= ntiles) return;
    const int lane = threadIdx.x & (kWave - 1), a = lane >> 4, li = lane & 15;
    const long row = (tile / steps) * 16 + li;
    const int c0 = static_cast<int>(tile % steps) * 128 + 32 * a;
    uint32_t vals[4] = {0u, 0u, 0u, 0u}, idx = 0u;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const int c = c0 + 4 * g;
        const bool in = row < m && c < k;  // k % 4 == 0: a group is wholly inside or outside
        uint32_t w = 0u;
        if (in) w = *reinterpret_cast<const uint32_t*>(A + row * k + c);
        const int v0 = static_cast<int8_t>(w), v1 = static_cast<int8_t>(w >> 8);
        const int v2 = static_cast<int8_t>(w >> 16), v3 = static_cast<int8_t>(w >> 24);
        const uint32_t nib = in ? i8_top2_nibble(v0, v1, v2, v3) : kI8EmptyNibble;
        const uint32_t p0 = nib & 3u, p1 = nib >> 2;
        const uint32_t b0 = (w >> (8 * p0)) & 0xFFu, b1 = (w >> (8 * p1)) & 0xFFu;
        vals[g >> 1] |= (b0 | (b1 << 8)) << (16 * (g & 1));
        idx |= nib << (4 * g);
        if (pruned && in)
            *reinterpret_cast<uint32_t*>(pruned + row * k + c) = (b0 << (8 * p0)) | (b1 << (8 * p1));
    }
    uint8_t* t = comp + tile * kI8TileBytes;
    *reinterpret_cast<v4i*>(t + lane * 16) =
        (v4i){static_cast<int>(vals[0]), static_cast<int>(vals[1]), static_cast<int>(vals[2]),
              static_cast<int>(vals[3])};
    *reinterpret_cast<uint32_t*>(t + kI8ValBytes + lane * 4) = idx;
}

// Groups of A with more than two non-zeros, counted into *bad (set to 0
// first by sparse_i8_zero_kernel on the same stream).
__global__ void sparse_i8_zero_kernel(int* bad) { *bad = 0; }

__global__ __launch_bounds__(256) void sparse_i8_check_kernel(const int8_t* __restrict__ A, int m,
                                                              int k, int* bad) {
    const long groups = static_cast<long>(m) * (k / 4);
    const long g = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    int over = 0;
    if (g < groups) {
        const long row = g / (k / 4);
        const int c = static_cast<int>(g - row * (k / 4)) * 4;
        const uint32_t w = *reinterpret_cast<const uint32_t*>(A + row * k + c);
        const int nz = ((w & 0xFFu) != 0) + ((w & 0xFF00u) != 0) + ((w & 0xFF0000u) != 0) +
                       ((w & 0xFF000000u) != 0);
        over = nz > 2;
    }
    const unsigned long long ball = __ballot(over);
    if ((threadIdx.x & (kWave - 1)) == 0 && ball) atomicAdd(bad, __popcll(ball));
}

// Compressed -> dense [m][k] (the pruned matrix): one thread per group.
__global__ __launch_bounds__(256) void sparse_i8_decompress_kernel(const uint8_t* __restrict__ comp,
                                                                   int8_t* __restrict__ out, int m,
                                                                   int k, int steps) {
    const long groups = static_cast<long>(m) * (k / 4);
    const long g = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (g >= groups) return;
    const long row = g / (k / 4);
    const int c = static_cast<int>(g - row * (k / 4)) * 4;
    const int j = c >> 7, cl = c & 127, a = cl >> 5, gl = (cl & 31) >> 2;
    const int lane = 16 * a + static_cast<int>(row & 15);
    const uint8_t* t = comp + ((row >> 4) * steps + j) * kI8TileBytes;
    const uint32_t nib = (*reinterpret_cast<const uint32_t*>(t + kI8ValBytes + lane * 4) >> (4 * gl)) & 0xFu;
    const uint32_t b0 = t[lane * 16 + 2 * gl], b1 = t[lane * 16 + 2 * gl + 1];
    const uint32_t p0 = nib & 3u, p1 = nib >> 2;
    *reinterpret_cast<uint32_t*>(out + row * k + c) = (b0 << (8 * p0)) | (b1 << (8 * p1));
}

// D[t][r] = sum_c A[r][c] B[t][c] on the matrix cores.  Block: W waves on
// S strips (16 S rows) and T token tiles (16 T tokens, grid.y); wave w takes
// the 128-column steps w, w + W, ... of every (strip, tile) and the W partial
// sums meet in LDS.  A tiles load straight from the compressed operand (one
// 16-byte and one 4-byte load per lane, 1.25 KB contiguous per wave); B
// lane (token i, group q) loads columns 16 q + [0, 16) and 64 + 16 q + [0,
// 16) of the step through a buffer resource covering B's n * k bytes, so
// tokens past n read zeros; columns past k meet zero A values.
template <int S, int T, int W>
__global__ __launch_bounds__(W * kWave) void sparse_i8_gemm_kernel(
    const uint8_t* __restrict__ comp, const int8_t* __restrict__ B, int32_t* __restrict__ D,
    int m, int k, int n, int steps, int strips, int quads) {
    __shared__ v4i red[W * S * T * kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, li = lane & 15;
    const int s0 = blockIdx.x * S, t0 = blockIdx.y * (16 * T);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(B), static_cast<short>(0), n * k, kI8RawBufferFlags);
    v4i acc[S][T];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[s][t] = (v4i){0, 0, 0, 0};
    // a step's operands, loaded one step ahead of their products; strips past
    // the matrix read its last one (their rows are not stored), and loads past
    // a wave's last step get empty extents: zeros, without a trip to memory.
    // Reading a step again there cost short rows most, us: 13824 x 1024, n = 128
    // / 256 9.7 -> 8.9, 14.4 -> 12.7; 30000 x 1024, n = 1 / 8 / 16 3.6 -> 3.6, 4.6
    // -> 4.4, 5.8 -> 5.2 (3.4, 4.1 and 4.9 without loads ahead, which
    // everywhere else are the faster form: 6912 x 6912, n = 16 8.1 -> 6.7).
    struct Step {
        v4i a[S];
        int idx[S];
        v4i lo[T], hi[T];
    };
    auto load = [&](int j, Step& o) {
        const bool live = j < steps;  // uniform
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int strip = s0 + s < strips ? s0 + s : strips - 1;
            const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t*>(comp + (static_cast<long>(strip) * steps + (live ? j : 0)) *
                                                kI8TileBytes),
                static_cast<short>(0), live ? kI8TileBytes : 0, kI8RawBufferFlags);
            o.a[s] = __builtin_bit_cast(
                v4i, __builtin_amdgcn_raw_buffer_load_b128(ra, lane * 16, 0, 0));
            o.idx[s] = static_cast<int>(
                __builtin_amdgcn_raw_buffer_load_b32(ra, kI8ValBytes + lane * 4, 0, 0));
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int off = live ? (t0 + 16 * t + li) * k + 128 * j + 16 * q : n * k;
            o.lo[t] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rb, off, 0, 0));
            o.hi[t] =
                __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rb, off + 64, 0, 0));
        }
    };
    auto multiply = [&](const Step& o) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const v8i b = (v8i){o.lo[t][0], o.lo[t][1], o.lo[t][2], o.lo[t][3],
                                o.hi[t][0], o.hi[t][1], o.hi[t][2], o.hi[t][3]};
#pragma unroll
            for (int s = 0; s < S; ++s)
                acc[s][t] =
                    __builtin_amdgcn_smfmac_i32_16x16x128_i8(o.a[s], b, acc[s][t], o.idx[s], 0, 0);
        }
    };
    Step x, y;
    load(wave, x);
    for (int j = wave; j < steps; j += 2 * W) {
        load(j + W, y);
        __builtin_amdgcn_sched_barrier(0);
        multiply(x);
        if (j + W >= steps) break;  // uniform
        load(j + 2 * W, x);
        __builtin_amdgcn_sched_barrier(0);
        multiply(y);
    }
    if (W > 1) {
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int t = 0; t < T; ++t) red[((wave * S + s) * T + t) * kWave + lane] = acc[s][t];
        __syncthreads();
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int t = 0; t < T; ++t)
                if ((s * T + t) % W == wave) {
                    v4i sum = red[(s * T + t) * kWave + lane];
#pragma unroll
                    for (int w = 1; w < W; ++w) sum += red[((w * S + s) * T + t) * kWave + lane];
                    acc[s][t] = sum;
                }
    }
    // lane (i, q) of (strip, tile) holds rows 16 strip + 4 q .. + 3 of token 16 tile + i
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int row = (s0 + s) * 16 + 4 * q;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int tok = t0 + 16 * t + li;
            if ((W == 1 || (s * T + t) % W == wave) && tok < n && row < m) {
                int32_t* y = D + static_cast<long>(tok) * m + row;
                if (quads) {
                    *reinterpret_cast<v4i*>(y) = acc[s][t];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (row + e < m) y[e] = acc[s][t][e];
                }
            }
        }
    }
}

// Any shape with k % 4 == 0 and any alignment: one wave per row, tokens on
// grid.y, groups decoded from the compressed operand.
__global__ __launch_bounds__(256) void sparse_i8_gemm_general_kernel(
    const uint8_t* __restrict__ comp, const int8_t* __restrict__ B, int32_t* __restrict__ D,
    int m, int k, int n, int steps) {
    const int lane = threadIdx.x & (kWave - 1);
    const long row = static_cast<long>(blockIdx.x) * 4 + threadIdx.x / kWave;
    const int tok = blockIdx.y;
    if (row >= m) return;
    const int8_t* x = B + static_cast<long>(tok) * k;
    int acc = 0;
    for (int g = lane; g < (k >> 2); g += kWave) {
        const int c = 4 * g, j = c >> 7, cl = c & 127, a = cl >> 5, gl = (cl & 31) >> 2;
        const int ln = 16 * a + static_cast<int>(row & 15);
        const uint8_t* t = comp + ((row >> 4) * steps + j) * kI8TileBytes;
        const uint32_t nib =
            (*reinterpret_cast<const uint32_t*>(t + kI8ValBytes + ln * 4) >> (4 * gl)) & 0xFu;
        const int v0 = static_cast<int8_t>(t[ln * 16 + 2 * gl]);
        const int v1 = static_cast<int8_t>(t[ln * 16 + 2 * gl + 1]);
        acc += v0 * static_cast<int>(x[c + (nib & 3u)]) + v1 * static_cast<int>(x[c + (nib >> 2)]);
    }
    acc = wave_sum(acc);
    if (lane == 0) D[static_cast<long>(tok) * m + row] = acc;
}

bool i8_aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

template <int S, int T, int W>
void launch_i8_gemm(const uint8_t* comp, const int8_t* B, int32_t* D, int m, int k, int n,
                    hipStream_t st) {
    const int steps = static_cast<int>(i8_steps(k)), strips = static_cast<int>(i8_strips(m));
    const dim3 grid((strips + S - 1) / S, (n + 16 * T - 1) / (16 * T));
    const int quads = (m % 4 == 0 && i8_aligned(D, 16)) ? 1 : 0;
    hipLaunchKernelGGL((sparse_i8_gemm_kernel<S, T, W>), grid, dim3(W * kWave), 0, st, comp, B, D,
                       m, k, n, steps, strips, quads);
}

// The tile for n tokens.  us per launch, the 32 x 64 tile without the loads a
// step ahead that every size above 16 took before -> now:
//   * more than 32 tokens and a grid of at least 5/8 wide blocks (256 x 128)
//     per CU: the wide kernel.  13824 x 2560, n = 512 / 1024 / 2048 72.8 -> 31.6,
//     135 -> 44.2, 263 -> 87.5; 6912 x 2560, n = 1024 / 2048 70.2 -> 32.5, 132 ->
//     45.5; 2560 x 6912, n = 2048 (160 blocks) 131 -> 67.
//     Up to 32 tokens one block of the tiles below holds them all: the tile that
//     they choose -> wide, 40960 x 2560 (160 wide blocks), n = 1 / 16 / 17 / 32
//     10.6 -> 19.6, 11.3 -> 20.5, 12.2 -> 20.8, 13.5 -> 21.9; 100352 x 2560 (392)
//     23.1 -> 28.6, 24.7 -> 29.8, 26.5 -> 30.0, 28.5 -> 31.6.
//     The line against the tiles that it displaces: 96 x 32 -> wide, 6912 x
//     2560, n = 640 / 768 / 896 / 1024 (135 / 162 / 189 / 216 blocks) 25.2 ->
//     29.9, 28.9 -> 30.4, 32.5 -> 30.8, 36.0 -> 31.4, 4096 x 4096, n = 1024 / 1280
//     (128 / 160) 54.7 -> 41.3, 65.2 -> 41.9; 128 x 32 -> wide, 2560 x 6912,
//     n = 1536 / 2048 / 2560 (120 / 160 / 200) 49.4 -> 65.0, 60.8 -> 66.1, 81.0 ->
//     66.5: for 2560 and 6912 columns it could lie at 190 blocks, for 4096 lower
//     than it does;
//   * long rows (over 4096 columns) with at least half a 128 x 32 block per
//     CU: each activation feeds eight strips; 2560 x 6912, n = 256 / 512 / 1024
//     27.8 -> 14.9, 41.3 -> 25.6, 78.7 -> 37.4 (54.4 with 96 x 32);
//   * enough 96 x 32 blocks (two per CU): 6912 x 2560, n = 256 / 512 22.3 ->
//     14.1, 36.7 -> 22.5; 13824 x 2560, n = 128 / 256 23.4 -> 14.0, 38.3 -> 21.7;
//   * else 64 x 32: 6912 x 2560, n = 128 12.1 -> 9.5; 2560 x 6912, n = 128
//     15.2 -> 10.7; 2560 x 2560, n = 256 12.0 -> 8.7.
int launch_i8_for(const uint8_t* comp, const int8_t* B, int32_t* D, int m, int k, int n,
                  hipStream_t st) {
    const long cus = device_cu_count(), passes = (n + 31) / 32;
    if (n > 32 && 8 * wide_blocks(m, n) >= 5 * cus) {
        const WideTiles src{comp, static_cast<int>(i8_strips(m)), static_cast<int>(i8_steps(k))};
        const Int32Out out{D, m, m % 4 == 0 && i8_aligned(D, 16)};
        return launch_wide(src, B, out, m, static_cast<int>(i8_steps(k)), n, k, st);
    }
    if (n <= 16)
        launch_i8_gemm<2, 1, 4>(comp, B, D, m, k, n, st);
    else if (k > 4096 && 2 * ((m + 127) / 128) * passes >= cus)
        launch_i8_gemm<8, 2, 4>(comp, B, D, m, k, n, st);
    else if ((m + 95) / 96 * passes >= 2 * cus)
        launch_i8_gemm<6, 2, 4>(comp, B, D, m, k, n, st);
    else
        launch_i8_gemm<4, 2, 4>(comp, B, D, m, k, n, st);
    return 0;
}

const char* i8_shape_error(int m, int k) {
    if (m < 0 || k < 0) return "negative shape";
    if (k % 4) return "k is not a multiple of 4 (2:4 groups along k)";
    if (static_cast<long>(m) * k >= (1L << 31)) return "m * k must stay below 2^31";
    return nullptr;
}

}  // namespace
}  // namespace spb

using namespace spb;

extern "C" long spb_sparse_i8_compressed_size(int m, int k) {
    clear_error();
    if (const char* e = i8_shape_error(m, k)) {
        set_error("spb_sparse_i8_compressed_size: %s", e);
        return -1;
    }
    return i8_strips(m) * i8_steps(k) * kI8TileBytes;
}

extern "C" int spb_sparse_i8_prune_compress(const int8_t* A, int8_t* pruned, void* compressed,
                                            int m, int k, spb_stream_t stream) {
    clear_error();
    const char* fn = "spb_sparse_i8_prune_compress";
    if (const char* e = i8_shape_error(m, k)) return invalid("%s: %s", fn, e);
    if (m == 0 || k == 0) return 0;
    if (!A || !compressed) return invalid("%s: null pointer", fn);
    if (!i8_aligned(A, 4) || (pruned && !i8_aligned(pruned, 4)) || !i8_aligned(compressed, 16))
        return invalid("%s: A and pruned need 4-byte, compressed 16-byte alignment", fn);
    const long ntiles = i8_strips(m) * i8_steps(k);
    hipLaunchKernelGGL(sparse_i8_prune_kernel, dim3(static_cast<unsigned>((ntiles + 3) / 4)),
                       dim3(256), 0, as_stream(stream), A, pruned,
                       static_cast<uint8_t*>(compressed), m, k, static_cast<int>(i8_steps(k)),
                       ntiles);
    return launch_status(fn);
}

extern "C" int spb_sparse_i8_prune_check(const int8_t* A, int m, int k, int* d_invalid,
                                         spb_stream_t stream) {
    clear_error();
    const char* fn = "spb_sparse_i8_prune_check";
    if (const char* e = i8_shape_error(m, k)) return invalid("%s: %s", fn, e);
    if (!d_invalid) return invalid("%s: null result pointer", fn);
    hipStream_t st = as_stream(stream);
    hipLaunchKernelGGL(sparse_i8_zero_kernel, dim3(1), dim3(1), 0, st, d_invalid);
    const long groups = static_cast<long>(m) * (k / 4);
    if (groups > 0) {
        if (!A) return invalid("%s: null pointer", fn);
        if (!i8_aligned(A, 4)) return invalid("%s: A needs 4-byte alignment", fn);
        hipLaunchKernelGGL(sparse_i8_check_kernel, dim3(static_cast<unsigned>((groups + 255) / 256)),
                           dim3(256), 0, st, A, m, k, d_invalid);
    }
    return launch_status(fn);
}

extern "C" int spb_sparse_i8_decompress(const void* compressed, int8_t* out, int m, int k,
                                        spb_stream_t stream) {
    clear_error();
    const char* fn = "spb_sparse_i8_decompress";
    if (const char* e = i8_shape_error(m, k)) return invalid("%s: %s", fn, e);
    if (m == 0 || k == 0) return 0;
    if (!compressed || !out) return invalid("%s: null pointer", fn);
    if (!i8_aligned(out, 4) || !i8_aligned(compressed, 16))
        return invalid("%s: out needs 4-byte, compressed 16-byte alignment", fn);
    const long groups = static_cast<long>(m) * (k / 4);
    hipLaunchKernelGGL(sparse_i8_decompress_kernel, dim3(static_cast<unsigned>((groups + 255) / 256)),
                       dim3(256), 0, as_stream(stream), static_cast<const uint8_t*>(compressed),
                       out, m, k, static_cast<int>(i8_steps(k)));
    return launch_status(fn);
}

extern "C" int spb_sparse_i8_gemm_kernel_id(const void* compressed, const int8_t* B, int m,
                                            int k, int n) {
    (void)compressed;
    (void)m;
    if (k <= 0 || k % 16 || !i8_aligned(B, 16)) return 0;
    if ((static_cast<long>(n) + 64) * k >= (1L << 31) || (n + 15) / 16 > 65535) return 0;
    return 1;
}

extern "C" int spb_sparse_i8_gemm(const void* compressed, const int8_t* B, int32_t* D, int m,
                                  int k, int n, spb_stream_t stream) {
    clear_error();
    const char* fn = "spb_sparse_i8_gemm";
    if (const char* e = i8_shape_error(m, k)) return invalid("%s: %s", fn, e);
    if (n < 0) return invalid("%s: negative n", fn);
    if (m == 0 || k == 0 || n == 0) return 0;  // a no-op, as the reference's wrappers
    if (!compressed || !D || !B) return invalid("%s: null pointer", fn);
    if (!i8_aligned(compressed, 16)) return invalid("%s: compressed needs 16-byte alignment", fn);
    hipStream_t st = as_stream(stream);
    const auto* comp = static_cast<const uint8_t*>(compressed);
    if (spb_sparse_i8_gemm_kernel_id(compressed, B, m, k, n)) {
        if (const int rc = launch_i8_for(comp, B, D, m, k, n, st)) return rc;
    } else {
        if (n > 65535) return invalid("%s: n = %d exceeds 65535 on the general kernel", fn, n);
        hipLaunchKernelGGL(sparse_i8_gemm_general_kernel,
                           dim3(static_cast<unsigned>((m + 3) / 4), static_cast<unsigned>(n)),
                           dim3(256), 0, st, comp, B, D, m, k, n, static_cast<int>(i8_steps(k)));
    }
    return launch_status(fn);
}
