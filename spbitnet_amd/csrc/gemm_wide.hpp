// gemm_wide.hpp -- the 2:4 sparse int8 GEMM for many tokens on the int8
// structured-sparse matrix cores of gfx950 (v_smfmac_i32_16x16x128_i8):
//   Y[t][r] = sum_c W[r][c] * X[t][c] (exact int32), X token-major int8.
// W comes either in spbitnet's packed ternary format (WideTernary) or in the
// tile order of sparse_i8.hip (WideTiles); the epilogue policy is that of
// gemm_staged.hpp.
//
// Tile: 256 rows x 128 tokens per block of eight waves (each 64 rows x 64
// tokens: 4 strips x 4 tiles of 16 x 16, 64 accumulator registers), two blocks
// per CU.  K goes in steps of 128 columns through two LDS buffers of 36 KB in
// operand order: a lane's operand is 16 (values), 4 (index word) or 2 x 16
// (activations) bytes at its own place, so every LDS access is consecutive
// over the wave.
//   * A is decoded once per block into LDS, not by every wave that uses it.
//   * A lane's 16-byte load of the bitmaps is one row's four lane groups of
//     one step; the four lane groups hold four steps, and exchanging them
//     (transpose) gives every lane its own words of four steps.
//   * Activations go from memory to LDS without passing registers.
// What bounds it: the length of a step, and the CU with the most blocks.  13824 x
// 2560, n = 2048 (864 blocks, 87 us): the matrix units are busy 17 % of the time,
// the LDS 20 % (no conflicts), the VALU 24 %; a wave spends 41 % of its life
// waiting for loads, LDS or the barrier and 44 % waiting to issue.  The
// decode does not hold it: the int8 operand, which needs none (VALU 8 %), takes
// the same 85-88 us.  20 steps take 32 us with a block on a CU and 46 with two
// (256 and 512 blocks), then 70, 84 and 108-120 us with a third, fourth and fifth
// on some CU (528 to 768, 864 to 1024 and 1026 to 1040 blocks), so a grid pays
// for whole blocks per CU.  Interleaving VALU and SMFMACs by hand, 128 x 64 tiles
// per wave and 256 tokens per block ran at the same speed.
#pragma once

#include "smfmac.hpp"

namespace spb {
namespace {

constexpr int kWideRows = 256, kWideTok = 128, kWideThreads = 512;
constexpr int kWideStrips = kWideRows / 16, kWideTiles = kWideTok / 16;
constexpr int kWideWaves = kWideThreads / kWave;
constexpr int kWideOwn = kWideStrips / kWideWaves;  // strips a wave loads and decodes

struct WideLds {
    v4i a[2][kWideStrips][kWave];         // 16 compressed values
    int idx[2][kWideStrips][kWave];       // index words
    u32x4v b[2][kWideTiles][2][kWave];    // activations: K 16 q + [0, 16), 64 + 16 q + [0, 16)
};

__device__ __forceinline__ void wide_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void wide_swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
// Register c of lane group g becomes register g of lane group c.
__device__ __forceinline__ void wide_transpose(uint32_t (&r)[4]) {
    wide_swap16(r[0], r[1]);
    wide_swap16(r[2], r[3]);
    wide_swap32(r[0], r[2]);
    wide_swap32(r[1], r[3]);
}

// 16 bytes per lane from the resource to LDS at base + 16 lane.
__device__ __forceinline__ void wide_load_lds(const __amdgpu_buffer_rsrc_t r, int offset,
                                              uint32_t base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 :
                 : "v"(offset), "s"(r), "s"(__builtin_amdgcn_readfirstlane(base))
                 : "memory", "m0");
}
// Every load, LDS store and LDS read of the wave is done, then of the block.
__device__ __forceinline__ void wide_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The packed ternary rows (cols % 128 == 0, 16-byte aligned bitmap rows and
// 8-byte aligned sign rows; stacked matrices whose boundaries are multiples of
// 16 rows).  Loads cover four steps.
struct WideTernary {
    static constexpr int kAhead = 4;  // steps per load
    const uint32_t* meta;
    const uint32_t* values;
    int rows, ms, vs;
    GemmSegs segs;
    struct Raw {
        u32x4v m[kWideOwn];
        uint2 v[kWideOwn];
    };
    struct Held {
        uint32_t m[kWideOwn][4], v[kWideOwn][4];
    };
    // Steps step0 .. step0 + 3 of strips strip0 .. strip0 + kWideOwn - 1.  Rows
    // past the matrix read its last row and steps past the row its last step;
    // neither feeds a stored result.
    __device__ void load(Raw& r, int strip0, int step0, int nsteps, int lane) const {
        const int st = min(step0 + (lane >> 4), nsteps - 1);
#pragma unroll
        for (int k = 0; k < kWideOwn; ++k) {
            const int s16 = (strip0 + k) * 16;  // uniform: the strip lies in one matrix
            long om = 0, ov = 0;
            if (s16 >= segs.end0) om = segs.om1, ov = segs.ov1;
            if (s16 >= segs.end1) om = segs.om2, ov = segs.ov2;
            const int row = min(s16 + (lane & 15), rows - 1);
            r.m[k] = *reinterpret_cast<const u32x4v*>(meta + om + (static_cast<long>(row) * ms + 4 * st));
            r.v[k] = *reinterpret_cast<const uint2*>(values + ov + (static_cast<long>(row) * vs + 2 * st));
        }
    }
    __device__ static void hold(const Raw& r, Held& h) {
#pragma unroll
        for (int k = 0; k < kWideOwn; ++k) {
            h.m[k][0] = r.m[k][0], h.m[k][1] = r.m[k][1];
            h.m[k][2] = r.m[k][2], h.m[k][3] = r.m[k][3];
            wide_transpose(h.m[k]);
            // the low 16 bits are the lane's signs
            h.v[k][0] = r.v[k].x, h.v[k][1] = r.v[k].x >> 16;
            h.v[k][2] = r.v[k].y, h.v[k][3] = r.v[k].y >> 16;
            wide_transpose(h.v[k]);
        }
    }
    // strip k's operand of the i-th held step
    __device__ static void operand(const Held& h, int k, int i, v4i& a, int& idx) {
        idx = smfmac_index(h.m[k][i]);
        a = smfmac_values(h.v[k][i]);
    }
};

// The tile order of sparse_i8.hip: strip s, step j at byte (s * steps + j) *
// 1280, values then index words, both by lane.
struct WideTiles {
    static constexpr int kAhead = 1;
    const uint8_t* comp;
    int strips, steps;
    struct Raw {
        v4i a[kWideOwn];
        int idx[kWideOwn];
    };
    using Held = Raw;
    __device__ void load(Raw& r, int strip0, int step0, int, int lane) const {
        const int st = min(step0, steps - 1);
#pragma unroll
        for (int k = 0; k < kWideOwn; ++k) {
            const uint8_t* t =
                comp + (static_cast<long>(min(strip0 + k, strips - 1)) * steps + st) * 1280;
            r.a[k] = *reinterpret_cast<const v4i*>(t + 16 * lane);
            r.idx[k] = *reinterpret_cast<const int*>(t + 1024 + 4 * lane);
        }
    }
    __device__ static void hold(const Raw& r, Held& h) { h = r; }
    __device__ static void operand(const Held& h, int k, int, v4i& a, int& idx) {
        a = h.a[k];
        idx = h.idx[k];
    }
};

// xstride: bytes per token of X (a multiple of 16, below 2^23; X 16-byte
// aligned).  A step may read past a token's bytes where A is zero
// (WideTiles); past the block's last token the loads return zeros.
template <class A, class Epi>
__global__ __launch_bounds__(kWideThreads, 4) void gemm_wide_kernel(A src,
                                                                    const int8_t* __restrict__ X,
                                                                    Epi epi, int rows, int nsteps,
                                                                    int n, int xstride) {
    extern __shared__ __align__(16) uint8_t wide_smem[];
    WideLds& sh = *reinterpret_cast<WideLds*>(wide_smem);
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int q = lane >> 4, li = lane & 15;
    const int r0 = blockIdx.x * kWideRows, t0 = blockIdx.y * kWideTok;
    const int ws = wave & 3, wt = wave >> 2;  // the wave's quarter of the strips and half of the tiles
    // activations: wave w stages tile w, both 64-byte halves
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(X + static_cast<long>(t0) * xstride), static_cast<short>(0),
        min(n - t0, kWideTok) * xstride, kRawBufferFlags);
    const int xo = (16 * wave + li) * xstride + 16 * q;
    // Straight to LDS (lane l's 16 bytes at M0 + 16 l): no registers to hold
    // the tile over a step, no LDS store instructions.
    const uint32_t lds_b = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) void*)&sh.b[0][wave][0][0]));
    auto load_b = [&](int s, int buf) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            wide_load_lds(rx, xo + 128 * s + 64 * h,
                          lds_b + buf * sizeof(sh.b[0]) + h * sizeof(sh.b[0][0][0]));
    };
    typename A::Raw raw;
    typename A::Held held;
    const int strip0 = r0 / 16 + kWideOwn * wave;
    auto store_a = [&](int buf, int i) {
#pragma unroll
        for (int k = 0; k < kWideOwn; ++k) {
            v4i a;
            int idx;
            A::operand(held, k, i, a, idx);
            sh.a[buf][kWideOwn * wave + k][lane] = a;
            sh.idx[buf][kWideOwn * wave + k][lane] = idx;
        }
    };
    v4i acc[4][4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[s][t] = (v4i){0, 0, 0, 0};
    auto compute = [&](int buf) {
        v4i a[4];
        int idx[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            a[s] = sh.a[buf][4 * ws + s][lane];
            idx[s] = sh.idx[buf][4 * ws + s][lane];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const u32x4v lo = sh.b[buf][4 * wt + t][0][lane], hi = sh.b[buf][4 * wt + t][1][lane];
            const v8i b = (v8i){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3],
                                (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                acc[s][t] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(a[s], b, acc[s][t], idx[s], 0, 0);
        }
    };
    // Step s from buffer i & 1 (i = s % 4), while s + 1 is loaded and laid out
    // in the other; past the last step that is done for nothing, so that a
    // step has no branch.
    auto step = [&](int s, int i) {
        load_b(s + 1, (i + 1) & 1);
        if (A::kAhead == 4 && i == 2) src.load(raw, strip0, s + 2, nsteps, lane);
        if (A::kAhead == 1) {
            A::hold(raw, held);
            src.load(raw, strip0, s + 2, nsteps, lane);
        }
        __builtin_amdgcn_sched_barrier(0);  // the loads go out here, not where they are used
        if (A::kAhead == 4 && i == 3) A::hold(raw, held);
        store_a((i + 1) & 1, A::kAhead == 4 ? (i + 1) & 3 : 0);
        compute(i & 1);
        wide_barrier();
    };

    src.load(raw, strip0, 0, nsteps, lane);
    load_b(0, 0);
    A::hold(raw, held);
    store_a(0, 0);
    if constexpr (A::kAhead == 1) src.load(raw, strip0, 1, nsteps, lane);
    wide_barrier();
    int s = 0;
    for (; s + 4 <= nsteps; s += 4) {
        step(s, 0);
        step(s + 1, 1);
        step(s + 2, 2);
        step(s + 3, 3);
    }
    if (s < nsteps) step(s, 0);  // uniform
    if (s + 1 < nsteps) step(s + 1, 1);
    if (s + 2 < nsteps) step(s + 2, 2);
    // lane (li, q) of tile (e, t) holds rows 16 (4 ws + e) + 4 q .. + 3 of token 16 (4 wt + t) + li
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = r0 + 16 * (4 * ws + e) + 4 * q;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int tok = t0 + 16 * (4 * wt + t) + li;
            if (tok < n && row < rows) epi.store4(tok, row, acc[e][t], epi.preload(tok, row));
        }
    }
}

template <class A, class Epi>
const void* wide_fn() {
    return reinterpret_cast<const void*>(&gemm_wide_kernel<A, Epi>);
}

template <class A, class Epi>
int launch_wide(const A& src, const int8_t* X, const Epi& epi, int rows, int nsteps, int n,
                int xstride, hipStream_t st) {
    const int lds = static_cast<int>(sizeof(WideLds));
    if (lds > device_lds_per_cu() || !gemm_allow_lds(wide_fn<A, Epi>()))
        return invalid("gemm_wide: %d bytes of LDS unavailable", lds);
    hipLaunchKernelGGL((gemm_wide_kernel<A, Epi>),
                       dim3((rows + kWideRows - 1) / kWideRows, (n + kWideTok - 1) / kWideTok),
                       dim3(kWideThreads), lds, st, src, X, epi, rows, nsteps, n, xstride);
    return 0;
}

long wide_blocks(int rows, int n) {
    return static_cast<long>((rows + kWideRows - 1) / kWideRows) * ((n + kWideTok - 1) / kWideTok);
}

// The packed ternary product takes the wide kernel when its grid is 1.5 blocks
// per CU or more (two fit a CU): below that a block per CU runs at its own
// latency, ~1 us per 128 columns, and the staged tiles win.  us per launch,
// staged -> wide: 13824 x 2560, n = 1024 / 2048 / 3000 (432 / 864 / 1296
// blocks) 53.8 -> 45.7, 104.6 -> 86.6, 147.0 -> 129.6; 6912 x 2560, n = 2048
// (432) 52.6 -> 46.5; 3840 x 2560, n = 3000 (360) 43.7 -> 43.4, n = 2048 (240)
// 30.9 -> 31.1; 2560 x 6912, n = 2048 (160) 59.8 -> 65.2.
//
// Not so in two places (same runs, staged -> wide):
//   * 17-32 tokens of 98,000 rows or more: the 64 x 32 tile holds them all and
//     wastes no products.  100352 x 2560, n = 16 / 17 / 32 / 48 / 64 / 65 31.8
//     -> 29.4, 19.2 -> 29.3, 21.2 -> 31.3, 34.2 -> 33.9, 36.3 -> 36.2, 48.5 ->
//     36.9; 552960 x 2560, n = 1 / 16 / 32 / 48 145 -> 130, 174 -> 144, 113 ->
//     153, 200 -> 168; 196608 x 1024, n = 16 / 17 / 32 / 48 55.5 -> 25.1, 17.8
//     -> 24.5, 18.9 -> 27.1, 32.1 -> 30.8.
//   * The first quarter of a third block per CU (513-576 blocks): a few CUs run
//     three.  2048 tokens, 8448 rows (528) at 512 / 1024 / 1536 / 2048 / 2560 /
//     4096 / 5120 / 6912 columns 26.0 -> 27.6, 34.2 -> 38.7, 44.5 -> 48.4, 58.6
//     -> 61.7, 66.2 -> 67.7, 95.1 -> 100, 113 -> 120, 156.4 -> 156.6; 9216 rows
//     (576) at 1024 / 2560 / 4096 / 6912 35.8 -> 38.8, 65.9 -> 64.4, 93.3 ->
//     97.3, 154 -> 146; 9472 (592) at 1024 / 2560 / 4096 37.9 -> 38.7, 71.6 ->
//     68.6, 104.5 -> 101.0.  Past a third and a fourth block the wide kernel
//     wins but for 1024-1536 columns, within 3 % (784 blocks at 1024 48.5 ->
//     50.0).
bool wide_ternary_ok(int rows, int cols, int n, const GemmSegs& g) {
    const long blocks = wide_blocks(rows, n), cus = device_cu_count();
    if (2 * blocks < 3 * cus || (n > 16 && n <= 32)) return false;
    if (blocks > 2 * cus && 4 * blocks <= 9 * cus && cols <= 5120) return false;
    return cols < (1 << 23) && (g.end0 >= rows || g.end0 % 16 == 0) &&
           (g.end1 >= rows || g.end1 % 16 == 0);
}

}  // namespace
}  // namespace spb
