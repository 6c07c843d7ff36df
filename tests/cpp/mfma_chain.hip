// What the prefill attention rests on, checked on the GPU: a chain of
// v_mfma_f32_16x16x4_f32 gives the bits of a chain of fused multiply-adds over k
// ascending, each rounded to nearest even, denormals kept.  16 x 16 sums of 32
// products per block, against fmaf on the host: ordinary values, exponents over
// the whole range (sums that overflow and underflow), denormals, and some
// infinities and NaN.  Prints the differing sums of each kind and returns 1 if
// there are any.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

namespace {
constexpr int kK = 32, kBlocks = 2048;
typedef float v4f __attribute__((ext_vector_type(4)));

// a: [block][k][16 rows], b: [block][k][16 columns], d: [block][16][16]
__global__ __launch_bounds__(64) void chain(const float* a, const float* b, float* d) {
    const int lane = threadIdx.x, i = lane & 15, g = lane >> 4;
    const float* pa = a + static_cast<long>(blockIdx.x) * kK * 16;
    const float* pb = b + static_cast<long>(blockIdx.x) * kK * 16;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0; s < kK; s += 4)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[(s + g) * 16 + i], pb[(s + g) * 16 + i], acc,
                                                   0, 0, 0);
    for (int v = 0; v < 4; ++v)
        d[static_cast<long>(blockIdx.x) * 256 + (4 * g + v) * 16 + i] = acc[v];
}

float from_bits(uint32_t u) {
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}
}  // namespace

int main() {
    std::mt19937 rng(5);
    std::normal_distribution<float> normal;
    const char* kinds[] = {"ordinary", "wide exponents", "denormal", "not finite"};
    const size_t n = static_cast<size_t>(kBlocks) * kK * 16, nd = static_cast<size_t>(kBlocks) * 256;
    std::vector<float> a(n), b(n), d(nd);
    float *da, *db, *dd;
    if (hipMalloc(&da, 4 * n) != hipSuccess || hipMalloc(&db, 4 * n) != hipSuccess ||
        hipMalloc(&dd, 4 * nd) != hipSuccess)
        return std::printf("no memory\n"), 2;
    long bad = 0;
    for (int kind = 0; kind < 4; ++kind) {
        auto draw = [&](int side) {
            const uint32_t u = rng();
            if (kind == 1) {  // products of exponents -180 .. 180, past both ends of the range
                const uint32_t e = 37 + rng() % 181;
                return from_bits((u & 0x807FFFFFu) | e << 23);
            }
            if (kind == 2)  // a denormal times a value around 1
                return side ? normal(rng) : from_bits(u & 0x807FFFFFu);
            if (kind == 3 && u % 400 == 0) return side ? INFINITY : (u & 512 ? NAN : -INFINITY);
            return normal(rng);
        };
        for (size_t i = 0; i < n; ++i) a[i] = draw(0), b[i] = draw(1);
        if (hipMemcpy(da, a.data(), 4 * n, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(db, b.data(), 4 * n, hipMemcpyHostToDevice) != hipSuccess)
            return std::printf("copy failed\n"), 2;
        hipLaunchKernelGGL(chain, dim3(kBlocks), dim3(64), 0, nullptr, da, db, dd);
        if (hipMemcpy(d.data(), dd, 4 * nd, hipMemcpyDeviceToHost) != hipSuccess)
            return std::printf("launch failed\n"), 2;
        long diff = 0, odd = 0;
        for (int blk = 0; blk < kBlocks; ++blk)
            for (int r = 0; r < 16; ++r)
                for (int c = 0; c < 16; ++c) {
                    float want = 0.0f;
                    const size_t base = static_cast<size_t>(blk) * kK * 16;
                    for (int k = 0; k < kK; ++k)
                        want = std::fmaf(a[base + k * 16 + r], b[base + k * 16 + c], want);
                    const float got = d[blk * 256 + r * 16 + c];
                    odd += std::fpclassify(want) != FP_NORMAL;
                    if (std::isnan(want) ? !std::isnan(got) : std::memcmp(&got, &want, 4) != 0)
                        ++diff;
                }
        std::printf("%s: %ld of %zu sums differ (%ld not normal)\n", kinds[kind], diff, nd, odd);
        bad += diff;
    }
    (void)hipFree(da);
    (void)hipFree(db);
    (void)hipFree(dd);
    return bad ? 1 : 0;
}
