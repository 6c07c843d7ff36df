// bitlinear.hip -- the BitLinear of the reference engine as one call:
// InferenceEngine::bitlinear (src/inference.cu:106-117) runs absmax_reduce_gpu
// into the engine's device scalar d_absmax_, then fused_sparse_bitlinear_gpu.
// Here the scalar (and the activation bit planes) live in a caller workspace:
//   bytes [0, 256)            absmax (float)
//   bytes [256, 256 + P)      bit planes of the quantised activations,
//                             P = 32 * ceil(cols / 32) (the plane layout of
//                             spb_absmax_quantize_planes_*)
// One launch where every block's rows are a few steps of the span kernel (the
// decode shapes: cols % 128 == 0, up to 8192, and ~25,000 rows at 2560 columns):
// each block quantises the vector for itself while its weights arrive, and one
// writes the workspace.  bf16 2560 x 6912: 3.7 + 4.4 us in two launches before,
// 4.7 us now.
// Else, when cols % 8 == 0 and x and the workspace are 16-byte aligned, the
// planes are built once (spb_absmax_quantize_planes_*, one block) and the GEMV reads
// them (spb_fused_sparse_bitlinear_planes_*), instead of every GEMV block
// quantising the vector again; otherwise the reference's pair runs on the
// workspace's absmax.  Both orders give the reference's bits:
//   q = clamp(rint(x * (absmax > 0 ? 127/absmax : 0)), -128, 127),
//   out[r] = 16-bit(float(W q) * ((gamma * absmax) / 127)).
#include <mutex>
#include <string>
#include <type_traits>

#include "bitplane.hpp"
#include "spbitnet_amd.h"

namespace spb {
namespace {

constexpr size_t kAbsmaxBytes = 256;

size_t planes_bytes(int cols) { return 32 * static_cast<size_t>((cols + 31) / 32); }

size_t workspace_bytes(int cols) { return cols > 0 ? kAbsmaxBytes + planes_bytes(cols) : 0; }

bool overlap(const void* a, size_t na, const void* b, size_t nb) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + nb && y < x + na;
}

// The BitLinear in one launch; false (nothing launched) when the shape, the
// alignment or an output over the input (blocks would read what others have
// written) does not allow it.
// Every block quantises the vector itself while its weights are in flight, so
// the launch and the dependent read of the planes go: bf16 2560 x 6912 3.7 + 4.4
// us in two kernels, 4.7 us in one.  The line lies where the span kernel's
// does (rows of a block within 4 steps; past it the weights' time, not the
// second launch, counts) and at two units of 8 columns per thread, which the
// thread holds in registers between the absmax and the planes.
template <class T>
bool bitlinear_span(const uint32_t* meta, const uint32_t* values, const uint16_t* x,
                    uint16_t* output, float gamma, int rows, int cols, int ms, int vs,
                    float* d_absmax, uint32_t* planes, hipStream_t s) {
    if (!bitplane_ok(meta, values, cols, ms, vs) || !aligned(x, 16) || !aligned(planes, 16) ||
        cols > 16 * kBlock ||
        overlap(x, 2 * static_cast<size_t>(cols), output, 2 * static_cast<size_t>(rows)))
        return false;
    const Weights wt{meta, values, rows, cols, ms, vs};
    const DequantOwnSink<T> sink{output, gamma, 0.0f};
    uint4* const p = reinterpret_cast<uint4*>(planes);
    if (cols <= 8 * kBlock)
        return launch_span(wt, AbsmaxPlanes<T, 1>{x, cols / 8, d_absmax, p, 0.0f}, sink, s);
    return launch_span(wt, AbsmaxPlanes<T, 2>{x, cols / 8, d_absmax, p, 0.0f}, sink, s);
}

// The BitLinear on a workspace already checked to hold workspace_bytes(cols).
template <class T>
int bitlinear_ws(const char* fn, const uint32_t* meta, const uint32_t* values, const uint16_t* x,
                 uint16_t* output, float gamma, int rows, int cols, int ms, int vs,
                 uint8_t* ws, hipStream_t s) {
    float* d_absmax = reinterpret_cast<float*>(ws);
    uint32_t* planes = reinterpret_cast<uint32_t*>(ws + kAbsmaxBytes);
    constexpr bool kBf16 = std::is_same<T, BF16>::value;
    int rc;
    if (bitlinear_span<T>(meta, values, x, output, gamma, rows, cols, ms, vs, d_absmax, planes, s)) {
        rc = launch_status(fn);
        if (rc) return rc;
    } else if (cols % 8 == 0 && aligned(x, 16) && aligned(ws, 16)) {
        rc = kBf16 ? spb_absmax_quantize_planes_bf16(x, planes, nullptr, d_absmax, cols, s)
                   : spb_absmax_quantize_planes_f16(x, planes, nullptr, d_absmax, cols, s);
        if (rc == 0)
            rc = kBf16 ? spb_fused_sparse_bitlinear_planes_bf16(meta, values, planes, output,
                                                                d_absmax, gamma, rows, cols, ms,
                                                                vs, s)
                       : spb_fused_sparse_bitlinear_planes_f16(meta, values, planes, output,
                                                               d_absmax, gamma, rows, cols, ms,
                                                               vs, s);
    } else {
        rc = kBf16 ? spb_absmax_reduce_bf16(x, d_absmax, cols, s)
                   : spb_absmax_reduce_f16(x, d_absmax, cols, s);
        if (rc == 0)
            rc = kBf16 ? spb_fused_sparse_bitlinear_bf16(meta, values, x, output, d_absmax, gamma,
                                                         rows, cols, ms, vs, s)
                       : spb_fused_sparse_bitlinear_f16(meta, values, x, output, d_absmax, gamma,
                                                        rows, cols, ms, vs, s);
    }
    if (rc) {
        const std::string inner = last_error();
        set_error("%s: %s", fn, inner.c_str());
    }
    return rc;
}

// Argument checks shared by the entry points (nothing is launched on failure).
int check_bitlinear(const char* fn, const uint32_t* meta, const uint32_t* values,
                    const uint16_t* x, const uint16_t* output, int rows, int cols, int ms,
                    int vs) {
    if (int e = check_weights(fn, meta, values, rows, cols, ms, vs)) return e;
    if (rows && cols && (!x || !output)) return invalid("%s: null activation pointer", fn);
    return 0;
}

template <class T>
int bitlinear(const char* fn, const uint32_t* meta, const uint32_t* values, const uint16_t* x,
              uint16_t* output, float gamma, int rows, int cols, int ms, int vs, void* workspace,
              size_t workspace_bytes_given, spb_stream_t stream) {
    clear_error();
    if (int e = check_bitlinear(fn, meta, values, x, output, rows, cols, ms, vs)) return e;
    if (rows == 0 || cols == 0) return 0;
    if (!workspace) return invalid("%s: null workspace", fn);
    if (!aligned(workspace, 16)) return invalid("%s: workspace must be 16-byte aligned", fn);
    if (workspace_bytes_given < workspace_bytes(cols))
        return invalid("%s: workspace of %zu bytes, %zu needed for %d columns", fn,
                       workspace_bytes_given, workspace_bytes(cols), cols);
    return bitlinear_ws<T>(fn, meta, values, x, output, gamma, rows, cols, ms, vs,
                           static_cast<uint8_t*>(workspace), as_stream(stream));
}

// ---- allocation-free form -------------------------------------------------------
// For callers that cannot allocate (code under HIP graph capture, serving
// loops that forbid hipMalloc): the workspace is `scratch`, a file-scope
// device array of workspace_bytes(kNoAllocMaxCols) bytes.  Each GPU the
// library runs on holds its own copy until the process ends.  Host code never
// passes the array's name to a kernel (on the host it is only a stand-in
// symbol, not a device address): the entry point looks up the copy's device
// address once per device with hipGetSymbolAddress, with that device
// current, and uses that pointer.  Every call on a GPU shares its copy, which
// keeps the last call's contents; nothing in it needs to start at zero (each
// call writes the absmax and every plane word the GEMV reads before reading
// them).  Calls that overlap on one GPU (different streams, host threads)
// race on it.
constexpr int kNoAllocMaxCols = kMaxPlaneCols;  // 32768
constexpr size_t kScratchBytes = kAbsmaxBytes + 32 * (kNoAllocMaxCols / 32);
static_assert(kNoAllocMaxCols % 32 == 0, "planes of the largest vector fill whole groups");

static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
uint8_t* g_scratch[kScratchDevices] = {};

// The device address of the current device's copy of `scratch` (looked up on
// the first call on each device); nullptr with the error recorded on failure.
uint8_t* scratch_on_current_device(const char* fn, int* rc) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        set_error("%s: hipGetDevice: %s", fn, hipGetErrorString(e));
        *rc = static_cast<int>(e);
        return nullptr;
    }
    if (dev < 0 || dev >= kScratchDevices) {
        *rc = invalid("%s: device %d beyond the %d devices the scratch table covers", fn, dev,
                      kScratchDevices);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_error("%s: hipGetSymbolAddress(scratch): %s", fn, hipGetErrorString(e));
            *rc = static_cast<int>(e != hipSuccess ? e : hipErrorInvalidSymbol);
            return nullptr;
        }
        g_scratch[dev] = static_cast<uint8_t*>(ptr);
    }
    return g_scratch[dev];
}

template <class T>
int bitlinear_noalloc(const char* fn, const uint32_t* meta, const uint32_t* values,
                      const uint16_t* x, uint16_t* output, float gamma, int rows, int cols,
                      int ms, int vs, spb_stream_t stream) {
    clear_error();
    if (int e = check_bitlinear(fn, meta, values, x, output, rows, cols, ms, vs)) return e;
    if (rows == 0 || cols == 0) return 0;
    if (cols > kNoAllocMaxCols)
        return invalid("%s: cols=%d exceeds the %d columns the static scratch holds (use "
                       "spb_bitlinear_* with a workspace)", fn, cols, kNoAllocMaxCols);
    int rc = 0;
    uint8_t* ws = scratch_on_current_device(fn, &rc);
    if (!ws) return rc;
    return bitlinear_ws<T>(fn, meta, values, x, output, gamma, rows, cols, ms, vs, ws,
                           as_stream(stream));
}

}  // namespace
}  // namespace spb

using namespace spb;

extern "C" size_t spb_bitlinear_workspace_size(int cols) { return workspace_bytes(cols); }

extern "C" int spb_bitlinear_f16(const uint32_t* meta, const uint32_t* values, const uint16_t* x,
                                 uint16_t* output, float gamma, int rows, int cols,
                                 int meta_row_stride, int values_row_stride, void* workspace,
                                 size_t workspace_size, spb_stream_t stream) {
    return bitlinear<F16>("spb_bitlinear_f16", meta, values, x, output, gamma, rows, cols,
                          meta_row_stride, values_row_stride, workspace, workspace_size, stream);
}

extern "C" int spb_bitlinear_bf16(const uint32_t* meta, const uint32_t* values, const uint16_t* x,
                                  uint16_t* output, float gamma, int rows, int cols,
                                  int meta_row_stride, int values_row_stride, void* workspace,
                                  size_t workspace_size, spb_stream_t stream) {
    return bitlinear<BF16>("spb_bitlinear_bf16", meta, values, x, output, gamma, rows, cols,
                           meta_row_stride, values_row_stride, workspace, workspace_size, stream);
}

extern "C" int spb_bitlinear_f16_noalloc(const uint32_t* meta, const uint32_t* values,
                                         const uint16_t* x, uint16_t* output, float gamma,
                                         int rows, int cols, int meta_row_stride,
                                         int values_row_stride, spb_stream_t stream) {
    return bitlinear_noalloc<F16>("spb_bitlinear_f16_noalloc", meta, values, x, output, gamma,
                                  rows, cols, meta_row_stride, values_row_stride, stream);
}

extern "C" int spb_bitlinear_bf16_noalloc(const uint32_t* meta, const uint32_t* values,
                                          const uint16_t* x, uint16_t* output, float gamma,
                                          int rows, int cols, int meta_row_stride,
                                          int values_row_stride, spb_stream_t stream) {
    return bitlinear_noalloc<BF16>("spb_bitlinear_bf16_noalloc", meta, values, x, output, gamma,
                                   rows, cols, meta_row_stride, values_row_stride, stream);
}
