// The engines' host code under a HIP runtime that fails on demand, on the CPU:
// this program defines the runtime calls that the library makes (the
// executable's definitions come before libamdhip64's), with host memory for
// device memory, launches that run nothing, a limit on the device's memory and
// a launch that fails.
//   engine_faults launches   every launch of a prompt's generate, and of the
//                            engines' create, failed once: none may return 0
//   engine_faults memory     creates on a device with less and less memory: the
//                            prompts' passes get shorter before create fails
// Prints one line per check and returns the number of failed ones.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "spbitnet_amd.h"

// ---- the runtime ---------------------------------------------------------------

namespace {
hipError_t g_pending = hipSuccess;  // what hipGetLastError returns
size_t g_limit = ~size_t{0}, g_used = 0;
std::map<void*, size_t> g_blocks;
long g_launches = 0, g_fail_at = -1;

hipError_t fail(hipError_t e) {
    g_pending = e;
    return e;
}
template <class T>
hipError_t handle(T* out) {
    *out = reinterpret_cast<T>(std::malloc(1));
    return hipSuccess;
}
template <class T>
hipError_t drop(T h) {
    std::free(reinterpret_cast<void*>(h));
    return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = *b = dim3(1);
    *lds = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    return g_launches++ == g_fail_at ? fail(hipErrorLaunchOutOfResources) : hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_pending;
    g_pending = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_limit - g_used) return fail(hipErrorOutOfMemory);
    *p = std::malloc(n);
    if (!*p) return fail(hipErrorOutOfMemory);
    g_blocks[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    g_used -= g_blocks[p];
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    return std::memset(d, v, n), hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return drop(s); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return drop(e); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return handle(x);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return drop(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return drop(x); }
}

// ---- a model whose weights nothing reads -------------------------------------------

namespace {
alignas(64) uint32_t g_words[1024];

struct Shape {
    spb_model_config cfg{};
    std::vector<spb_transformer_layer> layers;
};

Shape shape(int heads, int kv_heads, int head_dim, int ffn, int nlayers, int max_pos) {
    const int H = heads * head_dim, kvd = kv_heads * head_dim;
    Shape s;
    s.cfg = {H, nlayers, heads, kv_heads, ffn, 1024, max_pos, head_dim, 1e-5f, 1e4f, 1, 2};
    auto lin = [](int rows, int cols) {
        return spb_sparse_linear{g_words, g_words, 1.0f, rows, cols, (cols + 127) / 128 * 4,
                                 (cols + 255) / 256 * 4};
    };
    const float* w = reinterpret_cast<const float*>(g_words);
    for (int l = 0; l < nlayers; ++l)
        s.layers.push_back({lin(H, H), lin(kvd, H), lin(kvd, H), lin(H, H), lin(ffn, H),
                            lin(ffn, H), lin(H, ffn), w, w, w, w});
    return s;
}

int g_bad = 0;
void check(bool ok, const std::string& what) {
    std::printf("%s %s\n", ok ? "ok  " : "FAIL", what.c_str());
    g_bad += !ok;
}

const uint16_t* half_words() { return reinterpret_cast<const uint16_t*>(g_words); }
const float* float_words() { return reinterpret_cast<const float*>(g_words); }

// One engine of one sequence (batch 0) or a batch engine, under one interface.
struct Engine {
    spb_engine* one = nullptr;
    spb_batch_engine* many = nullptr;
    int create(const Shape& s, int max_seq, int batch) {
        return batch == 0 ? spb_engine_create(&s.cfg, s.layers.data(), half_words(), nullptr,
                                              float_words(), max_seq, &one)
                          : spb_batch_engine_create(&s.cfg, s.layers.data(), half_words(), nullptr,
                                                    float_words(), max_seq, batch, &many);
    }
    int generate(const std::vector<int>& lens) {
        std::vector<int> prompt, out(lens.size() + 1), got(lens.size());
        for (int n : lens) prompt.insert(prompt.end(), n, 3);
        return one ? spb_engine_generate(one, prompt.data(), lens[0], 1, 0, out.data(), got.data())
                   : spb_batch_engine_generate(many, prompt.data(), lens.data(),
                                               static_cast<int>(lens.size()), 1, 0, out.data(),
                                               got.data());
    }
    ~Engine() {
        if (one) spb_engine_destroy(one);
        if (many) spb_batch_engine_destroy(many);
    }
};

void arm(long at) {
    g_launches = 0;
    g_fail_at = at;
}

void launches() {
    const Shape s = shape(8, 2, 64, 1024, 2, 4096);
    for (int batch : {0, 3}) {
        const std::string kind = batch ? "batch engine" : "engine";
        Engine e;
        arm(-1);
        check(e.create(s, 4096, batch) == 0, kind + ": create");
        const long creating = g_launches;
        // a pass that ends inside a prompt and one after it
        const std::vector<int> lens = batch ? std::vector<int>{40, 2100, 1} : std::vector<int>{2100};
        arm(-1);
        check(e.generate(lens) == 0, kind + ": generate");
        const long total = g_launches;
        long silent = 0, unnamed = 0;
        for (long i = 0; i < total; ++i) {
            arm(i);
            const int rc = e.generate(lens);
            silent += rc == 0;
            unnamed += rc != 0 && !spb_last_error_string()[0];
            g_pending = hipSuccess;
        }
        check(total > 0 && silent == 0 && unnamed == 0,
              kind + ": generate with a failing launch, " + std::to_string(silent) + " of " +
                  std::to_string(total) + " returned 0, " + std::to_string(unnamed) +
                  " without a message");
        silent = 0;
        for (long i = 0; i < creating; ++i) {
            arm(i);
            Engine f;
            silent += f.create(s, 4096, batch) == 0 || f.one || f.many;
            g_pending = hipSuccess;
        }
        check(creating > 0 && silent == 0, kind + ": create with a failing launch, " +
                                               std::to_string(silent) + " of " +
                                               std::to_string(creating) + " returned 0");
        arm(-1);
        check(e.generate(lens) == 0, kind + ": generate afterwards");
    }
}

void memory() {
    const Shape s = shape(8, 2, 64, 1024, 2, 4096);
    for (int batch : {0, 3}) {
        const std::string kind = batch ? "batch engine" : "engine";
        const std::vector<int> lens = batch ? std::vector<int>{40, 2100, 1} : std::vector<int>{2100};
        size_t all = 0;
        long launched = 0;
        for (int part = 0; part < 5; ++part) {  // 1, 1/2, ... 1/16 of the memory that create takes
            g_limit = part ? all >> part : ~size_t{0};
            Engine e;
            const int rc = e.create(s, 4096, batch);
            if (!part) all = g_used;
            arm(-1);
            const bool ran = rc == 0 && g_pending == hipSuccess && e.generate(lens) == 0;
            check(ran && g_launches >= launched,
                  kind + ": 1/" + std::to_string(1 << part) + " of " + std::to_string(all >> 20) +
                      " MB, " + std::to_string(g_launches) + " launches");
            launched = g_launches;
        }
        g_limit = 1 << 20;
        {
            Engine e;
            check(e.create(s, 4096, batch) != 0 && g_used == 0 && g_pending == hipSuccess,
                  kind + ": 1 MB refused, all given back");
        }
        g_limit = ~size_t{0};
        Engine e;  // prompts that cannot fill a pass of 2048 tokens
        check(e.create(s, 64, batch) == 0 && g_used < all / 16,
              kind + ": 64 positions take " + std::to_string(g_used >> 20) + " MB");
    }
}
}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "launches") launches();
    else if (what == "memory") memory();
    else return std::fprintf(stderr, "usage: %s launches|memory\n", argv[0]), 2;
    return g_bad;
}
