// The engines' host code under a HIP runtime that fails on demand, on the CPU
// (fake_hip.hpp).
//   engine_faults launches   every launch of a prompt's generate, and of the
//                            engines' create, failed once: none may return 0
//   engine_faults memory     creates on a device with less and less memory: the
//                            prompts' passes get shorter before create fails
//   engine_faults folds      launches of a prompt: one less per layer where the
//                            o projection's producer folds the splits itself
// Prints one line per check and returns the number of failed ones.
#include <cstdio>
#include <string>
#include <vector>

#include "fake_hip.hpp"
#include "spbitnet_amd.h"

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
        g_pending = hipErrorNotReady;
        check(e.generate(lens) == 0, kind + ": generate afterwards, an earlier call's error pending");
        g_pending = hipErrorNotReady;
        Engine f;
        check(f.create(s, 4096, batch) == 0, kind + ": create with an earlier call's error pending");
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

void folds() {
    // prompts of 1-4, 5-8 and more splits, heads of a token 1024 and 4096 wide
    const bool narrow[3] = {true, true, false}, wide[3] = {true, false, false};
    for (int heads : {8, 32}) {
        const Shape s = shape(heads, 8, 128, 1024, 2, 1024);
        Engine e;
        check(e.create(s, 1024, 0) == 0, "create");
        long most = 0, got[3];
        for (int k : {2, 1, 0}) {
            const int tokens[3] = {257, 513, 514};  // the last is a step's
            arm(-1);
            check(e.generate({tokens[k]}) == 0, "generate");
            got[k] = g_launches;
            most = got[k] > most ? got[k] : most;
        }
        for (int k = 0; k < 3; ++k)
            check(got[k] == most - ((heads == 8 ? narrow : wide)[k] ? 2 : 0),
                  std::to_string(128 * heads) + " wide, prompt " + std::to_string(k) + ": " +
                      std::to_string(got[k]) + " launches of " + std::to_string(most));
    }
}
}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "launches") launches();
    else if (what == "memory") memory();
    else if (what == "folds") folds();
    else return std::fprintf(stderr, "usage: %s launches|memory|folds\n", argv[0]), 2;
    return g_bad;
}
