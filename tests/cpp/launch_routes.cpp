// Which kernel a call launches, by its grid, under the fake runtime of
// fake_hip.hpp (256 CUs): the lines between the tiles of the sparse GEMMs and
// between the forms of the per-op attention.
// Prints one line per check and returns the number of failed ones.
#include <cstdio>
#include <vector>

#include "fake_hip.hpp"
#include "spbitnet_amd.h"

namespace {
alignas(64) uint32_t g_words[1024];
int8_t* const g_x = reinterpret_cast<int8_t*>(g_words);
int32_t* const g_y = reinterpret_cast<int32_t*>(g_words);
int g_bad = 0;

// One launch whose blocks are tile_rows x tile_tokens.
void check(const char* what, int rc, int rows, int cols, int n, int tile_rows, int tile_tokens) {
    const bool ok = rc == 0 && g_launches == 1 &&
                    static_cast<int>(g_grid.x) == (rows + tile_rows - 1) / tile_rows &&
                    static_cast<int>(g_grid.y) == (n + tile_tokens - 1) / tile_tokens;
    std::printf("%s %s %d x %d, n = %d: %ld launches of %u x %u, tiles of %d x %d expected\n",
                ok ? "ok  " : "FAIL", what, rows, cols, n, g_launches, g_grid.x, g_grid.y,
                tile_rows, tile_tokens);
    g_bad += !ok;
}

void ternary(int rows, int cols, int n, int tile_rows, int tile_tokens) {
    g_launches = 0;
    const int rc = spb_sparse_ternary_gemm(g_words, g_words, g_x, g_y, rows, cols, n,
                                           (cols + 127) / 128 * 4, (cols + 255) / 256 * 4, nullptr);
    check("ternary", rc, rows, cols, n, tile_rows, tile_tokens);
}

void sparse_i8(int m, int k, int n, int tile_rows, int tile_tokens) {
    g_launches = 0;
    check("int8", spb_sparse_i8_gemm(g_words, g_x, g_y, m, k, n, nullptr), m, k, n, tile_rows,
          tile_tokens);
}

// Scores with the grid of 16 positions (head_dim 128) x kv heads x parts of a
// group, outputs with that of head_dim 128 / 8 x kv heads x parts of a group, or
// of one block per head (parts 0).
void attention(int nh, int nkv, int seq, int score_parts, int output_parts) {
    const uint16_t* w = reinterpret_cast<const uint16_t*>(g_words);
    float* f = reinterpret_cast<float*>(g_words);
    g_launches = 0;
    const int r0 = spb_attention_scores_f16(w, w, f, nh, nkv, 128, 8192, seq, 1.0f, nullptr);
    const dim3 s = g_grid;
    const int r1 = spb_attention_output_f16(f, w, reinterpret_cast<uint16_t*>(g_words), nh, nkv,
                                            128, 8192, seq, nullptr);
    const dim3 o = g_grid;
    const dim3 os = output_parts ? dim3(16, nkv, output_parts) : dim3(nh);
    const bool ok = r0 == 0 && r1 == 0 && g_launches == 2 &&
                    static_cast<int>(s.x) == (seq + 15) / 16 && static_cast<int>(s.y) == nkv &&
                    static_cast<int>(s.z) == score_parts && o.x == os.x && o.y == os.y &&
                    o.z == os.z;
    std::printf("%s attention %d on %d, %d positions: scores %u x %u x %u, output %u x %u x %u\n",
                ok ? "ok  " : "FAIL", nh, nkv, seq, s.x, s.y, s.z, o.x, o.y, o.z);
    g_bad += !ok;
}
}  // namespace

int main() {
    // the wide kernel from 384 blocks on
    ternary(6144, 2560, 2048, 256, 128);
    ternary(5888, 2560, 2048, 128, 64);
    // few tokens of many rows
    ternary(98304, 2560, 16, 256, 128);
    ternary(98304, 2560, 17, 64, 32);
    ternary(552960, 2560, 32, 64, 32);
    ternary(98304, 2560, 33, 256, 128);
    // a little past two blocks per CU
    ternary(8192, 1024, 2048, 256, 128);
    ternary(8193, 1024, 2048, 128, 64);
    ternary(9216, 5120, 2048, 128, 64);
    ternary(9217, 1024, 2048, 256, 128);
    ternary(8448, 5376, 2048, 256, 128);
    sparse_i8(40960, 2560, 1, 32, 16);
    sparse_i8(40960, 2560, 16, 32, 16);
    sparse_i8(40960, 2560, 32, 64, 32);
    sparse_i8(100352, 2560, 32, 96, 32);
    sparse_i8(41984, 6912, 32, 128, 32);
    sparse_i8(40960, 2560, 33, 256, 128);
    sparse_i8(6912, 2560, 768, 256, 128);
    sparse_i8(6912, 2560, 640, 96, 32);
    // heads of a group over blocks until there are 4 per CU
    attention(64, 1, 1, 64, 0);
    attention(64, 1, 24, 64, 0);
    attention(64, 1, 25, 64, 32);
    attention(64, 1, 1000, 16, 16);
    attention(8, 1, 1, 8, 0);
    attention(8, 1, 11, 8, 8);
    attention(8, 1, 8192, 2, 2);
    attention(20, 5, 13, 4, 0);
    attention(20, 5, 512, 4, 4);
    attention(20, 5, 513, 4, 1);
    attention(20, 5, 2500, 1, 1);
    return g_bad;
}
