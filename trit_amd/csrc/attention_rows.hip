// Trit's attention of many query rows: the choice of an instance
// (attention_rows.h). Key type by head size, each is a code object of its own,
// since a code object loads whole with its first kernel: all of them in one (750 KB)
// cost a process's first prompt about 1.4 ms, one of four (170-220 KB) 0.4.
#include <algorithm>

#include "decoder_impl.h"
#include "internal.h"

namespace trit {

bool attention_rows_f16_64(const RowsArgs& a, int max_tk, hipStream_t s);
bool attention_rows_f16_128(const RowsArgs& a, int max_tk, hipStream_t s);
bool attention_rows_f32_64(const RowsArgs& a, int max_tk, hipStream_t s);
bool attention_rows_f32_128(const RowsArgs& a, int max_tk, hipStream_t s);

bool attention_rows_mfma(RowsArgs a, int hd, bool f16, int max_tk, hipStream_t s) {
    if (hd != 64 && hd != 128) return false;
    if (a.pos_stride % 4 != 0 || a.head_stride % 4 != 0) return false;
    a.window_tiles = (std::min(a.window, a.rows) + 15) / 16;
    a.tiles = a.rows / a.window * a.window_tiles + (a.rows % a.window + 15) / 16;
    if ((int64_t)a.tiles * a.heads > (1 << 30)) return false;
    // 32-bit byte offsets of a tile past the last key.
    if ((max_tk + 8 * 16 * 32) * (int64_t)a.pos_stride * (f16 ? 2 : 4) >= (int64_t)1 << 31) return false;
    if (f16) return hd == 64 ? attention_rows_f16_64(a, max_tk, s) : attention_rows_f16_128(a, max_tk, s);
    return hd == 64 ? attention_rows_f32_64(a, max_tk, s) : attention_rows_f32_128(a, max_tk, s);
}

}  // namespace trit
