// Many-row attention over f32 keys of 64 dims (attention_rows.hip).
#include "attention_rows.h"

namespace trit {
bool attention_rows_f32_64(const RowsArgs& a, int max_tk, hipStream_t s) {
    return launch_budget<float, 64>(a, max_tk, s);
}
}  // namespace trit
