// Many-row attention over f16 keys of 64 dims (attention_rows.hip).
#include "attention_rows.h"

namespace trit {
bool attention_rows_f16_64(const RowsArgs& a, int max_tk, hipStream_t s) {
    return launch_budget<_Float16, 64>(a, max_tk, s);
}
}  // namespace trit
