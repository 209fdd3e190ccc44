// Many-row attention over f16 keys of 128 dims (attention_rows.hip).
#include "attention_rows.h"

namespace trit {
bool attention_rows_f16_128(const RowsArgs& a, int max_tk, hipStream_t s) {
    return launch_budget<_Float16, 128>(a, max_tk, s);
}
}  // namespace trit
