// The numbers by which a call's result chunks are marked as ready (stage_out, frk_runtime.cpp): plain C++, no device code.
#pragma once

#include <cstddef>
#include <cstdint>

namespace frk {

// The number of the call behind the one numbered `last` (0: none yet), one that no flag holds.  A flag keeps the number of the last call
// that had its chunk, so when all 32-bit numbers are used up -- a day and a half of calls of 30 us -- they are cleared and the
// numbers start again.  (A call has taken all of its chunks before the next one asks: no kernel is about to raise a flag.)
inline uint32_t next_epoch(uint32_t last, uint32_t *flags, size_t n_flags) {
    if (last != UINT32_MAX) return last + 1;
    for (size_t i = 0; i < n_flags; i++) flags[i] = 0;
    return 1;
}

}  // namespace frk
