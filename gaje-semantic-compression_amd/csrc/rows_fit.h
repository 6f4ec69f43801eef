// How many rows a pass over several token rows gets buffers for.
#pragma once

#include <algorithm>
#include <cstdint>

namespace gaje {

// Rows (at most `want`, which is at most `most`) that buffers of `have` rows take, or that
// reserve(rows) has made room for: a power of two from `want` up, so that prompts that
// lengthen slowly do not reserve on each call, and where that fails half as many at a
// time; 0 if not even two rows found room (reserve then holds nothing).
template <class Reserve>
int64_t rows_fit(int64_t want, int64_t have, int64_t most, Reserve reserve) {
    if (want <= have) return want;
    int64_t rows = 2;
    while (rows < want) rows *= 2;
    for (rows = std::min(rows, most); rows >= 2; rows /= 2)
        if (reserve(rows)) return std::min(rows, want);
    return 0;
}

}  // namespace gaje
