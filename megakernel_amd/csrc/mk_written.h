// Which cache rows a handle has written since they were last zeroed.  Plain
// C++ (no HIP), so that the CPU tests run the same code.
#pragma once
#include <algorithm>

namespace mk {

// Rows 0 .. high - 1 may hold something; no row at or past `high` does.
struct WrittenRows {
  int high = 0;

  void wrote(int end) { high = std::max(high, end); }

  // Zero them through clear(rows): rows is `high` rounded up to whole
  // 32-position blocks, and the result says whether every clear was issued.
  // Only then do they count as zero, so that a clear that could not be issued
  // leaves its rows to the next one.
  template <class Clear>
  bool clear(const Clear& clear_rows) {
    if (high > 0 && !clear_rows((high + 31LL) / 32 * 32)) return false;
    high = 0;
    return true;
  }
};

}  // namespace mk
