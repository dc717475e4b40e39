// Error reporting, library identity, launch grids.
#include "common.hpp"

namespace mv {

char *last_error_buffer() {
  static thread_local char buf[512] = {0};
  return buf;
}

int fail(int status, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(last_error_buffer(), 512, fmt, ap);
  va_end(ap);
  return status;
}

dim3 linear_grid(long workgroups, int threads) {
  const long row = ((1L << 32) - 1) / threads, rows = (workgroups + row - 1) / row;
  return dim3(static_cast<unsigned>((workgroups + rows - 1) / rows), static_cast<unsigned>(rows));
}

}  // namespace mv

extern "C" {
const char *mv_last_error(void) { return mv::last_error_buffer(); }
int mv_version(void) { return 1; }
}
