// check.hpp -- what the CPU programs of the transfer code share: a check that
// names what failed, the error message the library keeps per thread.
#pragma once

#include <cstdarg>
#include <cstdio>
#include <cstdlib>

#define CHECK(x)                                                    \
  do {                                                              \
    if (!(x)) {                                                     \
      std::printf("FAILED %s (%s:%d)\n", #x, __FILE__, __LINE__);   \
      std::exit(1);                                                 \
    }                                                               \
  } while (0)

namespace erm {
static thread_local char g_msg[1024] = "";
void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(g_msg, sizeof g_msg, fmt, ap);
  va_end(ap);
}
const char* last_error() { return g_msg; }
}  // namespace erm
