// The library's error text (apc_last_error) and argument checks, shared by its translation units.
#ifndef APCOST_ERROR_H
#define APCOST_ERROR_H

#include "apcost.h"

namespace apc_internal {
// Stores the formatted message for this thread and returns `code`.
__attribute__((visibility("hidden"), format(printf, 2, 3))) int fail(int code, const char *fmt, ...);
// The message of the exception in flight (a vector that no memory could be had for): called in a handler at an entry
// point, which no exception may leave.
__attribute__((visibility("hidden"))) int thrown(const char *who);
// The parameters' ranges and reciprocals.
__attribute__((visibility("hidden"))) int check_params(const apc_params *p);
}  // namespace apc_internal

#endif
