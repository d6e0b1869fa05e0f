// A C caller that records while host memory runs out: the library's allocations go through this program's
// operator new, which fails on demand.  Nothing may be thrown at the caller, the recorded call itself is
// made, and the incomplete list says so and is not run.  Needs no GPU: the problem is empty.
#include <stdio.h>
#include <stdlib.h>

#include <new>

#include "dcp_hip.h"

static bool g_no_memory = false;
void* operator new(size_t n) {
  void* p = g_no_memory ? nullptr : malloc(n ? n : 1);
  if (p == nullptr) throw std::bad_alloc();
  return p;
}
void* operator new(size_t n, const std::nothrow_t&) noexcept { return g_no_memory ? nullptr : malloc(n ? n : 1); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

#define CHECK(cond)                                  \
  do {                                               \
    if (!(cond)) {                                   \
      printf("failed: %s (%s)\n", #cond, dcp_last_error()); \
      return 1;                                      \
    }                                                \
  } while (0)

static int call() { return dcp_fused_copy_varlen(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 16, 2, nullptr); }

int main() {
  void* list = dcp_record_begin();
  CHECK(list != nullptr);
  CHECK(call() == DCP_OK);
  g_no_memory = true;
  const int status = call();
  g_no_memory = false;
  CHECK(status == DCP_OK);
  CHECK(dcp_record_end() != DCP_OK);
  CHECK(dcp_record_run(list, 0, dcp_record_size(list), nullptr) != DCP_OK);
  dcp_record_free(list);
  g_no_memory = true;
  list = dcp_record_begin();
  g_no_memory = false;
  CHECK(list == nullptr);
  CHECK(call() == DCP_OK);  // (not recorded)
  list = dcp_record_begin();
  CHECK(list != nullptr && call() == DCP_OK && dcp_record_end() == DCP_OK);
  CHECK(dcp_record_size(list) == 1 && dcp_record_run(list, 0, 1, nullptr) == DCP_OK);
  dcp_record_free(list);
  printf("ok\n");
  return 0;
}
