// CPU check of the host's choices of forms, teams and slices (built with g++ and
// AddressSanitizer/UBSan by tests/test_dispatch_cpu.py).
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../gaga_amd/csrc/xcs_hostlogic.h"

using namespace xcs;

static int fails = 0;
#define CHECK(c, ...)               \
  do {                              \
    if (!(c)) {                     \
      fprintf(stderr, __VA_ARGS__); \
      fprintf(stderr, "\n");        \
      if (++fails > 20) exit(1);    \
    }                               \
  } while (0)

// A warm start is read by the general form only.
static void check_form() {
  for (int planned : {FORM_GENERAL, FORM_RESIDENT, FORM_SPLIT}) {
    CHECK(solve_form(planned, true) == FORM_GENERAL, "form %d takes a warm start", planned);
    CHECK(solve_form(planned, false) == planned, "form %d is not kept", planned);
  }
}

int main() {
  check_form();
  if (fails) return 1;
  printf("dispatch checks passed\n");
  return 0;
}
