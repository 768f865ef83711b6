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

// The teams of a batch: what is scored is what is launched, no more workgroups than
// are resident, every large instance with a team at once where that fits, teams of
// exactly the configured size on request.
static void check_batch_teams() {
  for (int resident : {256, 512, 304, 100, 7})
    for (int count : {1, 2, 7, 8, 9, 20, 65, 70, 128, 300, 5000})
      for (int big : {1, 2, 7, 8, 9, 20, 64, 65, 128, 300})
        for (int c : {2, 3, 4, 8, 32, 100})
          for (double most : {1e5, 4e6, 16.8e6, 1e9})
            for (int grow = 0; grow < 2; grow++) {
              if (big > count || c > resident) continue;
              const BatchPick p = batch_pick(count, big, c, resident, 512, most, most / 50, grow != 0);
              CHECK(p.teams >= 1 && (long)p.teams * p.c <= resident, "%d/%d c %d of %d: %d teams of %d", count,
                    big, c, resident, p.teams, p.c);
              CHECK(p.c >= c && (p.c == c || grow), "teams of %d for %d", p.c, c);
              if (p.c > c) {
                CHECK(p.teams >= big, "grown teams of %d leave large instances waiting", p.c);
                CHECK(most / p.c >= GROW_BYTES, "teams of %d have less than the least work", p.c);
                CHECK(p.c % c == 0 && ((p.c / c) & (p.c / c - 1)) == 0, "teams of %d for %d", p.c, c);
              }
              // as many as want one, in whole groups of eight where those fit
              const int want = big + (count - big + p.c - 1) / p.c, full = (want + 7) / 8 * 8;
              if (full <= resident / p.c)
                CHECK(p.teams >= want, "%d/%d c %d of %d: %d teams for %d", count, big, p.c, resident, p.teams, want);
            }
  const BatchPick p = batch_pick(70, 65, 4, 512, 512, 1e5, 1e4, true);
  CHECK(p.c == 4 && p.teams == 72, "70 instances, 65 in teams of 4: %d teams of %d", p.teams, p.c);
}

int main() {
  check_form();
  check_batch_teams();
  if (fails) return 1;
  printf("dispatch checks passed\n");
  return 0;
}
