// keep_at_least with an allocator that can be made to fail: prints what a
// sequence of calls (units needed; negative: this allocation fails) leaves.
#include <stdio.h>
#include <stdlib.h>
#include "p7g_keep.h"

enum Err { OK = 0, NOMEM = 2 };
static bool fail;
static int live, calls;

static void release(void *p) { free(p); live--; }
static Err alloc(float **p, int64_t n)
{
  calls++;
  if (fail) { *p = (float *) 0x10; return NOMEM; }     // whatever a failed call leaves is not used
  *p = (float *) malloc(sizeof(float) * (size_t) n);
  live++;
  return OK;
}

int main(int argc, char **argv)
{
  float *p = nullptr;
  int64_t cap = 0;
  for (int i = 1; i < argc; i++) {
    const long need = atol(argv[i]);
    fail = need < 0;
    const Err e = keep_at_least(p, cap, labs(need), labs(need), release, alloc);
    if (e == OK) p[labs(need) - 1] = 1.0f;
    printf("%d %ld %d %d %d\n", (int) e, (long) cap, p != nullptr, live, calls);
  }
  free(p);
  return 0;
}
