// The host executor of the grid operators (grid_check.cpp) with every buffer
// filled with 0x7f bytes where it is mapped, as device memory may hold anything
// when it is allocated: grid_check.cpp then sets what the library sets at
// creation.  A list counter that a step reads before it clears it starts at
// 0x7f7f7f7f, far past its list.
#include <string.h>
#include <sys/mman.h>

static int mprotect_poisoned(void *p, size_t n, int prot)
{
  const int r = mprotect(p, n, prot);
  if (r == 0) memset(p, 0x7f, n);
  return r;
}
#define mprotect mprotect_poisoned
#include "grid_check.cpp"
