// A buffer that is kept between calls and grown when a call needs more.
#pragma once
#include <stdint.h>

// Makes p hold at least `need` units, `grown` of them when it has to be made
// anew (its contents are not kept). The capacity falls to 0 with the old buffer:
// when the allocation fails, a later call that needs less finds no buffer and
// allocates, instead of taking the old capacity for the null pointer.
// release(p) frees; alloc(&p, units) returns 0 or an error, which is returned.
template <typename T, typename Free, typename Alloc>
static inline auto keep_at_least(T *&p, int64_t &cap, int64_t need, int64_t grown, Free release, Alloc alloc)
  -> decltype(alloc(&p, grown))
{
  if (need <= cap) return {};
  if (p) release(p);
  p = nullptr; cap = 0;
  const auto e = alloc(&p, grown);
  if (e != decltype(alloc(&p, grown)){}) { p = nullptr; return e; }
  cap = grown;
  return e;
}
