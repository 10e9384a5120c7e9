// Growth of a buffer that kernels of earlier and later calls write through.
#pragma once

namespace bl {

// *buf with room for n elements (its contents are not kept).  The larger
// buffer is had before the old one is given back: when take(n) has none
// (null), the old one stays, with its capacity, and false is returned.
template <typename T, typename N, typename Take, typename Give>
bool grow(T** buf, N* cap, N n, Take take, Give give) {
  if (*buf && *cap >= n) return true;
  T* const p = take(n);
  if (!p) return false;
  if (*buf) give(*buf);
  *buf = p;
  *cap = n;
  return true;
}

}  // namespace bl
