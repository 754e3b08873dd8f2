// alloc_retry.h -- allocation that gives the library's own kept memory back
// before it fails (no HIP: also built on its own by the CPU tests).
#pragma once

namespace pkv {

// alloc(); while that runs out of memory (returns oom), once more after trim()
// -- which returns what no queued work uses any more -- and, where may_sync()
// (not while a stream is being captured), once more after sync() and trim().
template <class E, class Alloc, class Trim, class MaySync, class Sync>
E alloc_trimming(E oom, Alloc alloc, Trim trim, MaySync may_sync, Sync sync) {
  E e = alloc();
  if (e != oom) return e;
  trim();
  e = alloc();
  if (e != oom || !may_sync()) return e;
  sync();
  trim();
  return alloc();
}

}  // namespace pkv
