// qh_optional.h -- structures that only make a call faster.  Plain C++, without HIP.
#ifndef QH_OPTIONAL_H
#define QH_OPTIONAL_H
#include <new>

// Runs build(), which forms such a structure and returns 0 or an error code.  Without
// the memory for it (the code nomem, or std::bad_alloc) the call goes on without:
// none() notes that there is none and takes back the error that the allocation left.
template <typename Build, typename None>
int qh_optional(int nomem, Build &&build, None &&none) {
  int rc;
  try {
    rc = build();
  } catch (const std::bad_alloc &) {
    rc = nomem;
  }
  if (rc != nomem) return rc;
  none();
  return 0;
}

#endif
