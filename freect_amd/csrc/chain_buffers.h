// chain_buffers.h -- the order in which the buffers of whole chains are
// allocated, so that the faster layout of the filtered projections never takes
// memory that the chains cannot run without.
#pragma once

#include <cstddef>

namespace fct {

struct Buffer {
  void** at;   // null where it is still to be allocated
  size_t bytes;
};

// Filtered projections: their bytes as row pairs and in the interface's layout
// (FP32 rows: half of the pairs; FP16 / BF16 quads: twice).
struct FilteredBuffer {
  void** at;
  size_t pairs, plain;
};

// Allocates the other buffers first, then the filtered projections: all of
// them as pairs (*pairs) if room() bytes hold those, otherwise all in the plain
// layout, if that is smaller.  alloc(at, bytes) returns 0 or an error and leaves
// *at null then; room() is the memory that is free and that later calls on the
// same plans do not need.  What was allocated before an error stays with its
// owner.
template <class Alloc, class Free, class Room>
auto alloc_chain(const Buffer* other, int n_other, const FilteredBuffer* filt, int n_filt,
                 bool* pairs, Alloc alloc, Free release, Room room)
    -> decltype(alloc(nullptr, 0)) {
  decltype(alloc(nullptr, 0)) e{};
  for (int i = 0; i < n_other; ++i)
    if (!*other[i].at && other[i].bytes && (e = alloc(other[i].at, other[i].bytes))) return e;
  size_t as_pairs = 0, plain = 0;
  for (int i = 0; i < n_filt; ++i)
    if (!*filt[i].at) as_pairs += filt[i].pairs, plain += filt[i].plain;
  if (!as_pairs) return e;   // every one is there, in the layout of *pairs
  const bool smaller = plain < as_pairs;
  if (*pairs && (!smaller || room() >= as_pairs)) {
    for (int i = 0; i < n_filt && !e; ++i) e = alloc(filt[i].at, filt[i].pairs);
    if (!e || !smaller) return e;
    for (int i = 0; i < n_filt; ++i) {
      if (*filt[i].at) release(*filt[i].at);
      *filt[i].at = nullptr;
    }
  }
  *pairs = false;
  e = {};
  for (int i = 0; i < n_filt && !e; ++i) e = alloc(filt[i].at, filt[i].plain);
  return e;
}

}  // namespace fct
