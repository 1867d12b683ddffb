// Device memory that the reverse sweep takes for stage records.
#pragma once

#include <algorithm>
#include <cstddef>

namespace gocfd {
namespace capi {

// How many blocks of stage records (block bytes each, at most limit of them) a
// vjp keeps beside its fixed bytes of checkpoints: together a quarter of the
// device memory that is free or already held for them. Counting the held bytes
// keeps the answer of one call for the next one with the same arguments, which
// then allocates nothing; what is held may always be used.
inline int kept_blocks(size_t free, size_t held, size_t fixed, size_t block, int limit) {
  const size_t room = std::max(held, (free + held) / 4);
  return room > fixed ? int(std::min(size_t(limit), (room - fixed) / block)) : 0;
}

}  // namespace capi
}  // namespace gocfd
