// The keys of one part of a split forward (FwdParams::nsplit).
#pragma once

#include "sdpa_params.hpp"

namespace theria {

struct FwdPart {
  int64_t key0;  // first key
  int keys;      // number of keys
};

// Whole 64-key tiles, the same number in every part but the last.
__device__ __forceinline__ FwdPart fwd_part(const Shape& s, int nsplit, int part) {
  const int per = ((s.M + 63) / 64 + nsplit - 1) / nsplit * 64;
  return FwdPart{(int64_t)part * per, min(per, s.M - part * per)};
}

}  // namespace theria
