// Panel order: the activations of a prompt pass.  The rows are cut into panels
// of 32, each panel in the skinny GEMMs' operand order over its K values (32 x K
// bf16, 1 KiB blocks of 16 rows x 32 k): panel p starts at p * 32 * K.
#pragma once

#include "decode_common.h"

namespace tfd {

__device__ __forceinline__ int64_t panel_off(int64_t m, int k, int K) {
  const int r = (int)(m & 31);
  return (m >> 5) * 32 * K +
         ((int64_t)((k >> 5) * 2 + (r >> 4)) * 64 + (r & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}

}  // namespace tfd
