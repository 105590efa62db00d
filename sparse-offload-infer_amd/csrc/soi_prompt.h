// Layout of the token activations that the matrix-core products read (prompt_mfma.hip), written by their producers
// (prompt.hip, prompt_mfma.hip).
#pragma once

#include <stdint.h>

namespace soi {

// "Fragment" layout of x [T, K] (K % 128 == 0, room for T rounded up to 16): per tile of 16 tokens and step of 128
// elements, the four MFMA operands of that step, each 1 KB in lane order (lane = 16 g + token, 8 elements a lane).
// Element k of token t: step k / 128, operand (k / 8) % 4, lane group g = (k / 32) % 4. Eight elements from a
// multiple of 8 stay together, so producers write whole 16-byte units, and a load of an operand is 1 KB contiguous.
__host__ __device__ __forceinline__ int64_t frag_offset(int64_t t, int64_t k, int64_t K) {
    return ((((t >> 4) * (K >> 7) + (k >> 7)) * 4 + ((k >> 3) & 3)) * 64 + ((k >> 5) & 3) * 16 + (t & 15)) * 8 + (k & 7);
}

}  // namespace soi
