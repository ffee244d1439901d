// split3.hpp — the exact three-way BF16 split of FP32 values behind the
// matrix-core FP32 products of a 0/1 bitmap (spmm_planes.hip, spmm_direct.hip).
//
// An FP32 value has 24 significand bits, a BF16 value 8: b = hi + mid + lo
// with hi the top 8 bits of b, mid the top 8 of what is left and lo the rest,
// all three BF16 and without any rounding.  A's entries are 0 or 1, so every
// product is one of the three parts itself, and A·lo + A·mid + A·hi in FP32
// accumulators is the FP32 sum of the selected B rows in another order.
//
// The matrix unit does not round its sums to nearest, so one accumulator must
// not take all 3 K / 32 steps: chained like that at K = 4096 and 50% density they
// were 2.6e-7 of |A|·|B| off, against 9.8e-8 for the vector-add kernel.  The
// kernels keep the chains of the large parts short (see there); both are closer
// to the 64-bit product than the vector-add kernels over 1% to 100% density.
//
// Range: the parts of |b| in [2^-100, 2^128) are normal BF16 numbers.  Of a
// smaller b bits may be lost, and an Inf or NaN would spread to the rows that
// do not select it (0 x Inf).  The product over planes leaves columns that hold
// such values to the vector adds (spmm_planes.hip); the one-launch product, which
// meets them on the way, sums an output that is not finite, or is below 2^-80 where
// some b was tiny, again from A's bits and B in FP32 in ascending k, as the
// vector-add kernels do.
#pragma once

#include "mfma_common.hpp"

namespace bws {
namespace {

constexpr int kPlanes = 3;
constexpr uint32_t kTinyBits = (127u - 100u) << 23;  // 2^-100
constexpr uint32_t kHugeBits = (127u + 96u) << 23;   // 2^96
constexpr float kSmallOut = 0x1p-80f;

// 0/1 A fragment from a bitmap word (MSB first): K slot 8q + e of the 32-wide
// step is bit 7 - e of x, the word's byte q from the top.  For z = x | (x << 17),
// (z & (0x10001 << (7 - 2p))) * (ONE >> (7 - 2p)) puts ONE (BF16 1.0) into the low
// half iff slot 2p is set and into the high half iff slot 2p + 1 is.
__device__ __forceinline__ uint4 a_frag01(uint32_t w, int q) {
  const uint32_t x = __builtin_amdgcn_ubfe(w, 24 - 8 * q, 8);
  const uint32_t z = x | (x << 17);
  return make_uint4((uint32_t)__umul24(z & 0x00800080u, 0x3F80u >> 7),
                    (uint32_t)__umul24(z & 0x00200020u, 0x3F80u >> 5),
                    (uint32_t)__umul24(z & 0x00080008u, 0x3F80u >> 3),
                    (uint32_t)__umul24(z & 0x00020002u, 0x3F80u >> 1));
}

}  // namespace
}  // namespace bws
