// Shared by the int8 matrix-core projections: vector types and the biased
// accumulator start.
#pragma once
#include <stdint.h>

namespace ornith {

// Integer dots start from the bits of kDotBias = 1.5 * 2^23, so the int32
// result read as fp32 is kDotBias + dot exactly (|dot| < 2^19 << 2^22); with
// nb = -sa * kDotBias (exact: sa is an fp16 value, 11 significant bits, and
// kDotBias = 3 * 2^22) fma(sa, kDotBias + dot, nb) rounds sa * dot once:
// RN(sa * dot) without an integer-to-float conversion.
constexpr float kDotBias = 12582912.0f;
constexpr int kDotBiasBits = 0x4B400000;

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

}  // namespace ornith
