// Sizes and offsets whose products leave 32 bits (plain C++, host and device).
#pragma once

#include <cstddef>

// Offset of plane n of a stack of 2-D planes of P2 points: a stack of 16 planes
// leaves the ints from 2^27 points a plane on.
constexpr size_t plane_at(int n, int P2) { return (size_t)n * (size_t)P2; }

// Whether every byte of an FP64 level of P2 points has a 32-bit offset, as the
// kernels that address a level through a buffer descriptor need.
constexpr bool level_fits(long long P2) { return P2 * 8 < (1LL << 32); }
