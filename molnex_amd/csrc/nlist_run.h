// Part of a run of pairs that lies within the output (csrc/nlist.hip).  Plain C++ (constexpr: also
// a device function), so that the CPU tests compile it.
#pragma once

#include <cstdint>

namespace mnx {

// Of the components of `pairs` consecutive pairs (three each), starting with pair `first`, how many lie within
// `capacity` pairs: 64-bit until bounded, as a list may run past the output by more than 2^31 components.
constexpr int run_components(int64_t first, int64_t pairs, int64_t capacity) {
    const int64_t left = capacity - first;
    return left <= 0 ? 0 : int(3 * (left < pairs ? left : pairs));
}

}  // namespace mnx
