// host_rules.h — the host's decisions about a dispatch as plain functions,
// without HIP, so that the runtime and CPU tests call the same ones.
#pragma once

#include <cstdint>
#include <numeric>

namespace phip {

// Chunked staging of a host-buffer call's x [total][D] f32: the row where
// chunk i of n starts. Chunks start on whole 128-byte cache lines, since the
// host writes chunk i + 1 while the kernel of chunk i reads: no line is read
// that is still being written. A chunk may be empty (few, long rows).
inline int chunk_row(int total, int i, int n, int D) {
    if (i >= n) return total;
    const int lines = 32 / std::gcd(D, 32);   // rows that end on a line
    return (int)((int64_t)total * i / n / lines * lines);
}

}  // namespace phip
