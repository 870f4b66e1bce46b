// host_rules.h — the host's decisions about a dispatch as plain functions,
// without HIP, so that the runtime and CPU tests call the same ones. Geom is
// MatGeom (common.h) or anything with its fields; gg: gate and up, gd: down.
#pragma once

#include <cstdint>
#include <numeric>

#include "mfma_map.h"

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

// Whether a dispatch of R rows over n experts runs mfma_row_kernel (per-row
// weights and activations; items of up to 128 rows). It pays once experts
// average about 24 rows: 160 experts, D = 5120, I = 1536, int4, layer time of
// the 32-row kernel -> this one: 12.8 rows per expert (uniform routing) 387 ->
// 414 us, 25.6 rows 475 -> 455, 51 rows 859 -> 538; skewed routing 25.6 rows
// 563 -> 485, 89 rows 944 -> 745. With a short K its start and end weigh more
// (K = 1000, 30 rows per expert, int4 71 -> 74 us), so there from 64 rows on,
// or for int8 with many items (128 experts, K = 1536, 31 rows 134 -> 119 us).
// And it needs items to fill the chip: 13 x 12 of them, int4 (8 experts, D =
// 4096, 150 rows each) 101 -> 110 us, int8 128 -> 118; 20 x 2 53 -> 57 us; 35 x 6
// 92 -> 89.
template <class Geom>
bool row_groups(const Geom &gg, const Geom &gd, int R, int n, int ga) {
    if (ga == 32 || !(gg.per_row || gd.per_row)) return false;
    const long items = (long)mmap::row_lead_bound(R, n) * mmap::slab_count(true, gg.O);
    const bool many = (long)R >= (gg.nb >= 64 ? 24L : 64L) * n && items >= (gg.w4 ? 256 : 128);
    return many || (!gg.w4 && (long)R >= 24L * n && items >= 512);
}

// The arm of a dispatch of R rows when none is forced. The GEMV
// reads an expert's weights once per row (again from the caches where rows
// share it), the grouped GEMM once per expert, but a workgroup of the GEMM
// walks all of K block by block: 75 us at D = 5120 however little there is to
// read. Measured, layer times GEMV / GEMM in us. 160 experts, D = 5120, I =
// 1536, top-8: int4 gs = 32 16 rows 56 / 79, 40 rows 107 / 114 (skewed
// popularity 94 / 99), 48 rows 120 / 141 (skewed 102 / 98); per row 32 rows 79 /
// 88; gs = 128 48 rows 115 / 147; int8 16 rows 94 / 98, 24 rows 135 / 133 (skewed
// 128 / 102). 256 experts, D = 6144, I = 2048: int4 40 rows 162 / 181 (skewed 144
// / 137), int8 16 rows 128 / 121. Small layers: 16 experts, D = 2048, I = 768, 32
// rows int4 33 / 44, 24 rows int8 45 / 45; 64 experts, D = 1024, I = 512, 48 rows
// int4 30 / 35, 36 rows int8 36 / 35. Sharing does not turn it round: 1 expert,
// D = 5120, 16 rows int4 37 / 90, int8 59 / 68; 4 experts, D = 2048, 32 rows 28 / 47.
// So the bounds are on the safe side: 48 rows of the 160 experts lose to the
// GEMM only with skewed popularity, and the crossings were not looked for by
// activation mode (per-row activations gain most).
template <class Geom>
bool gemv_pays(const Geom &gg, const Geom &gd, int R) {
    const double bytes = (double)gg.Op * gg.Kp * (gg.w4 ? 1.0 : 2.0) + (double)gd.Op * gd.Kp * (gd.w4 ? 0.5 : 1.0);   // one expert's weights
    if (gg.w4 && gd.w4) return R <= (bytes <= 4e6 ? 48 : bytes <= 12e6 ? 40 : 32);
    return R <= (bytes <= 4e6 ? 24 : bytes <= 25e6 ? 16 : 8);
}

}  // namespace phip
