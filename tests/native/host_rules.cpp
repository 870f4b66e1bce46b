// The runtime's host decisions (peregrine_amd/csrc/host_rules.h) for the tests.
#include "../../peregrine_amd/csrc/host_rules.h"

using namespace phip;

namespace {
struct Geom {
    int Kp, nb, O, Op, w4, per_row;
};
Geom geom(int K, int O, int w4, int per_row) {
    return Geom{(K + 31) / 32 * 32, (K + 31) / 32, O, (O + 63) / 64 * 64, w4, per_row};
}
}  // namespace

extern "C" int chunk_row_c(int total, int i, int n, int D) { return chunk_row(total, i, n, D); }
extern "C" int gemv_pays_c(int D, int I, int w4, int w4_down, int R) {
    return gemv_pays(geom(D, I, w4, 1), geom(I, D, w4_down, 1), R);
}
extern "C" int row_groups_c(int D, int I, int w4, int per_row, int per_row_down, int R, int n, int ga) {
    return row_groups(geom(D, I, w4, per_row), geom(I, D, w4, per_row_down), R, n, ga);
}
