// The runtime's host decisions (peregrine_amd/csrc/host_rules.h) for the tests.
#include "../../peregrine_amd/csrc/host_rules.h"

using namespace phip;

extern "C" int chunk_row_c(int total, int i, int n, int D) { return chunk_row(total, i, n, D); }
