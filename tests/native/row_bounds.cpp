// Host-side checker of mfma_row_kernel's work items, copies and LDS layout,
// through the same functions (peregrine_amd/csrc/mfma_map.h): every (M tile,
// slab) is computed by exactly one item, every 16-byte copy of activations and
// weights lies inside its buffer, and the operand reads of a stage find the
// piece they want where a copy put it. Returns the number of violations.
#include <cstdio>
#include <vector>

#include "../../peregrine_amd/csrc/mfma_map.h"

using namespace phip::mmap;

static long g_bad = 0;
static void need(bool ok, const char *what, long a, long b, long c, long d) {
    if (!ok && g_bad++ < 8) std::fprintf(stderr, "row_bounds: %s (%ld %ld %ld %ld)\n", what, a, b, c, d);
}

extern "C" int off32_ok_c(uint64_t bytes) { return off32_ok(bytes); }
extern "C" int row_lead_bound_c(int R, int n) { return row_lead_bound(R, n); }

extern "C" long check_row_dispatch(int gateup, int w4, int nb, int O, int T, int lead_bound, const int *mt_exp,
                                   const int *mt_row0, const int *mt_rend, const int *mt_first, int R,
                                   const int *row_act, int rows_x, int x_stride, int n_desc) {
    g_bad = 0;
    const int NS = slab_count(gateup != 0, O), Op = (O + 63) / 64 * 64, ntile = Op / TILE_O;
    const long w_bytes = (long)Op * nb * (w4 ? 16 : 32), x_bytes = (long)rows_x * x_stride;
    const int nc = (nb + ROW_CB - 1) / ROW_CB;
    std::vector<int> seen((size_t)NS * (T > 0 ? T : 1), 0);
    std::vector<int> lead;
    for (int t = 0; t < T; ++t)
        if (row_leads(t, mt_first[t])) lead.push_back(t);
    const int G = (int)lead.size(), grid = row_grid(lead_bound);
    for (int by = 0; by < grid; ++by)
        for (int bx = 0; bx < NS; ++bx) {
            int slab, i;
            row_place(bx + NS * by, NS, &slab, &i);
            need(slab >= 0 && slab < NS && i >= 0 && i < grid, "place", bx, by, slab, i);
            if (i >= G) continue;
            const int tile = lead[(size_t)i];
            const int e = mt_exp[tile], r0 = mt_row0[tile];
            int rend = mt_rend[tile];
            if (rend > r0 + ROW_TILES * MT_ROWS) rend = r0 + ROW_TILES * MT_ROWS;
            const int nm = (rend - r0 + MT_ROWS - 1) / MT_ROWS;
            need(e >= 0 && e < n_desc, "descriptor", tile, e, n_desc, 0);
            need(r0 >= 0 && r0 < rend && rend <= R && nm <= ROW_TILES, "rows", tile, r0, rend, R);
            for (int m = 0; m < nm; ++m) seen[(size_t)(tile + m) * NS + slab]++;
            for (int wave = 0; wave < 4; ++wave)
                for (int lane = 0; lane < 64; ++lane) {
                    for (int i = 0; i < 2 && wave < nm; ++i) {
                        const int r = row_of(wave, i, lane), rr = r0 + r < rend ? r0 + r : rend - 1;
                        const int xr = row_act ? row_act[rr] : rr;
                        need(xr >= 0 && xr < rows_x, "activation row", tile, rr, xr, rows_x);
                        const int p = row_piece(r, lane & 3);
                        need(p >= 0 && p < 2 * ROW_CB, "piece", r, lane, p, 0);
                        for (int c = 0; c < nc; ++c) {
                            const bool one = c * ROW_CB + 1 >= nb;
                            const long col = (long)c * ROW_CB * BLK + row_col(p, one);
                            const uint32_t voff = x_off32(xr, x_stride) + row_col(p, one);   // as the kernel: 32 bits
                            const long at = (long)c * ROW_CB * BLK + (long)voff;
                            need(col + 16 <= (long)nb * BLK && at == (long)xr * x_stride + col && at + 16 <= x_bytes,
                                 "activation copy", tile, wave, lane, c);
                        }
                    }
                    for (int t = 0; t < (w4 ? 1 : 2); ++t) {
                        const long v = w4 ? (long)sa_voff_w4(gateup != 0, slab, wave, lane, ntile, nb)
                                          : (long)row_voff_w8(lane) + sa_tile8(gateup != 0, slab, wave, t, ntile, nb);
                        for (int b = 0; b < nb; ++b) {
                            const long at = v + (long)b * (w4 ? 512 : 1024);
                            need(at >= 0 && at + 16 <= w_bytes, "weight copy", tile, slab, wave * 64 + lane, b);
                        }
                    }
                }
        }
    for (int t = 0; t < T; ++t)
        for (int s = 0; s < NS; ++s) need(seen[(size_t)t * NS + s] == 1, "item coverage", t, s, seen[(size_t)t * NS + s], NS);
    // the stage's LDS: which (row, piece) each 16-byte slot holds, then every
    // operand read finds its own row's piece 2q + hh
    int held[128 * 4];
    for (int &h : held) h = -1;
    for (int wave = 0; wave < 4; ++wave)
        for (int i = 0; i < 2; ++i)
            for (int lane = 0; lane < 64; ++lane) {
                const int r = row_of(wave, i, lane), slot = (wave * 2 + i) * 64 + lane;
                need(slot == r * 4 + (lane & 3) && held[slot] == -1, "slot", wave, i, lane, slot);
                held[slot] = r * 4 + row_piece(r, lane & 3);
            }
    for (int m = 0; m < 4; ++m)
        for (int j = 0; j < 32; ++j)
            for (int q = 0; q < ROW_CB; ++q)
                for (int hh = 0; hh < 2; ++hh) {
                    const uint32_t at = (uint32_t)m * 2048u + row_rd(j, q, hh);
                    need(at % 16 == 0 && at < 128 * 64 && held[at / 16] == (32 * m + j) * 4 + 2 * q + hh, "operand", m, j, q, hh);
                }
    return g_bad;
}
