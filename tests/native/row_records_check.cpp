// CPU check of the row records (mf-lbm_amd/csrc/layout.h), built by tests/test_row_records.py: for every fluid node of
// a wall array and every direction, the neighbour's compact index derived from the row records equals the dense map's
// wherever the node has no link slot, and the phi view of the records (fluid and not an image) equals the set of
// interior fluid nodes at every padded position a stencil reaches.
// Input: int32 nx, ny, nz, open_z, jper, kper, fold_y, fold_z, tile and (nx + 4)(ny + 4)(nz + 4) int8 walls, halo 2.
#include <cstdio>
#include <vector>

#include "layout.h"

using namespace mflbm_dev;

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    FILE* fh = std::fopen(argv[1], "rb");
    int h[9];
    if (!fh || std::fread(h, 4, 9, fh) != 9) return 2;
    std::vector<int8_t> w2((size_t)(h[0] + 4) * (h[1] + 4) * (h[2] + 4));
    if (std::fread(w2.data(), 1, w2.size(), fh) != w2.size()) return 2;
    std::fclose(fh);
    const Layout L = make_layout(h[0], h[1], h[2]);
    std::vector<int8_t> wp(L.total, 1);
    pack_host(L, 2, w2.data(), wp.data());
    CompactSet cs;
    Fold F;
    F.y = h[6] != 0;
    F.z = h[7] != 0;
    build_compact(L, TileOrder{h[8], L}, wp, h[3] != 0, h[5] != 0, h[4] != 0, {}, cs, F);
    std::vector<RowRec> rows;
    build_rows(L, cs, rows);
    if ((long)rows.size() * 16 != L.total) return 1;
    long links = 0;
    for (int m = 0; m < cs.nfl; ++m) {
        const int o = cs.cpos[m];
        for (int r = 1; r < 19; ++r) {
            const int want = cs.cidx[o + L.off(r)];
            if (want < 0) return std::printf("node %d direction %d: nothing stored\n", m, r), 1;
            if (want >= cs.nfl) {   // a link slot; the records are not asked
                ++links;
                continue;
            }
            const int ex = lat::EX[r];
            const RowRec R = rows.at((size_t)((o >> 4) + lat::EY[r] * (L.px >> 4) + lat::EZ[r] * (L.pxy >> 4)));
            const unsigned got = row_rank(R, o) + (ex < 0 ? ~0u : ex > 0 ? row_fluid(R, o, 0) : 0u);
            if (got != (unsigned)want || !row_fluid(R, o, ex)) return std::printf("node %d direction %d: %u, want %d\n", m, r, got, want), 1;
        }
    }
    std::vector<int> pm(L.total, -1);
    for (int m = 0; m < cs.nfl; ++m) pm[cs.cpos[m]] = m;
    for (int k = -2; k <= L.nz + 3; ++k)
        for (int j = -2; j <= L.ny + 3; ++j)
            for (int i = -2; i <= L.nx + 3; ++i)
                for (int ex = -1; ex <= 1; ++ex) {
                    const int o = L.at(i, j, k);
                    const RowRec R = rows.at((size_t)(o >> 4));
                    const bool fl = !(R.bits & ROW_IMAGE) && row_fluid(R, o, ex);
                    if (fl != (pm[o + ex] >= 0)) return std::printf("phi view at (%d, %d, %d) %+d\n", i, j, k, ex), 1;
                    const unsigned at = row_rank(R, o) + (ex < 0 ? ~0u : ex > 0 ? row_fluid(R, o, 0) : 0u);
                    if (fl && at != (unsigned)pm[o + ex]) return std::printf("phi index at (%d, %d, %d) %+d\n", i, j, k, ex), 1;
                }
    std::printf("ok %d %ld\n", cs.nfl, links);
    return 0;
}
