// Cell-order images of lattices read from stdin: per lattice "nx ny torus" and
// nx*ny pore values (0 / 1).  Prints per lattice: cells, RAW cells, LINKS cells,
// whether steps run in place, and the first rule of the in-place steps that does
// not hold ("-": all hold, or steps do not run in place).
//
// In place, slot j of cell c is the element L(c, j) of the nine planes: plane j
// of its source where it streams, plane opp(j) of c where the wall rule feeds it.
#include <cstdio>
#include <map>
#include <utility>

#include "mts_common.h"

using namespace mts;

static int wrap(int v, int n) { return v < 0 ? v + n : v >= n ? v - n : v; }

int main() {
    Physics ph;
    ph.Cl = 1e-9;
    compute_physics(ph);
    int nx, ny, torus;
    while (std::scanf("%d %d %d", &nx, &ny, &torus) == 3) {
        std::vector<int32_t> pore((size_t)nx * ny);
        for (auto& p : pore)
            if (std::scanf("%d", &p) != 1) return 2;
        std::vector<double> kn(pore.size()), lp(pore.size());
        for (size_t p = 0; p < pore.size(); p++) kn[p] = pore[p] ? 0.1 : 0.0, lp[p] = pore[p] ? 7.73 : 0.0;
        Geometry g;
        std::string err;
        if (int rc = build_single_grid(nx, ny, pore.data(), kn.data(), lp.data(), ph, torus != 0, g, err)) {
            std::printf("error %d %s\n", rc, err.c_str());
            continue;
        }
        CompactImage ci;
        build_compact(g, ci);
        int64_t nlinks = 0;
        const int64_t S = ci.cstride;
        const char* bad = "-";
        const bool inplace = compact_inplace(ci);
        auto source = [&](int64_t c, int j) -> int64_t {  // as the kernels find it (IN slots)
            const uint32_t cw = ci.cw[c], rw = ci.rw[c];
            if (cw & CW_COMPLEX) return ci.aux[(size_t)rw * AUXW + j - 1];
            const int64_t ru = c + (int16_t)(rw & 0xffffu), rd = c - (int16_t)(rw >> 16);
            const int64_t src[9] = {c, c - 1, rd, c + 1, ru, rd - 1, rd + ((cw >> 23) & 1u), ru + ((cw >> 24) & 1u), ru - 1};
            return src[j];
        };
        auto in = [&](int64_t c, int j) { return j > 0 && ((ci.cw[c] >> (j - 1)) & 1u); };
        std::map<int64_t, std::pair<int64_t, int>> at;  // element -> its slot
        for (int64_t c = 0; c < ci.ncell; c++) {
            nlinks += (ci.cw[c] & CW_LINKS) == CW_LINKS && (ci.cw[c] & CW_RAW) != CW_RAW;
            if (!inplace) continue;
            const int x = ci.cellPos[c] % nx, y = ci.cellPos[c] / nx;
            for (int j = 0; j < 9; j++) {
                int64_t L = c;
                if (j && in(c, j)) {
                    const int64_t s = source(c, j);
                    if (s != ci.cidx[(size_t)wrap(y - EY[j], ny) * nx + wrap(x - EX[j], nx)]) bad = "source";
                    if (s < 0 || s >= ci.ncell) {
                        bad = "range";
                        continue;
                    }
                    // what c sends the other way arrives in the slot that reads this element
                    if (!in(s, OPP[j]) || source(s, OPP[j]) != c) bad = "partner";
                    L = j * S + s;
                } else if (j) {
                    if (!((ci.cw[c] >> (CW_WALL_SHIFT + OPP[j] - 1)) & 1u)) bad = "unfed";
                    L = OPP[j] * S + c;
                }
                if (!at.emplace(L, std::make_pair(c, j)).second) bad = "shared";
            }
        }
        std::printf("%lld %lld %lld %d %s\n", (long long)ci.ncell, (long long)ci.nraw, (long long)nlinks, (int)inplace, bad);
    }
}
