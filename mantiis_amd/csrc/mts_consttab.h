// Tables per boundary type that the kernels keep in constant memory, formed at
// compile time from the embedded tables: they are the same for every handle, so
// nothing writes them at run time and handles may be made on several threads.
// Row MTS_NTYPES is the typeless wall link of a buffer cell (full bounce-back:
// target = opposite); types past the tables (TYPE_NONE) have no wall link.
#pragma once
#include "mts_common.h"
#include "mts_tables.inc"

namespace mts {

// 0-based specular target of link ic (utils.hpp:749-767; 0: none)
constexpr int icsr_target(int t, int ic) {
    return t >= MTS_NTYPES ? OPP[ic] : MTS_ICSR[t][ic] < 0 ? 0 : MTS_ICSR[t][ic];
}

struct IcsrTable {
    signed char v[MTS_NTYPES + 1][9];
    constexpr const signed char* operator[](int t) const { return v[t]; }
};
constexpr IcsrTable icsr_table() {
    IcsrTable r{};
    for (int t = 0; t <= MTS_NTYPES; t++)
        for (int ic = 0; ic < 9; ic++) r.v[t][ic] = (signed char)icsr_target(t, ic);
    return r;
}

struct TypeWords {
    uint32_t v[64];
    constexpr uint32_t operator[](uint32_t t) const { return v[t]; }
};
// the targets of ic = 1..8 in bits 4(ic-1)..4ic-1
constexpr TypeWords icsr_words() {
    TypeWords r{};
    for (int t = 0; t < 64; t++)
        for (int ic = 1; ic < 9; ic++) r.v[t] |= (uint32_t)icsr_target(t, ic) << (4 * (ic - 1));
    return r;
}
// slot j (bits 4(j-1)..4j-1) <- the link ic that is not streamed for the type
// and whose specular direction is j (the first such link when two share a slot)
constexpr TypeWords spec_words() {
    TypeWords r{};
    for (int t = 0; t <= MTS_NTYPES; t++)
        for (int ic = 8; ic >= 1; ic--) {
            const int sr = icsr_target(t, ic);
            if ((t < MTS_NTYPES && MTS_IFSTREAM[t][ic]) || sr <= 0) continue;
            r.v[t] = (r.v[t] & ~(15u << (4 * (sr - 1)))) | ((uint32_t)ic << (4 * (sr - 1)));
        }
    return r;
}
struct NormTable {
    double v[MTS_NTYPES][2];
    constexpr const double* operator[](int t) const { return v[t]; }
};
constexpr NormTable norm_table() {
    NormTable r{};
    for (int t = 0; t < MTS_NTYPES; t++)
        for (int k = 0; k < 2; k++) r.v[t][k] = MTS_XYNORM[t][k];
    return r;
}
// MDBB (coreLB.hpp:936-967): the directions j = 1..8 with e_j . n > 0 (bits
// 0..7) and with e_j . n < 0 (bits 8..15) for the wall normal n of the type
// (xy_norm.txt); 0 for types without a normal.
constexpr TypeWords mdbb_words() {
    TypeWords r{};
    for (int t = 0; t < MTS_NTYPES; t++)
        for (int j = 1; j < 9; j++) {
            const double cn = EY[j] * MTS_XYNORM[t][1] + EX[j] * MTS_XYNORM[t][0];
            if (cn > 0) r.v[t] |= 1u << (j - 1);
            else if (cn < 0) r.v[t] |= 1u << (8 + j - 1);
        }
    return r;
}

}  // namespace mts
