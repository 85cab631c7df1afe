// spk_prodlay.hpp -- layout of the RHS products between their z pass and the spectral
// epilogue (host and device; integers only).
#pragma once

namespace spk {

// The 2/3 mask zeroes every product mode with k_z or k_y beyond its threshold,
// whatever k_x is, so the forward transforms make only the columns the mask
// keeps: the z pass stores the first kc of NZ/2+1 modes of a row, the y pass
// transforms those columns and stores the rows with |k_y| index <= jc, moved
// together (mode j > jc sits in row j - nskip).  At 256^3 that is 85 of 129
// columns and 169 of 256 rows: the forward y pass reads 0.66 and writes 0.43 of
// the full spectrum and the x pass reads 0.43 of it (8 fields at 256^3 FP64:
// y pass 409 -> 254 us, x pass 447 -> 193 us).  Rows have a pitch of kp elements
// (88 there), a multiple of 128 bytes where a row is long enough (at the full row's
// 129 elements the y pass took 338 us); planes of one x are xs elements apart.
// Without a mask kc = kp = NZ/2+1 and every row is kept.
struct ProdLay {
    int kc, kp, jc, nskip;
    long long xs;
};
// row of mode j in the products after the forward y pass, -1 where it is masked
constexpr int prod_row(const ProdLay &l, int j) {
    return j <= l.jc ? j : (j > l.jc + l.nskip ? j - l.nskip : -1);
}
// Where column (j, k) of a tile reads its products at x = 0: a column without any reads
// the nearest one's in its row or the next row's first, mostly in lines that the tile
// reads anyway (they are multiplied by m = 0, and are NaN exactly when its own would be).
constexpr int prod_column(const ProdLay &l, int nzh, int j, int k) {
    const int own = prod_row(l, j), r = own >= 0 ? own : l.jc;
    if (k < l.kc) return r * l.kp + k;
    return 2 * k > nzh + l.kc - 1 && r < 2 * l.jc ? (r + 1) * l.kp : r * l.kp + l.kc - 1;
}

}  // namespace spk
