// spk_halo.hpp -- where the 16-byte chunks of a closure brick's halo lie in a
// periodic n^3 field of nq chunks per point (host and device; integers only).
#pragma once

namespace spk {

constexpr int HX = 6, HY = 6, HZ = 34;  // brick 4 x 4 x 32 with a one-point halo

// A chunk's place relative to the brick's first point never changes: its offset in
// chunks, above six bits that name the halo faces the chunk is on (31 bits up to
// n = 1024 with 4 chunks a point).
constexpr int halo_place(int chunk, int n, int nq) {
    const int q = chunk % nq, hp = chunk / nq;
    const int hz = hp % HZ, hy = (hp / HZ) % HY, hx = hp / (HZ * HY);
    const int off = (((hx - 1) * n + hy - 1) * n + hz - 1) * nq + q;
    return off * 64 + (hx == 0) + 2 * (hx == HX - 1) + 4 * (hy == 0) + 8 * (hy == HY - 1) + 16 * (hz == 0) +
           32 * (hz == HZ - 1);
}

// The chunks at[] of the brick with first point (x0, y0, z0), which at a face of the
// grid wrap there, as indices into the field.  Counted modulo 2^32: a field of n = 1024
// and 4 chunks a point has 2^32 of them, so every index is exact, while the wraps
// alone, n^3 nq, exceed 31 bits from n = 832 on.
template <int N>
constexpr void halo_chunks(const int (&at)[N], unsigned (&o)[N], int n, int nq, int x0, int y0, int z0) {
    const unsigned z1 = (unsigned)(n * nq), y1 = z1 * (unsigned)n, x1 = y1 * (unsigned)n;  // one period along z, y, x
    const unsigned first = ((unsigned)(x0 * n + y0) * (unsigned)n + (unsigned)z0) * (unsigned)nq;
    for (int k = 0; k < N; k++) o[k] = first + (unsigned)(at[k] >> 6);
    auto wrap = [&](bool face, int bit, unsigned by) {
        if (face)
            for (int k = 0; k < N; k++) o[k] += (at[k] & bit) ? by : 0u;
    };
    wrap(x0 == 0, 1, x1);
    wrap(x0 + 4 == n, 2, 0u - x1);
    wrap(y0 == 0, 4, y1);
    wrap(y0 + 4 == n, 8, 0u - y1);
    wrap(z0 == 0, 16, z1);
    wrap(z0 + 32 == n, 32, 0u - z1);
}

}  // namespace spk
