// packed.h -- the projections of a real field that determine the others (molecular symmetry order 2).
//
// The projections p(m, mup, mu2) of a real field satisfy p(m, -mup, 0) = (-1)^mup conj p(m, mup, 0), and
// p(m, 0, 0) is real.  The evaluation therefore keeps, per grid point, only
//   mu2 = 0, mup = 1 .. L;  mu2 = 1 .. L/2, mup = -L .. L   (for each, m = max(|mup|, 2 mu2) .. L), and
//   p(2 j, 0, 0) + i p(2 j + 1, 0, 0), j = 0 .. L/2:
// 70 of 88 complex numbers at mmax 5, 20 of 28 at 3, 2 of 4 at 1, which its transforms along the axes
// and its reads and writes of the field shrink by.  In q space the relation reads
// p(m, -mup, 0)(q) = (-1)^mup conj p(m, mup, 0)(-q); the q-space step handles q and -q together.
#pragma once

template <int L> struct Packed {
    static constexpr int H = L / 2, W = 2 * L + 1;
    static constexpr int mlo(int mup, int mu2) {
        const int a = mup < 0 ? -mup : mup;
        return a > 2 * mu2 ? a : 2 * mu2;
    }
    // first entry (m = mlo) of an item (mup, mu2), not of (0, 0)
    static constexpr int off(int mup, int mu2) {
        int o = 0;
        for (int k = 1; k <= L; k++) {
            if (mu2 == 0 && k == mup) return o;
            o += L + 1 - k;
        }
        for (int u = 1; u <= H; u++)
            for (int k = -L; k <= L; k++) {
                if (u == mu2 && k == mup) return o;
                o += L + 1 - mlo(k, u);
            }
        return o;
    }
    static constexpr int pair0 = off(L + 1, H + 1);   // the pairs of real projections
    static constexpr int np = pair0 + L / 2 + 1;
};
static_assert(Packed<0>::np == 1 && Packed<1>::np == 2 && Packed<2>::np == 10 && Packed<3>::np == 20 &&
              Packed<4>::np == 43 && Packed<5>::np == 70, "");
