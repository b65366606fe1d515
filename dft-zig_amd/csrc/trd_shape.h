// Launch shape of the tridiagonalisation (heev.hip): host arithmetic only.
#pragma once

namespace dzhip {

constexpr int kTrdWaves = 4;  // wavefronts per workgroup of the tridiagonalisation, one per SIMD

// The instances (NQ, CW): matrices of up to 64 NQ rows, CW columns per wavefront.  Two and four columns
// are for devices of fewer CUs (a partition of 128, 64 or 32), from the sizes on whose grids of one and
// two columns do not fit those: there from 129 and 257 rows.
#define DZ_TRD_INSTANCES(X)                                              \
    X(1, 1) X(2, 1) X(3, 1) X(4, 1) X(6, 1) X(8, 1) X(11, 1) X(13, 1) X(16, 1) \
    X(3, 2) X(4, 2) X(6, 2) X(8, 2) X(11, 2) X(13, 2) X(16, 2)           \
    X(6, 4) X(8, 4) X(11, 4)

struct TrdPick {
    int nq, cw, groups;  // nq = 0: no instance
};

// The instance for m rows on a device of `cus` CUs and its workgroups, all of which must be resident at
// once (one per CU): the fewest columns a wavefront that fit, at least `cols` per workgroup where an
// instance has as many.  A step's chain is latency and each wavefront's redundant vector work, which a
// second column only lengthens.
inline TrdPick trd_pick(int m, int cus, int cols) {
    for (int cw = 1; cw <= 4; cw *= 2) {
        const int groups = (m + kTrdWaves * cw - 1) / (kTrdWaves * cw);
        if (groups > cus || (cw < 4 && kTrdWaves * 2 * cw <= cols)) continue;
#define DZ_TRD_FITS(NQ, CW) \
    if (cw == CW && m <= 64 * NQ) return TrdPick{NQ, CW, groups};
        DZ_TRD_INSTANCES(DZ_TRD_FITS)
#undef DZ_TRD_FITS
    }
    return cols > 0 ? trd_pick(m, cus, cols / 2) : TrdPick{0, 0, 0};
}

}  // namespace dzhip
