// How the FP32 batch kernel (cq_batch.h) covers a batch, and what that costs.
#pragma once

#include "common.h"

#include <cstdio>
#include <cstdlib>

namespace nd {

struct BatchPick {
    int nb, ks;   // batch rows per workgroup, K parts
    double cost;  // of the pick, in issue slots of a SIMD over 64 positions
};

// Tile height (batch rows per workgroup) and K parts. A SIMD issues about one
// wave instruction per 4 clocks, so a wave's cost per position is its adds,
// its MFMAs and ~2 for the centroid lookups, times the waves of the SIMD on the
// fullest CU (384 tiles: two a CU; three parts of them as if they filled it left
// 48 x 2028 x 768 CQ2 g128 at 5 rows at 54 us, 35 counted so), a little more for
// two waves of 4-bit codes, which have twice the lookups, and 1.6 times for one
// wave (16.3, 17.4, 27.7 ns, see cq_batch.h). Fewer rows per tile repeat the
// lookups, more rows leave SIMDs idle; four parts divide a row's walk by four, in
// whole rounds, where tiles alone do not fill the chip. Over 1372 shapes of
// groups of 128 and 256 the picks take 5% less time than with the average of the
// chip's waves in place of the fullest CU's, at 128 and 384 tiles 14%.
// NEEDLE2_GPU_FP32_BATCH = "rows,parts" picks them, where the group has such a
// kernel.
inline BatchPick batch_pick(int kind, int group, int groups, int blocks, int batch) {
    auto parts_ok = [&](int ks) {
        return ks == 1 || (group >= 32 && groups * (group < 64 ? group : 64) >= 4 * 64 && groups >= 4);
    };
    auto rows_ok = [&](int nb) { return group >= 32 || (nb != 3 && nb != 6); };
    auto cost = [&](int nb, int ks) {
        const int walk = group < 64 ? (groups * group + 64 * ks - 1) / (64 * ks)
                                    : (groups + ks - 1) / ks * (group / 64);  // blocks of 64 positions per part
        const long tiles = static_cast<long>(blocks) * ((batch + nb - 1) / nb);
        const double per_simd = static_cast<double>(ks) * ((tiles + device_cus() - 1) / device_cus());
        const double turns = per_simd <= 1 ? 1.6 : per_simd <= 2 ? (kind == kNib ? 2.13 : 2.0) : per_simd;
        return turns * walk * (nb + (nb + 3) / 4 + 2.0) * (ks > 1 ? 1.05 : 1.0);
    };
    if (const char *mode = std::getenv("NEEDLE2_GPU_FP32_BATCH")) {
        int nb = 0, ks = 0;
        if (std::sscanf(mode, "%d,%d", &nb, &ks) == 2 && (ks == 1 || ks == 4) && parts_ok(ks) &&
            (nb == 2 || nb == 3 || nb == 4 || nb == 6 || nb == 8) && rows_ok(nb))
            return {nb, ks, cost(nb, ks)};
    }
    BatchPick best{2, 1, 0};
    for (int ks : {1, 4}) {
        if (!parts_ok(ks)) continue;
        for (int nb : {2, 3, 4, 6, 8}) {
            if (!rows_ok(nb)) continue;
            const double c = cost(nb, ks);
            if (best.cost == 0 || c < best.cost) best = {nb, ks, c};
        }
    }
    return best;
}

}  // namespace nd
