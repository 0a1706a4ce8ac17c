// Calls of 65 to some thousand rows on a matrix of one K segment: 32-token tiles in the part-split form.
//
// The resident kernel walks units behind one another and covers the round trips of one wave (descriptor, first weight batch, second
// row's batch) by the products of the three others of its SIMD.  Where a wave has one unit only, all waves wait for the same round
// trips at the same time, and with few rows few workgroups exist at all.  Here a wave requests its weights before the tile is staged, and
// a unit is spread over up to four waves, as far as the workgroups stay within one round of the chip.
//
// us per launch (graph replay), resident kernel -> this: gate_up of d_model 768 at 65 / 200 / 512 / 1000 rows 8.0 -> 5.5, 8.1 -> 5.6,
// 8.4 -> 6.4, 8.9 -> 7.2, of 1024 at 200 / 700 rows 9.0 -> 6.6, 9.5 -> 7.8, of 2048 at 100 / 300 rows 9.4 -> 8.1, 10.8 -> 10.1; `down` of d_model
// 768 at 200 / 512 rows 6.7 -> 5.1, 6.7 -> 5.8.  Requesting the batches of both rows of a wave with two (16 units) spilled and was slower
// than the resident kernel throughout (1536, 300 rows: 8.5 against 11.4).
#include "mortar_spmm_core.h"

namespace {

template <int CODE>
int launch(int kind, int uw, SpmmParams &p, hipStream_t st) {
    switch (kind * 100 + uw + (p.y_tiled ? 1000 : 0)) {
        case 1108: return mortar_launch_partsplit<32, 2, false, false, 2, 8, CODE, 0, true>(p, st);
        case 1116: return mortar_launch_partsplit<32, 2, false, false, 1, 16, CODE, 0, true>(p, st);
        case 2: return mortar_launch_partsplit<32, 1, false, false, 4, 2, CODE, 4>(p, st);
        case 4: return mortar_launch_partsplit<32, 1, false, false, 4, 4, CODE, 4>(p, st);
        case 8: return mortar_launch_partsplit<32, 1, false, false, 2, 8, CODE, 2>(p, st);
        case 302: return mortar_launch_partsplit<32, 1, false, true, 4, 2, CODE, 4>(p, st);
        case 304: return mortar_launch_partsplit<32, 1, false, true, 4, 4, CODE, 4>(p, st);
        case 308: return mortar_launch_partsplit<32, 1, false, true, 2, 8, CODE, 2>(p, st);
        case 104: return mortar_launch_partsplit<32, 2, false, false, 4, 4, CODE, 2>(p, st);
        case 108: return mortar_launch_partsplit<32, 2, false, false, 2, 8, CODE>(p, st);
        case 116: return mortar_launch_partsplit<32, 2, false, false, 1, 16, CODE>(p, st);
    }
    return -1;
}

}  // namespace

int mortar_mid_launch(int kind, int code, SpmmParams &p, hipStream_t st) {
    if (kind == 2 || p.nseg != 1 || tile_bytes(32, p.Cb) > LDS_BUDGET) return -1;
    const int64_t tiles = (p.M + 31) / 32;
    for (int uw : {2, 4, 8, 16}) {
        if (tiles * ((p.n_units + uw - 1) / uw) > 256) continue;
        if (kind == 1 && uw == 2) continue;
        // Two waves on one row add in another order than one.  Not where that shows: gated gate_up gives the bits of the token-list kernels,
        // and from 513 rows the products give those of the MLP in one call, whose `down` has no such form.  (The product with an input mask has the
        // forms too: it gives the bits of the plain one on masked input.)
        if (uw < (kind == 1 ? 8 : 16) && (p.M > MLP_SEPARATE_MAX_ROWS || p.gates)) continue;
        if (kind != 1 && uw == 16) return -1;      // one part per wave and sixteen units: no faster than the resident kernel's (1000 rows: 6.9 against 7.3)
        switch (code) {
            case CODE_4BIT | CODE_UNIFORM: return launch<CODE_4BIT | CODE_UNIFORM>(kind, uw, p, st);
            case CODE_4BIT: return launch<CODE_4BIT>(kind, uw, p, st);
            default: return launch<CODE_2BIT>(kind, uw, p, st);
        }
    }
    return -1;
}
