// Decode launches (one matrix, up to 64 rows) that spread few units over the whole chip: the part-split kernel with its row parts cut
// into chunks, fewer units per workgroup and more waves per unit.
//
// A workgroup of four units leaves most CUs idle where a product has few: at one row `down` of d_model 2048 was 32 workgroups, of
// d_model 768 twelve.  The units per workgroup come down to what one round of the chip (256 workgroups) holds, and every row part is
// cut into runs of whole octets on waves of their own.
#include "mortar_spmm_core.h"

namespace {

// Waves per part for a unit of `nparts` parts of about `octets` octets each, UW units per workgroup: 4 or 2 where built, at most one
// wave per octet (a part of one octet is cut in two all the same: the waves then share the staging); 0: none.
int chunk_waves(int nparts, int octets, int uw) {
    for (int cs : {4, 2}) {
        const int pw = nparts * cs;
        if (cs > 2 && cs > octets) continue;
        if (uw == 1 ? pw == 8 || pw == 12 : uw == 2 ? pw == 4 || pw == 6 || pw == 8 : pw == 4) return cs;
    }
    return 0;
}

template <int MT, int NACC, int CODE>
int launch(int pw, int cs, int uw, SpmmParams &p, hipStream_t st) {
    switch (uw * 1000 + pw * 10 + cs) {
        case 1082: return mortar_launch_partsplit<MT, NACC, false, false, 8, 1, CODE, 2>(p, st);
        case 1084: return mortar_launch_partsplit<MT, NACC, false, false, 8, 1, CODE, 4>(p, st);
        case 1122: return mortar_launch_partsplit<MT, NACC, false, false, 12, 1, CODE, 2>(p, st);
        case 1124: return mortar_launch_partsplit<MT, NACC, false, false, 12, 1, CODE, 4>(p, st);
        case 2042: return mortar_launch_partsplit<MT, NACC, false, false, 4, 2, CODE, 2>(p, st);
        case 2044: return mortar_launch_partsplit<MT, NACC, false, false, 4, 2, CODE, 4>(p, st);
        case 2062: return mortar_launch_partsplit<MT, NACC, false, false, 6, 2, CODE, 2>(p, st);
        case 2082: return mortar_launch_partsplit<MT, NACC, false, false, 8, 2, CODE, 2>(p, st);
        case 2084: return mortar_launch_partsplit<MT, NACC, false, false, 8, 2, CODE, 4>(p, st);
        case 4042: return mortar_launch_partsplit<MT, NACC, false, false, 4, 4, CODE, 2>(p, st);
        case 4044: return mortar_launch_partsplit<MT, NACC, false, false, 4, 4, CODE, 4>(p, st);
    }
    return -1;
}

// gate_up over two K segments with the norm of wide rows in it
template <int MT, int CODE>
int launch_norm_wide(int cs, int uw, SpmmParams &p, hipStream_t st) {
    if (cs != 2 || p.nseg != 2) return -1;
    if (uw == 1) return mortar_launch_partsplit<MT, 2, false, false, 8, 1, CODE, 2, false, NORM_WIDE_MAX_CB>(p, st);
    if (uw == 2) return mortar_launch_partsplit<MT, 2, false, false, 8, 2, CODE, 2, false, NORM_WIDE_MAX_CB>(p, st);
    return -1;
}

template <int MT, int CODE>
int launch_kind(int kind, int cs, int uw, SpmmParams &p, hipStream_t st) {
    if (p.norm == NORM_WIDE) return launch_norm_wide<MT, CODE>(cs, uw, p, st);
    return kind == 0 ? launch<MT, 1, CODE>(p.nseg * cs, cs, uw, p, st) : launch<MT, 2, CODE>(2 * p.nseg * cs, cs, uw, p, st);
}

}  // namespace

int mortar_chunk_launch(int kind, int mt, SpmmParams &p, hipStream_t st) {
    // (gated gate_up stays with the form that adds in the order of the token-list kernels: the two give the same bits)
    if ((kind != 0 && kind != 1) || (kind == 1 && p.gates)) return -1;
    const int nacc = kind + 1, nparts = p.nseg * nacc;
    const int64_t tiles = (p.M + mt - 1) / mt;
    for (int uw : {1, 2, 4}) {
        // gate_up in workgroups of four units has two waves per unit to begin with.  Four share the normalising of the rows, which is
        // longer the wider they are, and cost an exchange more.  Two against four, us, 13 to 64 rows wherever this form is
        // taken: with the norm 48 block-columns 4.7 against 4.9, 64 4.8 against 4.9, 72 to 88 5.2 to 5.5 either way, 96 5.46 against 5.43,
        // 104 and 112 equal, 128 5.8 against 5.7; without it two are faster at every width (48 3.6 against 3.9, 88 4.1 against
        // 4.4, 96 4.1 against 4.5, 128 4.4 against 4.6).  So the line lies where the norm's side turns: by the width alone,
        // not by the norm, so that the fused norm gives the bits of the separate one.
        if (uw == 4 && kind == 1 && p.Cb < 96) continue;
        if (tiles * ((p.n_units + uw - 1) / uw) > 256) continue;
        const int cs = chunk_waves(nparts, p.avg_octets, uw);
        if (cs == 0 || tile_bytes(mt, p.Cb) + cs * nparts * uw * nacc * 1024 > 160 * 1024) continue;
        if (p.uscale != 0.f) return mt == 4 ? launch_kind<4, CODE_UNIFORM>(kind, cs, uw, p, st) : launch_kind<8, CODE_UNIFORM>(kind, cs, uw, p, st);
        return mt == 4 ? launch_kind<4, CODE_2BIT>(kind, cs, uw, p, st) : launch_kind<8, CODE_2BIT>(kind, cs, uw, p, st);
    }
    return -1;
}
