// Wave shapes of the split-operand attention kernels and the LDS each takes: one
// table for the kernels that hold the shapes (attn_fwd.hip, attn_bwd.hip) and the
// launcher that picks among them (zt_attn.cpp), so that a shape the launcher asks
// for is one its kernel has.
#pragma once
#include <initializer_list>

// Split tiles in LDS: row-major rows of dp bf16 values, one plane of `rows` rows
// per part.  The row stride is 2 dp + 32 bytes, 8 banks beyond a multiple
// of 16 (dp a multiple of 32): eight rows then cover the 64 banks, both for an
// operand read along the row (a lane per row, 16 bytes) and for a transposed
// read (four rows x 32 bytes per 16 lanes).
constexpr int split_stride(int dp) { return 2 * dp + 32; }
constexpr int split_bytes(int dp, int rows) { return 3 * rows * split_stride(dp); }

// ---- Forward: nw waves, nq 16-row blocks per wave, ks key parts ----------------
//
// A kernel per role, width and shape, each with the LDS and the registers that its
// shape needs: one kernel for all of a width's shapes takes the most of any, and at
// d = 32 that left one workgroup on a CU (147 KB, 154 registers) where one row block and
// two key parts (74 KB, 107 registers) let two share it.  8 x 1070 rows of 8 heads over 8
// at d = 32: two row blocks, all in one kernel, 97 us; one row block in its own 61;
// the f32 kernels 67.  The symbol is zt_<role>_d<dp>_k32_<nw><nq><ks>.  Roles: several
// heads of a kv group per workgroup (zt_fwd8p_*, zt_fwd8ps_*); one (zt_fwdp_*, also
// four waves, where forced); one on a small grid (zt_fwdpk_*).  The first of a list
// stands in for a forced shape that the list does not have.
#define ZT_FWD_HEADS_32(X) X(8, 2, 1) X(8, 1, 2) X(8, 1, 4)
#define ZT_FWD_HEADS_64(X) X(8, 2, 1) X(8, 2, 2) X(8, 1, 2)
#define ZT_FWD_HEADS_96(X) X(8, 2, 1) X(8, 1, 2)
#define ZT_FWD_HEADS_128(X) X(8, 2, 1) X(8, 1, 2)
#define ZT_FWD_HEADS_192(X) X(8, 2, 1) X(8, 1, 1)
#define ZT_FWD_HEADS_256(X) X(8, 2, 1) X(8, 1, 1)
#define ZT_FWD_ONE_32(X) X(8, 1, 2) X(4, 2, 1)
#define ZT_FWD_ONE_64(X) X(8, 2, 1) X(8, 2, 2) X(8, 1, 2) X(4, 2, 1)
#define ZT_FWD_ONE_96(X) X(8, 2, 1) X(8, 1, 2) X(4, 2, 1)
#define ZT_FWD_ONE_128(X) X(8, 2, 1) X(8, 1, 2) X(4, 2, 1)
#define ZT_FWD_ONE_192(X) X(8, 2, 1) X(8, 1, 1) X(4, 2, 1)
#define ZT_FWD_ONE_256(X) X(8, 2, 1) X(8, 1, 1) X(4, 2, 1)
#define ZT_FWD_SMALL_32(X) X(8, 1, 2) X(8, 1, 4)
#define ZT_FWD_SMALL_64(X) X(8, 1, 2) X(8, 1, 4)
#define ZT_FWD_SMALL_96(X) X(8, 1, 2)
#define ZT_FWD_SMALL_128(X) X(8, 1, 2)

struct FwdWaves {
    int nw, nq, ks;
};
struct FwdWavesList {
    FwdWaves s[4];  // nw 0: none
};
enum class FwdRole { Heads, One, Small };
constexpr int fwd_ds(int dp) { return dp > 128 ? 2 : 1; }  // column halves

#define ZT_FWD_ENTRY(NW, NQ, KS) {NW, NQ, KS},
constexpr FwdWavesList fwd_waves(FwdRole role, int dp) {
    switch (role) {
    case FwdRole::Heads:
        return dp == 32    ? FwdWavesList{{ZT_FWD_HEADS_32(ZT_FWD_ENTRY)}}
               : dp == 64  ? FwdWavesList{{ZT_FWD_HEADS_64(ZT_FWD_ENTRY)}}
               : dp == 96  ? FwdWavesList{{ZT_FWD_HEADS_96(ZT_FWD_ENTRY)}}
               : dp == 128 ? FwdWavesList{{ZT_FWD_HEADS_128(ZT_FWD_ENTRY)}}
               : dp == 192 ? FwdWavesList{{ZT_FWD_HEADS_192(ZT_FWD_ENTRY)}}
                           : FwdWavesList{{ZT_FWD_HEADS_256(ZT_FWD_ENTRY)}};
    case FwdRole::One:
        return dp == 32    ? FwdWavesList{{ZT_FWD_ONE_32(ZT_FWD_ENTRY)}}
               : dp == 64  ? FwdWavesList{{ZT_FWD_ONE_64(ZT_FWD_ENTRY)}}
               : dp == 96  ? FwdWavesList{{ZT_FWD_ONE_96(ZT_FWD_ENTRY)}}
               : dp == 128 ? FwdWavesList{{ZT_FWD_ONE_128(ZT_FWD_ENTRY)}}
               : dp == 192 ? FwdWavesList{{ZT_FWD_ONE_192(ZT_FWD_ENTRY)}}
                           : FwdWavesList{{ZT_FWD_ONE_256(ZT_FWD_ENTRY)}};
    default:
        return dp == 32   ? FwdWavesList{{ZT_FWD_SMALL_32(ZT_FWD_ENTRY)}}
               : dp == 64 ? FwdWavesList{{ZT_FWD_SMALL_64(ZT_FWD_ENTRY)}}
               : dp == 96 ? FwdWavesList{{ZT_FWD_SMALL_96(ZT_FWD_ENTRY)}}
                          : FwdWavesList{{ZT_FWD_SMALL_128(ZT_FWD_ENTRY)}};
    }
}
// Alternating wave halves (fwd_split_tile): two buffers each for K and V.
constexpr bool fwd_alt(int dp, FwdWaves s) {
    return s.nw == 8 && fwd_ds(dp) == 1 && 4 * split_bytes(dp, 32 * s.ks) + 16 <= 160 * 1024;
}
constexpr int fwd_tiles_lds(int dp, FwdWaves s) { return (fwd_alt(dp, s) ? 4 : 2) * split_bytes(dp, 32 * s.ks); }
// The tiles, the partial scores that the column halves exchange, and the big-value flags.
constexpr int fwd_lds(int dp, FwdWaves s) { return fwd_tiles_lds(dp, s) + (fwd_ds(dp) > 1 ? s.nw * 2 * s.nq * 1024 : 0) + 16; }
// The most any of a width's kernels takes (the small-grid role is built for dp <= 128).
constexpr int fwd_lds_most(int dp) {
    int most = 0;
    for (FwdRole r : {FwdRole::Heads, FwdRole::One, FwdRole::Small})
        for (int i = 0; i < 4 && !(r == FwdRole::Small && dp > 128); ++i) {
            const FwdWaves s = fwd_waves(r, dp).s[i];
            if (s.nw && fwd_lds(dp, s) > most) most = fwd_lds(dp, s);
        }
    return most;
}

// ---- dk/dv from the forward's scores: `parts` parts of `kblocks` 16-key blocks ---
//
// (No four blocks at d = 32: dkdv_split_shape in zt_attn.cpp.)
// Kernels as the forward's, with _<parts><kblocks> behind the name.
#define ZT_DKDV_32(X) X(4, 2) X(8, 1)
#define ZT_DKDV_64(X) X(2, 4) X(4, 2) X(4, 1)
#define ZT_DKDV_96(X) X(2, 4) X(2, 2)
#define ZT_DKDV_128(X) X(2, 4) X(2, 2)
struct BwdWaves {
    int parts, kblocks;
};
struct BwdWavesList {
    BwdWaves s[3];  // parts 0: none
};
#define ZT_DKDV_ENTRY(PARTS, KBLOCKS) {PARTS, KBLOCKS},
constexpr BwdWavesList dkdv_waves(int dp) {
    return dp == 32   ? BwdWavesList{{ZT_DKDV_32(ZT_DKDV_ENTRY)}}
           : dp == 64 ? BwdWavesList{{ZT_DKDV_64(ZT_DKDV_ENTRY)}}
           : dp == 96 ? BwdWavesList{{ZT_DKDV_96(ZT_DKDV_ENTRY)}}
                      : BwdWavesList{{ZT_DKDV_128(ZT_DKDV_ENTRY)}};
}
// A dO and a Q tile of 32 rows, their rows' statistics and the big-value flags, per part.
constexpr int dkdv_lds(int dp, BwdWaves s) { return s.parts * (2 * split_bytes(dp, 32) + 64 * 4 + 8); }
constexpr int dkdv_lds_most(int dp) {
    int most = 0;
    for (const BwdWaves s : dkdv_waves(dp).s)
        if (s.parts && dkdv_lds(dp, s) > most) most = dkdv_lds(dp, s);
    return most;
}
