// Wave shapes of the split-operand attention kernels and the LDS each takes: one
// table for the kernels that hold the shapes (attn_fwd.hip, attn_bwd.hip) and the
// launcher that picks among them (zt_attn.cpp), so that a shape the launcher asks
// for is one its kernel has.
#pragma once

// Split tiles in LDS: row-major rows of dp bf16 values, one plane of `rows` rows
// per part.  The row stride is 2 dp + 32 bytes, 8 banks beyond a multiple
// of 16 (dp a multiple of 32): eight rows then cover the 64 banks, both for an
// operand read along the row (a lane per row, 16 bytes) and for a transposed
// read (four rows x 32 bytes per 16 lanes).
constexpr int split_stride(int dp) { return 2 * dp + 32; }
constexpr int split_bytes(int dp, int rows) { return 3 * rows * split_stride(dp); }

// ---- Forward: nw waves, nq 16-row blocks per wave, ks key parts ----------------
//
// Roles: several heads of a kv group per workgroup (zt_fwd8p_*, zt_fwd8ps_*); one
// (zt_fwdp_*, also four waves, where forced); one on a small grid (zt_fwdpk_*).
//
// A kernel holds all shapes of its role and width, except at d = 32, where each
// shape is a kernel of its own, _<nw><nq><ks> behind its name.  A common kernel takes
// the LDS and the registers of its largest shape: at d = 32 147 KB and 154, one workgroup
// on a CU, where one row block and two key parts alone (74 KB, 107) let two share it.  8 x
// 1070 rows of 8 heads over 8: two row blocks in the common kernel 97 us, one in its
// own 61; the f32 kernels 67.  Wider heads fill a CU with either, and the compiler
// schedules a shape alone no better: 333 rows at 2007 of 32 over 8 heads at d = 128 123 in
// the common kernel, 128 in its own.  The first of a list stands in for a forced shape
// that the list does not have.
struct FwdWaves {
    int nw, nq, ks;
};
struct FwdWavesList {
    int n;
    FwdWaves s[4];
};
enum class FwdRole { Heads, One, Small };
constexpr int fwd_ds(int dp) { return dp > 128 ? 2 : 1; }  // column halves
constexpr bool fwd_shape_kernels(int dp) { return dp == 32; }

#define ZT_FWD_HEADS_32(X) X(8, 2, 1) X(8, 1, 2) X(8, 1, 4)
#define ZT_FWD_ONE_32(X) X(8, 1, 2) X(4, 2, 1)
#define ZT_FWD_SMALL_32(X) X(8, 1, 2) X(8, 1, 4)
#define ZT_FWD_ENTRY(NW, NQ, KS) {NW, NQ, KS},
constexpr FwdWavesList fwd_waves(FwdRole role, int dp) {
    if (dp == 32)
        return role == FwdRole::Small ? FwdWavesList{2, {ZT_FWD_SMALL_32(ZT_FWD_ENTRY)}}
               : role == FwdRole::One ? FwdWavesList{2, {ZT_FWD_ONE_32(ZT_FWD_ENTRY)}}
                                      : FwdWavesList{3, {ZT_FWD_HEADS_32(ZT_FWD_ENTRY)}};
    if (role == FwdRole::Small) return dp <= 64 ? FwdWavesList{2, {{8, 1, 2}, {8, 1, 4}}} : FwdWavesList{1, {{8, 1, 2}}};
    if (role == FwdRole::One)
        return dp <= 64    ? FwdWavesList{4, {{8, 2, 1}, {8, 2, 2}, {8, 1, 2}, {4, 2, 1}}}
               : dp <= 128 ? FwdWavesList{3, {{8, 2, 1}, {8, 1, 2}, {4, 2, 1}}}
                           : FwdWavesList{3, {{8, 2, 1}, {8, 1, 1}, {4, 2, 1}}};
    return dp <= 64    ? FwdWavesList{3, {{8, 2, 1}, {8, 2, 2}, {8, 1, 2}}}
           : dp <= 128 ? FwdWavesList{2, {{8, 2, 1}, {8, 1, 2}}}
                       : FwdWavesList{2, {{8, 2, 1}, {8, 1, 1}}};
}
// Alternating wave halves (fwd_split_tile): two buffers each for K and V.
constexpr bool fwd_alt(int dp, FwdWaves s) {
    return s.nw == 8 && fwd_ds(dp) == 1 && 4 * split_bytes(dp, 32 * s.ks) + 16 <= 160 * 1024;
}
constexpr int fwd_tiles_lds(int dp, FwdWaves s) { return (fwd_alt(dp, s) ? 4 : 2) * split_bytes(dp, 32 * s.ks); }
// The tiles, the partial scores that the column halves exchange, and the big-value flags.
constexpr int fwd_lds(int dp, FwdWaves s) { return fwd_tiles_lds(dp, s) + (fwd_ds(dp) > 1 ? s.nw * 2 * s.nq * 1024 : 0) + 16; }
// The most any shape of a role takes, and any of a width (Small is built for dp <= 128).
constexpr int fwd_lds(FwdRole role, int dp) {
    int most = 0;
    for (int i = 0; i < fwd_waves(role, dp).n; ++i) {
        const int x = fwd_lds(dp, fwd_waves(role, dp).s[i]);
        most = x > most ? x : most;
    }
    return most;
}
constexpr int fwd_lds(int dp) {
    int most = fwd_lds(FwdRole::Heads, dp);
    if (fwd_lds(FwdRole::One, dp) > most) most = fwd_lds(FwdRole::One, dp);
    if (dp <= 128 && fwd_lds(FwdRole::Small, dp) > most) most = fwd_lds(FwdRole::Small, dp);
    return most;
}

// ---- dk/dv from the forward's scores: `parts` parts of `kblocks` 16-key blocks ---
//
// A kernel per shape, _<parts><kblocks> behind its name.
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
