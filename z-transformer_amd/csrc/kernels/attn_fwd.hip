// Fused causal grouped-query attention, forward, f32 (gfx950): on FP32 MFMA, and
// on split operands (split.h, the second half of the file) wherever rows are whole
// 16-byte chunks and the width allows.
//
// Computes what src/cuda/attn_kernels.cu:197-369 (fusedAttnForward) computes
// -- O = softmax(Q K^T / sqrt(d), causal) V with query row t at absolute
// position q_offset + t seeing keys s <= q_offset + t, s < n_keys -- but with
// a different schedule:
//   * a workgroup is NW = 4 or 8 waves; each wave owns 16 query rows of one
//     query head.  The waves are HW query heads of ONE kv group x (NW / HW) row blocks,
//     so each K/V tile staged in LDS is read from HBM/L2 once per kv group
//     instead of once per query (the reference re-reads the prefix per query);
//   * Q stays in registers for the whole key loop, pre-scaled by
//     log2(e)/sqrt(d) so the softmax runs on exp2;
//   * S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_16x16x4_f32, with P passed
//     register to register (layout notes in common.h);
//   * online softmax with a per-lane partial denominator that is reduced once
//     at the end; only the running max is exchanged across lanes per tile.
// The grid is 1-D, heaviest (latest) row tiles first, with the kv group as the
// fastest-varying index so that consecutive workgroups -- which the dispatcher
// spreads across the XCDs -- keep one kv group's K/V per XCD L2.
#include "common.h"
#include "args.h"
#include "split.h"


template <int DP, int BK, int NW, bool PF>
__device__ __forceinline__ void attn_fwd_tile(const FwdArgs &a, const int tile) {
    constexpr int LW = DP + 4;  // LDS row stride: +16 B spreads row starts over banks
    constexpr int DQ = DP / 4;  // d values per lane group
    constexpr int NT = DP / 16; // 16-wide column tiles of the output
    constexpr int NJ = BK / 16; // 16-key sub-blocks per LDS tile
    constexpr int NTH = 64 * NW;
    __shared__ float smem[2 * BK * LW];
    float *const Ks = smem, *const Vs = smem + BK * LW;

    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, grp = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // in a scalar register: wave-uniform branches stay scalar
    const int RB = NW / a.HW;  // 16-row blocks per head in this workgroup
    const int per_tile = a.n_head_blocks * a.B;
    const int rem = (int)blockIdx.x % per_tile;
    const int hb = rem % a.n_head_blocks, b = rem / a.n_head_blocks;
    const int group = a.H / a.Hkv;
    const int h = hb * a.HW + (w % a.HW);
    const int kvh = ZT_PLANT == 2 ? 0 : h / group;
    const int wg_row0 = tile * 16 * RB;
    const int row0 = wg_row0 + 16 * (w / a.HW);
    const bool vec4 = (a.dim & 3) == 0;
    const size_t qld = (size_t)a.H * a.dim, kld = (size_t)a.Hkv * a.dim;
    const float *qb = a.q + (size_t)b * a.T * qld + (size_t)h * a.dim;
    const float *kb = a.k + (size_t)b * a.kv_rows * kld + (size_t)kvh * a.dim;
    const float *vb = a.v + (size_t)b * a.kv_rows * kld + (size_t)kvh * a.dim;

    const int my_row = row0 + l16;
    float qr[DQ];
    load_row_seg<DQ>(qr, qb + (size_t)my_row * qld, grp * DQ, a.dim, vec4, my_row < a.T,
                     ZT_PLANT == 4 ? kLog2e : a.scale_log2e);

    f4 o[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) o[i] = zero4();
    float m = -INFINITY, lsum = 0.f;
    const int qpos = a.q_offset + my_row;
    const int kend_wg = min(a.n_keys, a.q_offset + min(a.T, wg_row0 + 16 * RB));
    const int kend_w = row0 < a.T ? min(a.n_keys, a.q_offset + min(a.T, row0 + 16)) : 0;

    // Register prefetch (PF): thread tid holds float4 chunks e = tid + n * NTH
    // of the next K/V tile (2 x BK x DP floats), loaded while the current tile
    // computes and written to LDS after the next barrier.  Every load is
    // unconditional and in bounds, so the pieces can be issued between the
    // score products: keys past n_keys load key n_keys - 1 (their scores are
    // masked, so P is 0 there) and columns past dim the row's last four floats
    // (met by Q's zero columns, or landing in output columns never stored); the
    // host picks this kernel only for dim % 4 == 0, whose rows are 16-byte aligned.
    constexpr int CPR = DP / 4;
    constexpr int NPF = PF ? 2 * BK * CPR / NTH : 1;
    static_assert(!PF || (2 * BK * CPR) % NTH == 0, "prefetch split");
    f4 pf[NPF];
    // A thread's byte offsets within a tile's rows (rows tid / CPR + j RPN,
    // its column), fixed for the kernel: a piece is one load from the tile's
    // base in scalar registers plus the offset clamped (one min) to key
    // n_keys - 1, with no per-piece address arithmetic (C3 training forward
    // 1.092 -> 1.066 ms, C5 0.563 -> 0.551 ms).
    constexpr int RPN = NTH / CPR;
    constexpr int NOFF = PF && (BK * CPR) % NTH == 0 && BK % RPN == 0 ? BK / RPN : 1;
    unsigned voff[NOFF];
    const unsigned coff = (unsigned)min((tid % CPR) * 4, a.dim - 4) * 4u;
#pragma unroll
    for (int j = 0; j < NOFF; ++j) voff[j] = (unsigned)((tid / CPR + j * RPN) * (int)kld) * 4u + coff;
    auto fetch_piece = [&](int n, int k0) {
        const int e = tid + n * NTH;
        // With whole arrays per piece, the piece's array follows from n alone
        // (tid < NTH): the base stays in scalar registers.
        const int arr = (NOFF > 1 ? n * NTH : e) / (BK * CPR);
        if constexpr (NOFF > 1) {
            // Key n_keys - 1, counted within the tile (no 32-bit overflow however many keys).
            const unsigned last = (unsigned)(min(a.n_keys - 1 - k0, BK - 1) * (int)kld) * 4u + coff;
            const unsigned off = min(voff[(n * RPN % BK) / RPN], last);
            pf[n] = *reinterpret_cast<const f4 *>(reinterpret_cast<const char *>((arr ? vb : kb) + (size_t)k0 * kld) + off);
        } else {
            const int r = min((e / CPR) % BK, a.n_keys - 1 - k0), c = min((e % CPR) * 4, a.dim - 4);
            pf[n] = *reinterpret_cast<const f4 *>((arr ? vb : kb) + (size_t)k0 * kld + (r * (int)kld + c));
        }
    };
    auto fetch = [&](int k0) {
#pragma unroll
        for (int n = 0; n < NPF; ++n) fetch_piece(n, k0);
    };
    if constexpr (PF) fetch(0);

    for (int ks0 = 0; ks0 < kend_wg; ks0 += BK) {
        __syncthreads();
        // The tile the prefetch loads meanwhile (the last one loads itself again, unused).
        const int kn = ks0 + BK < kend_wg ? ks0 + BK : ks0;
        const int k0 = ks0;
        if constexpr (PF) {
#pragma unroll
            for (int n = 0; n < NPF; ++n) {
                const int e = tid + n * NTH;
                const int arr = e / (BK * CPR), r = (e / CPR) % BK, c = (e % CPR) * 4;
                *reinterpret_cast<f4 *>((arr ? Vs : Ks) + r * LW + c) = pf[n];
            }
            __syncthreads();
        } else {
            const int nvalid = min(BK, a.n_keys - k0);
            stage_rows<DP, LW, NTH>(Ks, kb + (size_t)k0 * kld, kld, BK, nvalid, a.dim, vec4, tid);
            stage_rows<DP, LW, NTH>(Vs, vb + (size_t)k0 * kld, kld, BK, nvalid, a.dim, vec4, tid);
            __syncthreads();
        }
        if (k0 >= kend_w) {  // wave-uniform: nothing here is visible to this wave
            if constexpr (PF) fetch(kn);
            continue;
        }

        // Scores for every 16-key sub-block, the NJ accumulation chains
        // interleaved so consecutive MFMAs are independent.  A sub-block that is
        // wholly invisible to this wave is computed and then masked.
        f4 s[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) s[j] = zero4();
        const float *krow = Ks + l16 * LW + grp * DQ;
#pragma unroll
        for (int kk = 0; kk < DQ; kk += 4) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const f4 kx = *reinterpret_cast<const f4 *>(krow + 16 * j * LW + kk);
                s[j] = mfma16(kx.x, qr[kk + 0], s[j]);
                s[j] = mfma16(kx.y, qr[kk + 1], s[j]);
                s[j] = mfma16(kx.z, qr[kk + 2], s[j]);
                s[j] = mfma16(kx.w, qr[kk + 3], s[j]);
            }
            if constexpr (PF) {  // the prefetch pieces go out between the score products
                constexpr int NI = DQ / 4;
#pragma unroll
                for (int n = (kk / 4) * NPF / NI; n < (kk / 4 + 1) * NPF / NI; ++n) fetch_piece(n, kn);
            }
        }
        if (a.s_out) {
            // Element (t = row0 + l16, s = k0 + 16 j + 4 grp + r) goes to lane
            // (s & 15) + 16 ((t & 15) >> 2), element t & 3 of its tile: four
            // lanes write each 16-byte run.  (A quad transpose to one 16-byte
            // store per lane measured no faster.)  Nontemporal: the 1 GB of
            // tiles would otherwise displace the K/V rows the workgroups share
            // in L2 (C3 1.100 -> 1.092 ms, C5 0.576 -> 0.563 ms).
            // Row tile row0 / 16 keeps its tiles 0..row0 / 16 contiguous, so
            // sub-block j of this key tile is j tiles after its first.
            const int nt = (a.T + 15) >> 4;
            float *srow = a.s_out + (((size_t)b * a.H + h) * zt_tri_count(nt) + zt_tri_index(row0 >> 4, k0 >> 4)) * 256 +
                          (16 * (l16 >> 2)) * 4 + (l16 & 3);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if (k0 + 16 * j >= kend_w) continue;  // wave-uniform: above the diagonal
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    __builtin_nontemporal_store(ZT_PLANT == 5 ? s[j][r] / a.scale_log2e : s[j][r],
                                                srow + j * 256 + (4 * grp + r) * 4);
            }
        }
        if (k0 + BK - 1 > a.q_offset + row0 || k0 + BK > a.n_keys) {  // wave-uniform: a key past a row or past n_keys
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = k0 + 16 * j + 4 * grp + r;
                    if ((ZT_PLANT != 1 && key > qpos) || key >= a.n_keys) s[j][r] = -INFINITY;
                }
            }
        }
        float sv[4 * NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) sv[4 * j + r] = s[j][r];
        const float mt = max4grp(vmax_n(sv));
        // Lazy rescaling: a row's exponent base m moves only when the row meets
        // a tile maximum more than 8 (log2 units) above it, so between moves
        // every exp2 stays at most 2^8 and the running sum and O need no
        // rescaling (C3 training forward 1.114 -> 1.099 ms, C5 0.587 -> 0.577 ms;
        // the rescale's 32 multiplies per tile ran beside no MFMA).  The first tile always moves it (m
        // starts at -inf; key 0 is visible to every row, so mt is finite
        // there); the result is the eager rescaling's up to rounding.  Decided
        // per row (the four lanes of a row agree), not per wave: a row's
        // arithmetic then depends on no other row, and the branch is skipped
        // when no row of the wave moves.
        if (ZT_PLANT == 3 || mt > m + 8.f) {
            const float mnew = fmaxf(m, mt);
            const float corr = fast_exp2(m - mnew);
            m = mnew;
            lsum = ZT_PLANT == 3 ? lsum : lsum * corr;
#pragma unroll
            for (int i = 0; i < NT; ++i) o[i] *= ZT_PLANT == 3 ? 1.f : corr;
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[j][r] = fast_exp2(s[j][r] - m);
        float ps = s[0][0];  // = 0 + s[0][0]: the weights are >= +0
#pragma unroll
        for (int i = 1; i < 4 * NJ; ++i) ps += s[i / 4][i % 4];
        lsum += ps;

#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (k0 + 16 * j >= kend_w) continue;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                // A operand V^T in the row-owner layout: V[key 16 j + 4 grp + kk][l16 * NT + i].
                float vx[NT];
                lds_run<NT>(vx, Vs + (16 * j + 4 * grp + kk) * LW, l16);
#pragma unroll
                for (int i = 0; i < NT; ++i) o[i] = mfma16(vx[i], s[j][kk], o[i]);
            }
        }
    }

    const float l = sum4grp(lsum);
    const float inv = 1.f / l;
    if (a.lse && grp == 0 && my_row < a.T)  // natural log: (m + log2 l) ln 2
        a.lse[((size_t)b * a.T + my_row) * a.H + h] = (m + log2f(l)) * 0.69314718055994531f;
    if (my_row < a.T) {
        float *orow = a.out + (size_t)b * a.T * qld + (size_t)my_row * qld + (size_t)h * a.dim;
#pragma unroll
        for (int r = 0; r < 4; ++r) store_run<NT>(orow, 4 * grp + r, a.dim, vec4, o, r, inv);
    }
}

// Row tile n - 1 - p (latest, heaviest first); with a.pair also row tile p,
// so that every workgroup has the same causal work.
template <int DP, int BK, int NW, bool PF>
__device__ __forceinline__ void attn_fwd_body(const FwdArgs &a) {
    const int p = (int)blockIdx.x / (a.n_head_blocks * a.B);
    attn_fwd_tile<DP, BK, NW, PF>(a, a.n_row_tiles - 1 - p);
    if (a.pair && p < a.n_row_tiles - 1 - p) {  // workgroup-uniform
        __syncthreads();  // the first tile's last LDS reads before the second's writes
        attn_fwd_tile<DP, BK, NW, PF>(a, p);
    }
}

// ---- The forward on split operands (split.h) --------------------------------
//
// The schedule of the wide-row kernels (dim % 4 == 0): the same two products
// S^T = K Q^T and O^T += V^T P^T and the same softmax as attn_fwd_tile, on the
// bf16 matrix cores.  A wave owns NQ blocks of 16 query rows of one head, the
// workgroup HW heads of one kv group x RB row blocks x KS key parts x DS column
// halves of waves.
//   * K and V tiles of 32 keys (per key part) are split once while they are
//     staged and shared by the workgroup's waves, row-major in LDS; the V^T
//     operand comes from the same layout through the transposing LDS read.
//   * Two phases per step, a barrier after each: scores, then softmax and
//     output product.  Eight waves, where two buffers each of K and V fit in
//     LDS (ALT): the second four waves, one per SIMD, run half a step behind
//     the first, so that on every SIMD one wave's softmax and staging run
//     beside the other's MFMAs; the score phase stages the next K and the
//     output phase the next V.  Otherwise one buffer each: the waves write this
//     step's V while they multiply K and the next K while they multiply V.
//   * Q's split stays in registers (12 per 32 columns and row block), P's is
//     formed from the score registers.
//   * O accumulates 32-key sums with f32 adds: four vector adds beside six
//     MFMAs, and a long row takes T / 32 roundings instead of 6 T / 32.
// What bounds it: on a full chip the MFMAs, which are busy 55 % of the time, and the
// vector work beside them, two instructions of 4 cycles to each MFMA of 16 (a 16 x 16
// score block at d = 128 is 48 MFMAs; its softmax and split about 70 vector
// instructions), at two waves per SIMD, with power holding the clock to 2.27 GHz (2.15
// with the scores kept; counters).  A loop of such MFMAs on operands like these
// reaches 371 TFLOP/s of f32 products alone and 312 with two vector instructions
// beside each.  32 over 8 heads,
// d = 128, T = 4096: 1012 us on f32 MFMAs, 614 us here (224 TFLOP/s), with the
// scores kept 1053 / 705 us; d = 256, 2 x 2048 rows of 16 over 4 heads 538 / 437 us.
// On small grids, the latency of a step (fetch, split, barrier, two dependent
// products): 512 rows of that first shape 70 / 34 us.  Two row blocks per wave (NQ = 2) read each K and V
// operand from LDS once for 32 rows: at one block the operand reads alone
// (49 KB per wave and tile at d = 128) would take as long as the MFMAs.
template <int DP, int NW, int NQ, int KS>
struct FwdSplit {
    static constexpr FwdWaves W{NW, NQ, KS};
    static constexpr int DS = fwd_ds(DP);   // column halves
    static constexpr int DW = DP / DS;      // columns per wave
    static constexpr int NT = DW / 16;      // 16-wide output tiles per wave
    static constexpr int NKS = DW / 32;     // 32-wide contraction steps of the score product
    static constexpr int ROWS = 32 * KS;    // keys staged per step
    static constexpr int TILE = split_bytes(DP, ROWS);
    static constexpr int MERGE = (KS - 1) * (NW / KS) * 64 * (4 * NQ * NT + 2 * NQ) * 4;
    // Alternating wave halves (below): two buffers each for K and V.
    static constexpr bool ALT = fwd_alt(DP, W);
    static constexpr int XCHG = fwd_tiles_lds(DP, W);  // offset of the column halves' partial scores
    static constexpr int BYTES = fwd_lds(DP, W);
    static constexpr int FLAGS = BYTES - 16;           // offset of the big-value flags
    static_assert(MERGE <= XCHG, "the key parts merge in the tiles' space");
    static_assert(BYTES <= 160 * 1024, "LDS");
};

// 4 x 4 transpose within each group of four lanes: lane i ends with element i
// of the group's lanes 0..3.
DEVI f4 quad_transpose(f4 x, int lane) {
    const bool o1 = lane & 1, o2 = lane & 2;
    // (The lane exchanges are outside the selects: every lane takes part.)
    auto xor1 = [](float v) { return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xb1, 0xf, 0xf, true)); };
    auto xor2 = [](float v) { return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x4e, 0xf, 0xf, true)); };
    const float x0 = xor1(x.x), x1 = xor1(x.y), x2 = xor1(x.z), x3 = xor1(x.w);
    const float a0 = o1 ? x1 : x.x, a1 = o1 ? x.y : x0, a2 = o1 ? x3 : x.z, a3 = o1 ? x.w : x2;
    const float y0 = xor2(a0), y1 = xor2(a1), y2 = xor2(a2), y3 = xor2(a3);
    return f4{o2 ? y2 : a0, o2 ? y3 : a1, o2 ? a2 : y0, o2 ? a3 : y1};
}

template <int DP, int NW, int NQ, int KS, int SC>
DEVI void fwd_split_tile(const FwdArgs &a, const int tile, char *const smem, int &sid) {
    using C = FwdSplit<DP, NW, NQ, KS>;
    constexpr int DS = C::DS, DW = C::DW, NT = C::NT, NKS = C::NKS, ROWS = C::ROWS, NTH = 64 * NW, NWR = NW / (KS * DS);
    constexpr bool ALT = C::ALT;
    char *const xchg = smem + C::XCHG;
    // The K (V) tile of a step, and the flag that holds the step's id if the tile has a big value.
    auto ktile = [&](int id) { return smem + (ALT ? (id & 1) * 2 * C::TILE : 0); };
    auto vtile = [&](int id) { return ktile(id) + C::TILE; };
    auto kflag = [&](int id) { return reinterpret_cast<int *>(smem + C::FLAGS) + (ALT ? (id & 1) * 2 : 0); };
    auto vflag = [&](int id) { return kflag(id) + 1; };

    const int tid = opaque((int)threadIdx.x), lane = tid & 63, l16 = lane & 15, grp = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kh = w / (NW / KS);       // key part
    const int dh = (w / NWR) % DS;      // column half
    const int wr = w % NWR;             // (head, row block) slot
    const int RB = NWR / a.HW;
    const int per_tile = a.n_head_blocks * a.B;
    const int rem = (int)blockIdx.x % per_tile;
    const int hb = rem % a.n_head_blocks, b = rem / a.n_head_blocks;
    const int h = hb * a.HW + (wr % a.HW);
    const int kvh = ZT_PLANT == 2 ? 0 : h / (a.H / a.Hkv);
    const int wg_row0 = tile * 16 * NQ * RB;
    const int row0 = wg_row0 + 16 * NQ * (wr / a.HW);
    const size_t qld = (size_t)a.H * a.dim, kld = (size_t)a.Hkv * a.dim;
    const float *qb = a.q + (size_t)b * a.T * qld + (size_t)h * a.dim;
    const float *kb = a.k + (size_t)b * a.kv_rows * kld + (size_t)kvh * a.dim;
    const float *vb = a.v + (size_t)b * a.kv_rows * kld + (size_t)kvh * a.dim;
    const float qscale = ZT_PLANT == 4 ? kLog2e : a.scale_log2e;

    // Staging: thread tid takes the 8-column chunks e = tid + n NTH of the
    // step's ROWS x DP tile.  Loads are unconditional and in bounds: rows past
    // n_keys load row n_keys - 1 (masked scores, weight 0), columns past dim
    // the row's last floats (replaced by 0).
    constexpr int CPR = DP / 8, CH = ROWS * CPR, NP = (CH + NTH - 1) / NTH;
    constexpr bool EVEN = CH % NTH == 0;
    // Byte offsets within a tile's rows, fixed for the kernel; a fetch clamps
    // them (one min) to row n_keys - 1 counted within the tile.  ROWS kld 4 <
    // 2^32 at every width and head count admitted (ROWS DP <= 8192).
    constexpr int NC = NTH % CPR == 0 ? 1 : NP;  // distinct columns among a thread's chunks
    unsigned voff[NP], vcol[NC], vcol2[NC];
#pragma unroll
    for (int n = 0; n < NP; ++n) voff[n] = (unsigned)((tid + n * NTH) / CPR) * (unsigned)kld * 4u;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = (tid + n * NTH) % CPR * 8;
        vcol[n] = (unsigned)min(c, a.dim - 4) * 4u;
        // The chunk's second half; past dim it is replaced by 0, so anything in bounds will do.
        vcol2[n] = c + 4 < a.dim ? vcol[n] + 16u : vcol[n];
    }
    auto fetch = [&](f4 (&x)[NP][2], const float *base, int k0) {
        const unsigned last = (unsigned)min(a.n_keys - 1 - k0, ROWS - 1) * (unsigned)kld * 4u;
        const char *p = reinterpret_cast<const char *>(base + (size_t)k0 * kld);
#pragma unroll
        for (int n = 0; n < NP; ++n) {
            if (!EVEN && tid + n * NTH >= CH) break;  // wave-uniform: CH is a multiple of 64
            const unsigned r = min(voff[n], last);
            x[n][0] = *reinterpret_cast<const f4 *>(p + (r + vcol[n % NC]));
            x[n][1] = *reinterpret_cast<const f4 *>(p + (r + vcol2[n % NC]));
        }
    };
    auto put = [&](const f4 (&x)[NP][2], char *t, int *flag, int id, auto split) {
#pragma unroll
        for (int n = 0; n < NP; ++n) {
            const int e = tid + n * NTH;
            if (!EVEN && e >= CH) break;
            const int c = (e % CPR) * 8;
            float y[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) y[i] = x[n][i / 4][i % 4];
            if (a.dim < DP) {
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = c + (i & 4) < a.dim ? y[i] : 0.f;
            }
            if (any_big(max_abs(y))) {
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = small_part(y[i]);
                if (lane == 0) *flag = id;
            }
            put_tri<DP>(t, ROWS, e / CPR, c, split(y));
        }
    };

    // Q: the B operand of the score product, lane l16 = row, k slot = column.
    Tri q[NKS][NQ];
    float qmax = 0.f;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int row = row0 + 16 * n + l16;
        const float *qrow = qb + (size_t)min(row, a.T - 1) * qld;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const int c = dh * DW + 32 * ks + 8 * grp;
            float y[8];
#pragma unroll
            for (int i = 0; i < 8; i += 4) {
                // Unconditional and in bounds; rows past T and columns past dim are 0.
                const f4 x = *reinterpret_cast<const f4 *>(qrow + min(c + i, a.dim - 4));
                const bool in = row < a.T && c + i < a.dim;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[i + e] = in ? x[e] * qscale : 0.f;
            }
            const float mx = max_abs(y);
            qmax = vmax(qmax, mx);
            if (any_big(mx)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = small_part(y[i]);
            }
            q[ks][n] = split8_as_is(y);
        }
    }
    const bool qbig = any_big(qmax);

    f4 o[NT][NQ];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int n = 0; n < NQ; ++n) o[i][n] = zero4();
    float m[NQ], lsum[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) { m[n] = -INFINITY; lsum[n] = 0.f; }
    const int kend_wg = min(a.n_keys, a.q_offset + min(a.T, wg_row0 + 16 * NQ * RB));
    const int kend_w = row0 < a.T ? min(a.n_keys, a.q_offset + min(a.T, row0 + 16 * NQ)) : 0;

    // Scores (kept if SC) to weights in s, the row state updated.
    f4 s[2 * NQ];  // s[j NQ + n]: keys k0 + 16 j + 4 grp + r of row block n
    auto softmax = [&](const int k0) {
        if (SC == 1 || (SC == 2 && a.s_out)) {
        // Element (t = row + l16, s = k0 + 16 j + 4 grp + r) belongs at lane
        // (s & 15) + 16 ((t & 15) >> 2), element t & 3 of its tile: after the
        // quad transpose a lane holds four consecutive rows of one key, and
        // the wave's 16-byte stores cover the tile's 1 KB (nontemporal: the
        // tiles would displace the K/V rows the workgroups share in L2).
        const int nt = (a.T + 15) >> 4;
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            if (DS > 1 && n % DS != dh) continue;
            const int r0 = row0 + 16 * n;
            const int kend = r0 < a.T ? min(a.n_keys, min(a.T, r0 + 16)) : 0;
            float *srow = a.s_out +
                          (((size_t)b * a.H + h) * zt_tri_count(nt) + zt_tri_index(r0 >> 4, k0 >> 4)) * 256 +
                          (4 * grp + (l16 & 3) + 16 * (l16 >> 2)) * 4;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (k0 + 16 * j >= kend) continue;  // wave-uniform: above the diagonal
                f4 x = quad_transpose(s[j * NQ + n], lane);
                if (ZT_PLANT == 5) x = x / a.scale_log2e;
                __builtin_nontemporal_store(x, reinterpret_cast<f4 *>(srow + j * 256));
            }
        }
        }
        if (k0 + 31 > a.q_offset + row0 || k0 + 32 > a.n_keys) {  // wave-uniform
#pragma unroll
        for (int i = 0; i < 2 * NQ; ++i) {
            const int qpos = a.q_offset + row0 + 16 * (i % NQ) + l16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = k0 + 16 * (i / NQ) + 4 * grp + r;
                if ((ZT_PLANT != 1 && key > qpos) || key >= a.n_keys) s[i][r] = -INFINITY;
            }
        }
        }
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = s[(i / 4) * NQ + n][i % 4];
        const float mt = max4grp(vmax_n(y));
        // Lazy rescaling, per row (attn_fwd_tile).
        if (ZT_PLANT == 3 || mt > m[n] + 8.f) {
            const float mnew = fmaxf(m[n], mt);
            const float corr = fast_exp2(m[n] - mnew);
            m[n] = mnew;
            lsum[n] = ZT_PLANT == 3 ? lsum[n] : lsum[n] * corr;
#pragma unroll
            for (int i = 0; i < NT; ++i) o[i][n] *= ZT_PLANT == 3 ? 1.f : corr;
        }
        // A row whose every key so far is masked (a later row block, or a
        // key part past the first) keeps base -inf, taken as 0 here so that
        // exp2(-inf) = 0.
        const float mb = m[n] == -INFINITY ? 0.f : m[n];
        float ps = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            y[i] = fast_exp2(y[i] - mb);
            s[(i / 4) * NQ + n][i % 4] = y[i];
            ps = i == 0 ? y[0] : ps + y[i];
        }
        lsum[n] += ps;
        }
    };
    // Where registers allow (DEEP) a tile is fetched a whole step before it is
    // written to LDS, else in the phase that writes it, which is shorter than the
    // loads' latency for small tiles.
    constexpr bool DEEP = NQ == 1 || DW <= 64;
    f4 px[NP][2], py[DEEP ? NP : 1][2];
    const auto as_is = [](const float (&y)[8]) { return split8_as_is(y); };
    const auto scaled = [](const float (&y)[8]) { return split8(y); };
    auto stage_k = [&](int id) { put(px, ktile(id), kflag(id), id, as_is); };
    auto stage_v = [&](int id) {
        if constexpr (DEEP) put(py, vtile(id), vflag(id), id, scaled);
        else put(px, vtile(id), vflag(id), id, scaled);
    };
    const int klast = (kend_wg - 1) / ROWS * ROWS;  // the last step's first key
    fetch(px, kb, 0);
    stage_k(sid + 1);
    if constexpr (DEEP) fetch(py, vb, 0);
    if constexpr (ALT) {
        if constexpr (!DEEP) fetch(px, vb, 0);
        stage_v(sid + 1);
        if constexpr (DEEP) fetch(py, vb, min(ROWS, klast));
    }
    if constexpr (DEEP) fetch(px, kb, min(ROWS, klast));
    __syncthreads();
    // Half a step behind: the second half's waves meet one barrier more here, the first half's one more at the end.
    if (ALT && w >= NW / 2) __syncthreads();
    for (int ks0 = 0; ks0 < kend_wg; ks0 += ROWS) {
        ++sid;
        // The steps after this one (the last loads itself again, unused).
        const int kn = min(ks0 + ROWS, klast), kn2 = min(ks0 + 2 * ROWS, klast);
        const int k0 = ks0 + 32 * kh;
        const bool active = k0 < kend_w;  // wave-uniform
        // Phase A: scores; this step's V (ALT: the next K) into LDS.
        if constexpr (!DEEP) fetch(px, ALT ? kb : vb, ALT ? kn : ks0);
        const char *const Ks = ktile(sid), *const Vs = vtile(sid);
        if (active) {
#pragma unroll
            for (int i = 0; i < 2 * NQ; ++i) s[i] = zero4();
            // One 16-key block at a time: step (j, ks) = (i / NKS, i % NKS).
            stream_parts<2 * NKS, 3>(
                [&](int i, int part) {
                    return get_row<DP>(Ks, ROWS, 32 * kh + 16 * (i / NKS), dh * DW + 32 * (i % NKS), l16, grp, part);
                },
                [&](int i, auto part, u4 x) {
                    f4 t[NQ];
#pragma unroll
                    for (int n = 0; n < NQ; ++n) t[n] = s[(i / NKS) * NQ + n];
                    mfma_parts<part>(t, x, [&](int n) -> const Tri & { return q[i % NKS][n]; });
#pragma unroll
                    for (int n = 0; n < NQ; ++n) s[(i / NKS) * NQ + n] = t[n];
                });
            const bool kbig = __builtin_amdgcn_readfirstlane(*kflag(sid)) == sid;
            if (kbig || qbig) {
                // Products with a big operand, from the full values.
                if (kbig && qbig) {  // both sides: the whole product in f32
#pragma unroll
                    for (int i = 0; i < 2 * NQ; ++i) s[i] = zero4();
                }
                const int ll = opaque(lane), lrow = ll & 15, lgrp = ll >> 4;
#pragma unroll 1
                for (int cc = 0; cc < 8 * NKS; ++cc) {
                        const int c = dh * DW + 32 * (cc >> 3) + 8 * lgrp + (cc & 7);
                        float kv[2], qv[NQ];
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const int key = min(k0 + 16 * j + lrow, a.n_keys - 1);
                            kv[j] = c < a.dim ? kb[(size_t)key * kld + c] : 0.f;
                            if (!qbig) kv[j] = big_part(kv[j]);
                        }
#pragma unroll
                        for (int n = 0; n < NQ; ++n) {
                            const int row = row0 + 16 * n + lrow;
                            qv[n] = row < a.T && c < a.dim ? qb[(size_t)row * qld + c] * qscale : 0.f;
                            if (!kbig) qv[n] = big_part(qv[n]);
                        }
#pragma unroll
                        for (int i = 0; i < 2 * NQ; ++i) s[i] = mfma16(kv[i / NQ], qv[i % NQ], s[i]);
                    }
            }
            if constexpr (DS == 1) {
                softmax(k0);
            } else {
#pragma unroll
                for (int i = 0; i < 2 * NQ; ++i)
                    *reinterpret_cast<f4 *>(xchg + ((w * 2 * NQ + i) * 64 + lane) * 16) = s[i];
            }
        }
        if constexpr (ALT) {
            stage_k(sid + 1);
            if constexpr (DEEP) fetch(px, kb, kn2);
        } else {
            stage_v(sid);
            if constexpr (DEEP) fetch(py, vb, kn);
        }
        __syncthreads();

        // Phase B: softmax and the output product; the next K (ALT: V) into LDS.
        if constexpr (!DEEP) fetch(px, ALT ? vb : kb, kn);
        if (active) {
            if constexpr (DS > 1) {  // f32 addition commutes: both halves get the same scores
                const int other = w ^ NWR;
#pragma unroll
                for (int i = 0; i < 2 * NQ; ++i)
                    s[i] += *reinterpret_cast<const f4 *>(xchg + ((other * 2 * NQ + i) * 64 + lane) * 16);
            }
            if constexpr (DS > 1) softmax(k0);
            Tri p[NQ];
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                float y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = s[(i / 4) * NQ + n][i % 4];
                p[n] = split8_as_is(y);
            }
            f4 t[NQ];
            stream_parts<NT, 3>(
                [&](int i, int part) { return get_col<DP>(Vs, ROWS, 32 * kh, dh * DW + 16 * i, lane, part); },
                [&](int i, auto part, u4 x) {
                    if constexpr (part == 0) {
#pragma unroll
                        for (int n = 0; n < NQ; ++n) t[n] = zero4();
                    }
                    mfma_parts<part>(t, x, [&](int n) -> const Tri & { return p[n]; });
                    if constexpr (part == 2) {
#pragma unroll
                        for (int n = 0; n < NQ; ++n) o[i][n] += t[n] * kUnscale1;
                    }
                });
            if (__builtin_amdgcn_readfirstlane(*vflag(sid)) == sid) {
                // V's big values, from the full rows (P is at most 2^8, or NaN).
                const int ll = opaque(lane), lcol = ll & 15, lgrp = ll >> 4;
#pragma unroll 1
                for (int jr = 0; jr < 8; ++jr) {
                        const int key = min(k0 + 16 * (jr >> 2) + 4 * lgrp + (jr & 3), a.n_keys - 1);
                        float pv[NQ];
#pragma unroll
                        for (int n = 0; n < NQ; ++n) {
                            unsigned ph = p[n].h.x, pm = p[n].m.x, pl = p[n].l.x;
#pragma unroll
                            for (int e = 1; e < 4; ++e) {
                                ph = jr >> 1 == e ? p[n].h[e] : ph;
                                pm = jr >> 1 == e ? p[n].m[e] : pm;
                                pl = jr >> 1 == e ? p[n].l[e] : pl;
                            }
                            pv[n] = join_bf16(ph, pm, pl, jr & 1);
                        }
#pragma unroll
                        for (int i = 0; i < NT; ++i) {
                            const int c = dh * DW + 16 * i + lcol;
                            const float vv = c < a.dim ? big_part(vb[(size_t)key * kld + c]) : 0.f;
#pragma unroll
                            for (int n = 0; n < NQ; ++n) o[i][n] = mfma16(vv, pv[n], o[i][n]);
                        }
                    }
            }
        }
        if constexpr (ALT) {
            stage_v(sid + 1);
            if constexpr (DEEP) fetch(py, vb, kn2);
        } else {
            stage_k(sid + 1);
            if constexpr (DEEP) fetch(px, kb, kn2);
        }
        __syncthreads();
    }
    if (ALT && w < NW / 2) __syncthreads();
    ++sid;  // the last step staged tiles for the step that does not follow

    if constexpr (KS > 1) {
        // Merge the key parts: parts 1.. leave their base, partial sum and output
        // in LDS, part 0 rescales to the larger base and adds them, in part order (a
        // part that saw no visible key has m = -inf and contributes nothing).  (The
        // loop ended with a barrier.)
        constexpr int SF = 4 * NQ * NT + 2 * NQ;
        auto slot = [&](int part) {
            return reinterpret_cast<float *>(smem) + (((part - 1) * (NW / KS) + (w % (NW / KS))) * SF) * 64 + lane * 4;
        };
        if (kh > 0) {
            float *mb = slot(kh);
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int n = 0; n < NQ; ++n) *reinterpret_cast<f4 *>(mb + (i * NQ + n) * 256) = o[i][n];
            float *ml = mb + 4 * NQ * NT * 64 - lane * 4 + lane;
#pragma unroll
            for (int n = 0; n < NQ; ++n) { ml[(2 * n) * 64] = m[n]; ml[(2 * n + 1) * 64] = lsum[n]; }
        }
        __syncthreads();
        if (kh == 0) {
#pragma unroll
            for (int part = 1; part < KS; ++part) {
                const float *mb = slot(part);
                const float *ml = mb + 4 * NQ * NT * 64 - lane * 4 + lane;
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    const float m2 = ml[(2 * n) * 64], l2 = ml[(2 * n + 1) * 64];
                    const float mm = fmaxf(m[n], m2);
                    const float f1 = ZT_PLANT == 3 ? 1.f : m[n] == -INFINITY ? 0.f : fast_exp2(m[n] - mm);
                    const float f2 = ZT_PLANT == 3 ? 1.f : m2 == -INFINITY ? 0.f : fast_exp2(m2 - mm);
                    lsum[n] = lsum[n] * f1 + l2 * f2;
#pragma unroll
                    for (int i = 0; i < NT; ++i)
                        o[i][n] = o[i][n] * f1 + *reinterpret_cast<const f4 *>(mb + (i * NQ + n) * 256) * f2;
                    m[n] = mm;
                }
            }
        }
        __syncthreads();  // the merge's reads before the next tile's staging
        if (kh != 0) return;
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int el = opaque(lane), egrp = el >> 4;
        const int row = row0 + 16 * n + (el & 15);
        const float l = sum4grp(lsum[n]);
        const float inv = 1.f / l;
        if (row >= a.T) continue;
        if (a.lse && egrp == 0 && dh == 0)  // natural log: (m + log2 l) ln 2
            a.lse[((size_t)b * a.T + row) * a.H + h] = (m[n] + log2f(l)) * 0.69314718055994531f;
        float *orow = a.out + (size_t)b * a.T * qld + (size_t)row * qld + (size_t)h * a.dim;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int c = dh * DW + 16 * i + 4 * egrp;
            if (c < a.dim) *reinterpret_cast<f4 *>(orow + c) = o[i][n] * inv;
        }
    }
}

template <int DP, int NW, int NQ, int KS, int SC>
DEVI void fwd_split_body(const FwdArgs &a, char *smem) {
    const int p = (int)blockIdx.x / (a.n_head_blocks * a.B);
    using C = FwdSplit<DP, NW, NQ, KS>;
    if (threadIdx.x < 4) reinterpret_cast<int *>(smem + C::FLAGS)[threadIdx.x] = 0;
    __syncthreads();
    int sid = 0;
    // One copy of the tile's code: a second one would cost registers, which at d = 128 spill as it is (2 to 22).
    const int second = a.n_row_tiles - 1 - p;
    int tile = second;
#pragma unroll 1
    for (;;) {  // workgroup-uniform (every tile ends after a barrier)
        fwd_split_tile<DP, NW, NQ, KS, SC>(a, tile, smem, sid);
        if (!a.pair || tile == p || p >= second) break;
        tile = p;
    }
}
#define ZT_FWD(DP, BK)                                                                             \
    extern "C" __global__ void __launch_bounds__(256) zt_fwd_d##DP##_k##BK(FwdArgs a) {          \
        attn_fwd_body<DP, BK, 4, false>(a);                                                        \
    }                                                                                              \
    extern "C" __global__ void __launch_bounds__(512) zt_fwd8_d##DP##_k##BK(FwdArgs a) {         \
        attn_fwd_body<DP, BK, 8, false>(a);                                                        \
    }
// Kernels on split operands: one per role and width, each holding the role's wave
// shapes (shapes.h), of which the launcher picks by the grid (FwdArgs::nq, ks); at
// d = 32 one per shape.
// SC: 0 never keeps the scores, 1 always, 2 where s_out is set.
template <int DP, int SC, int NW, int NQ, int KS>
DEVI bool fwd_shape(const FwdArgs &a, char *smem) {
    if (a.nq != NQ || a.ks != KS || blockDim.x != 64 * NW) return false;  // workgroup-uniform
    fwd_split_body<DP, NW, NQ, KS, SC>(a, smem);
    return true;
}
template <FwdRole R, int DP, int SC>
DEVI void fwd_shapes(const FwdArgs &a) {
    __shared__ __attribute__((aligned(16))) char smem[fwd_lds(R, DP)];
    constexpr FwdWavesList L = fwd_waves(R, DP);
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (void)(fwd_shape<DP, SC, L.s[I].nw, L.s[I].nq, L.s[I].ks>(a, smem) || ...);
    }(std::make_integer_sequence<int, L.n>{});
}
template <int DP, int SC, int NW, int NQ, int KS>
DEVI void fwd_one_shape(const FwdArgs &a) {
    __shared__ __attribute__((aligned(16))) char smem[fwd_lds(DP, {NW, NQ, KS})];
    fwd_split_body<DP, NW, NQ, KS, SC>(a, smem);
}
// zt_fwd8ps_* is zt_fwd8p_* keeping the scores: its own name, so that a profile tells the two apart.
#define ZT_FWD_SPLIT(NAME, ROLE, DP, SC)                                                             \
    extern "C" __global__ void __launch_bounds__(512, 2) NAME##_d##DP##_k32(FwdArgs a) {          \
        fwd_shapes<FwdRole::ROLE, DP, SC>(a);                                                        \
    }
#define ZT_FWD_SHAPE(NAME, SC, NW, NQ, KS)                                                           \
    extern "C" __global__ void __launch_bounds__(512, 2) NAME##_d32_k32_##NW##NQ##KS(FwdArgs a) { \
        fwd_one_shape<32, SC, NW, NQ, KS>(a);                                                        \
    }
#define ZT_8P_32(NW, NQ, KS) ZT_FWD_SHAPE(zt_fwd8p, 0, NW, NQ, KS)
#define ZT_8PS_32(NW, NQ, KS) ZT_FWD_SHAPE(zt_fwd8ps, 1, NW, NQ, KS)
#define ZT_P_32(NW, NQ, KS) ZT_FWD_SHAPE(zt_fwdp, 2, NW, NQ, KS)
#define ZT_PK_32(NW, NQ, KS) ZT_FWD_SHAPE(zt_fwdpk, 2, NW, NQ, KS)

// Register-prefetched variants on f32 MFMA (32-key tiles; widths whose halves
// are not whole 32-column groups).
#define ZT_FWD_PF(DP)                                                                              \
    extern "C" __global__ void __launch_bounds__(256) zt_fwdp_d##DP##_k32(FwdArgs a) {           \
        attn_fwd_body<DP, 32, 4, true>(a);                                                         \
    }                                                                                              \
    extern "C" __global__ void __launch_bounds__(512, (DP) <= 128 ? 4 : 1) zt_fwd8p_d##DP##_k32(FwdArgs a) { \
        attn_fwd_body<DP, 32, 8, true>(a);                                                         \
    }

#if ZT_PLANT == 0
ZT_FWD(32, 32) ZT_FWD(32, 64)
ZT_FWD(64, 32) ZT_FWD(64, 64)
ZT_FWD(96, 32) ZT_FWD(96, 64)
ZT_FWD(128, 32) ZT_FWD(128, 64)
ZT_FWD(160, 32) ZT_FWD(160, 64)
ZT_FWD(192, 32) ZT_FWD(192, 64)
ZT_FWD(224, 32) ZT_FWD(224, 64)
ZT_FWD(256, 32) ZT_FWD(256, 64)
ZT_FWD_PF(160) ZT_FWD_PF(224)
ZT_FWD_HEADS_32(ZT_8P_32) ZT_FWD_SPLIT(zt_fwd8p, Heads, 64, 0)
ZT_FWD_SPLIT(zt_fwd8p, Heads, 96, 0) ZT_FWD_SPLIT(zt_fwd8p, Heads, 128, 0)
ZT_FWD_HEADS_32(ZT_8PS_32) ZT_FWD_SPLIT(zt_fwd8ps, Heads, 64, 1)
ZT_FWD_SPLIT(zt_fwd8ps, Heads, 96, 1) ZT_FWD_SPLIT(zt_fwd8ps, Heads, 128, 1)
ZT_FWD_SPLIT(zt_fwd8p, Heads, 192, 2) ZT_FWD_SPLIT(zt_fwd8p, Heads, 256, 2)
ZT_FWD_ONE_32(ZT_P_32) ZT_FWD_SPLIT(zt_fwdp, One, 64, 2)
ZT_FWD_SPLIT(zt_fwdp, One, 96, 2) ZT_FWD_SPLIT(zt_fwdp, One, 128, 2)
ZT_FWD_SPLIT(zt_fwdp, One, 192, 2) ZT_FWD_SPLIT(zt_fwdp, One, 256, 2)
ZT_FWD_SMALL_32(ZT_PK_32) ZT_FWD_SPLIT(zt_fwdpk, Small, 64, 2)
ZT_FWD_SPLIT(zt_fwdpk, Small, 96, 2) ZT_FWD_SPLIT(zt_fwdpk, Small, 128, 2)
#else
// A planted-defect build (test-only): the kernels of the negative-control
// shapes, d = 32 (the reference entry points) and d = 128 (the training path).
ZT_FWD_HEADS_32(ZT_8P_32) ZT_FWD_SPLIT(zt_fwd8p, Heads, 128, 0)
ZT_FWD_SPLIT(zt_fwd8ps, Heads, 128, 1)
#endif
