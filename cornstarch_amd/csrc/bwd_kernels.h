// Backward kernels of bitfield-masked attention for gfx950 (templates; instantiated by bwd_dkdv.hip, bwd_dq.hip
// and bwd_long.hip).
// Reference semantics: cornstarch/kernel/bitfield_attention.py:527-572 (delta) and :598-929
// (dQ, dK, dV).  The reference accumulates dQ, dK and dV with fp32 atomics; here every output
// element has exactly one owner, so nothing is atomic and the sums are deterministic:
//   dkdv kernel : one workgroup per (batch, kv head, 128-key tile); it loops over the q heads
//                 of the group and over the query blocks its flag column lists.
//   dq kernel   : one workgroup per (batch, q head, 128-query block), looping over key tiles
//                 exactly like the forward kernel.
// Both recompute P = exp(scale * s - lse) from the saved log-sum-exp.
#pragma once
#include "bam_common.h"
#include "bam_launch.h"
#include "../../include/bam_hip.h"
#include "bam_tiles.h"
#include <type_traits>

namespace bam {

// ---------------------------------------------------------------------------------------
// One 16-byte chunk of o . do.  (The delta pre-pass and the dQ kernel sum the chunks of a row in the same order, so that
// it does not matter which of them computes delta.)
template <typename T>
__device__ __forceinline__ float chunk_dot(const u32x4& x, const u32x4& y) {
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        acc = fmaf(T::to_float((unsigned short)(x[i] & 0xFFFFu)), T::to_float((unsigned short)(y[i] & 0xFFFFu)), acc);
        acc = fmaf(T::to_float((unsigned short)(x[i] >> 16)), T::to_float((unsigned short)(y[i] >> 16)), acc);
    }
    return acc;
}

// delta[b,h,i] = sum_d o * do   (fp32).  LDS_COLS/8 lanes per row, 16 bytes per lane per tensor.
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_preprocess_kernel(const AttnParams p) {
    constexpr int LPR = LDS_COLS<D> / 8;
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = gid / LPR;
    const int c = (int)(gid % LPR);
    const int64_t total = (int64_t)p.B * p.Sq * p.Hq;
    const bool valid = row < total;
    int h = 0, i = 0, b = 0;
    float acc = 0.f;
    if (valid) {
        h = (int)(row % p.Hq);
        const int64_t bi = row / p.Hq;
        i = (int)(bi % p.Sq);
        b = (int)(bi / p.Sq);
        u32x4 ov = {0u, 0u, 0u, 0u}, gv = {0u, 0u, 0u, 0u};
        if (8 * c < p.d) {
            ov = *(const u32x4*)((const char*)p.o.ptr +
                                 2 * ((int64_t)b * p.o.sb + (int64_t)i * p.o.ss + (int64_t)h * p.o.sh) + c * 16);
            gv = *(const u32x4*)((const char*)p.dout.ptr +
                                 2 * ((int64_t)b * p.dout.sb + (int64_t)i * p.dout.ss + (int64_t)h * p.dout.sh) + c * 16);
        }
        acc = chunk_dot<T>(ov, gv);
    }
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (valid && c == 0) p.delta[(int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded + i] = acc;
}

// ---------------------------------------------------------------------------------------
// dK, dV.  One workgroup = one 128-key tile of one (batch, kv head), 8 waves: wave w owns keys
// [32 (w & 3), +32) and works on rows [32 (w >> 2), +32) of every 64-row tile of Q / dO that streams
// through LDS (two or four buffers), so each SIMD holds two waves whose MFMA and softmax phases
// interleave.  A 64-row tile is a PAIR of 32-row slices taken from the list of slices that have work
// for this key tile (they need not be neighbours in the sequence), one slice per row stream; a wave
// whose own 32 x 32 class is "empty" sits the tile out.  K and V of the tile sit in LDS for the whole kernel and are
// read as MFMA B operands; dK^T and dV^T (d x keys) stay in accumulators.
// With S = Q K^T computed as queries x keys, a lane of the C fragment owns ONE key and 16
// query rows, so P and dS feed dV^T = dO^T P and dK^T = Q^T dS as B operands from registers;
// Q^T and dO^T come from the transposing LDS read of the same row-major tiles.
// The two waves that share a key group hold partial sums; they add them to the caller's
// buffers one after the other (workgroup barrier in between), so the result stays
// deterministic and atomic free.
constexpr int DKDV_QT = 64;
constexpr int DKDV_THREADS = 512;

// MODE (MASK_*): MASK_INDEXED = explicit global positions p.posq / p.posk and gathered bitfield arrays;
// MASK_DENSE = a materialized bool mask read from global memory in partial tiles.
// BIAS: the forward added p.bias to scale * q.k (reference bitfield_attention.py:815-835); P is recomputed with it.
// LONG: sequences of more than MAX_SLICE_LIST 32-row slices (131072 rows), walked in several passes; the short form has
// no pass loop at all (a loop around the main loop costs registers and a few per cent).
// SAVE: every wave also stores its 32 x 32 block of -dS / scale (the packed operand of the dK product) to p.ds_ws, where
// the dQ kernel of bwd_dq_saved.h picks it up instead of recomputing S and dP.  Record and block layout: AttnParams.
// SCALED (head dims up to 64, where the dQ kernel runs first): the rows' lse * log2(e) comes from there (p.lse_scaled), the same
// numbers with one of some seven vector instructions per MFMA less.  dK/dV alone, us: 8 x 4096 tokens, 16 heads, D 64 581 -> 571
// (0.6 % of the step), 3001, 32 / 8 heads 103.4 -> 101.5, D 32, 4096 118 -> 112.  (Above D 64 the delta pre-pass would have to write it: 8192 tokens, 32 / 8
// heads, D 128 dK/dV 957 -> 943 but the pre-pass 22.9 -> 27.2, 25.6 with the rows of a head side by side; 4 x 1537 no gain.)
template <typename T, int D, int MODE, bool BIAS, bool LONG, bool SAVE = false, bool SCALED = false>
__global__ __launch_bounds__(DKDV_THREADS, 2) void bwd_dkdv_kernel(const AttnParams p) {
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = MODE == MASK_DENSE, SORTED = MODE == MASK_SORTED;
    constexpr bool ROW_POS = IDX || SORTED;  // the rows' positions travel with the tiles
    static_assert(!(SORTED && LONG), "no plan for so many rows");
    // A tile is 16 MFMAs per wave at head dims up to 64, half of what it is above, and there is room for four buffers: two tiles
    // are copied ahead and the workgroup meets after every second one.  dK/dV alone, us, a meeting per tile -> per two: D 64, 3001
    // tokens, 32 / 8 heads 190 -> 180, 2 x 700 57.7 -> 54.9, 8 x 4096, 16 heads 555 -> 532; D 32: 3001 148.8 -> 139.8.
    // (SORTED has row numbers to copy one tile earlier still.)
    constexpr bool DEEP = D <= 64 && !SORTED && !LONG;
    constexpr int NB = DEEP ? 4 : 2;  // tile buffers
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    __shared__ u32x4 sK[128 * NCH];
    __shared__ u32x4 sV[128 * NCH];
    __shared__ u32x4 sQ[NB][DKDV_QT * NCH];
    __shared__ u32x4 sDO[NB][DKDV_QT * NCH];
    __shared__ __attribute__((aligned(16))) float sLse[NB][DKDV_QT];      // natural-log lse of the rows
    __shared__ __attribute__((aligned(16))) float sDelta[NB][DKDV_QT];
    __shared__ __attribute__((aligned(16))) int64_t sQbf[NB][DKDV_QT];    // raw bitfields of the rows
    // their positions (ROW_POS).  SORTED: a tile's rows are gathered, so their numbers have to be here a tile earlier
    __shared__ __attribute__((aligned(16))) int sQpos[SORTED ? 3 : NB][DKDV_QT];
    __shared__ __attribute__((aligned(16))) unsigned sWq[DKDV_THREADS / 64][5][32];  // per-wave rule constants
    // DENSE with packed mask bits: for the two slices of the tile, one word per key of the workgroup's 128 keys
    __shared__ unsigned sColBits[MODE == MASK_DENSE ? NB : 1][2][MODE == MASK_DENSE ? 128 : 1];
    __shared__ int sListStore[MAX_SLICE_LIST + 1];  // entry -1: partner of the first entry of an odd count
    int* const sList = sListStore + 1;
    __shared__ int sCount;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave & 3, st = wave >> 2;
    const int hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
    const int Sq = p.Sq, Sk = p.Sk;
    const int G = p.Hq / p.Hkv;

    const int unit = blockIdx.x;
    const int hk = unit % p.Hkv;
    constexpr bool PARTS = !LONG;  // (a kv head's q heads may be dealt to several workgroups)
    const int kv_head = PARTS && p.kv_parts > 1 ? hk / p.kv_parts : hk;
    int ub = unit / p.Hkv;  // position of the (batch, key tile) in the order of falling work
    {
        // The hardware deals the workgroups of an XCD to its four shader engines in turn and launches them strictly
        // in order: a workgroup waits for a free compute unit on ITS engine while free units of the other engines sit
        // idle behind it.  In a plainly sorted list one engine would get the heaviest workgroup of every four and
        // hold everybody back (measured: units idle 19 us at the median, up to 90 us, before their second workgroup),
        // so every other run of 32 workgroups -- four per XCD, one per engine -- takes its tiles in reverse.
        const int P = (p.Hkv <= 32 && 32 % p.Hkv == 0) ? 32 / p.Hkv : 1;
        const int g = ub / P, r = ub - g * P;
        if ((g & 1) && (g + 1) * P <= p.num_kt * p.B) ub = g * P + (P - 1 - r);
    }
    int b = ub % p.B;
    int nt = ub / p.B;  // early key tiles (most queries under causality) first
    if (p.tile_order != nullptr) {  // with a plan: the tiles by falling amount of work, whatever the mask looks like
        const int code = p.tile_order[ub];
        b = code / p.num_kt;
        nt = code - b * p.num_kt;
    }

    // With sorted rows there are two launches: this one is for the sequences whose rows have been moved, or for the others.
    if ((SORTED || MODE == MASK_BITFIELD) && p.rows_moved != nullptr && (p.rows_moved[b] != 0) != SORTED) return;

    const int ns_total = (Sq + 31) >> 5;
    // ---- K, V of the tile -> LDS (once) ---------------------------------------------------
    {
        TileStage<D, 128, DKDV_THREADS> stK, stV;
        stK.setup(2 * p.k.ss, p.d / 8, tid);
        stV.setup(2 * p.v.ss, p.d / 8, tid);
        RowView<LONG> rows;
        rows.init((const char*)p.k.ptr + 2 * ((int64_t)b * p.k.sb + (int64_t)kv_head * p.k.sh), 2 * p.k.ss, Sk, 2 * p.d);
        stK.template load<WAIT>(rows.at(nt * 128), lds_addr(sK));
        rows.init((const char*)p.v.ptr + 2 * ((int64_t)b * p.v.sb + (int64_t)kv_head * p.v.sh), 2 * p.v.ss, Sk, 2 * p.d);
        stV.template load<WAIT>(rows.at(nt * 128), lds_addr(sV));
    }
    const int key = nt * 128 + kg * 32 + l32;
    const bool kvalid = key < Sk;
    // bitfields of the query rows
    const int64_t* bfrow = SORTED ? p.rows_bits + (int64_t)b * p.rows_sb : p.bfq + (int64_t)b * p.bfq_sb;
    const int64_t kf = (!DENSE && kvalid) ? p.bfk[(int64_t)b * p.bfk_sb + key] : 0;
    int kpos = (IDX && kvalid) ? p.posk[key] : key;  // global position of this lane's key
    unsigned klo = (unsigned)(kf & 0xFFFFFFFFll);
    unsigned khi = (unsigned)((uint64_t)kf >> 32);
    // first pass (usually the only one): the last MAX_SLICE_LIST slices.  (Its first class bytes asked for ahead of the K and V rows:
    // 8192 tokens, 32 / 8 heads, D 128, step 1778 -> 1795 us.)
    if (wave == 0) {
        const int s_begin = max(0, ns_total - MAX_SLICE_LIST);
        build_slice_list(p, b, nt, lane, s_begin, ns_total, load_slice_classes(p, b, nt, s_begin + lane, ns_total), sList, &sCount);
    }

    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            dk[db][i] = 0.f;
            dv[db][i] = 0.f;
        }
    f32x16 zero16;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero16[i] = 0.f;
    const float c2 = BIAS ? LOG2E : p.scale * LOG2E;  // with a bias the scores become scale * s + bias first

    // Flip the sign of every element of the V tile in LDS (once per workgroup, after the tile has landed and
    // before anybody reads it; the caller brackets it with workgroup barriers).  Where the head dim is below D, the
    // columns past it become zero in K and V: the Q and dO tiles hold other numbers there.
    auto negate_v_tile = [&]() {
#pragma unroll
        for (int i = 0; i < (128 * NCH) / DKDV_THREADS; ++i) {
            const int id = tid + DKDV_THREADS * i;
            u32x4 x = sV[id];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] ^= 0x80008000u;
            if (p.d < D) {
                const u32x4 z = {0u, 0u, 0u, 0u};
                if (8 * ((id % NCH) ^ swz<D>(id / NCH)) >= p.d) sK[id] = x = z;
            }
            sV[id] = x;
        }
    };
    bool v_negated = false;
    // Head dims up to 64 leave room for this wave's K and (negated) V operands of the S / dP phase in registers:
    // they are the same for every tile, and the phase then reads half as much from LDS.
    constexpr bool KV_REGS = D <= 64;
    u32x4 kfrag[KV_REGS ? KK : 1], vfrag[KV_REGS ? KK : 1];
    bool kv_loaded = false;
    auto load_kv_operands = [&]() {  // after the V tile has been negated and a barrier has published it
        if (KV_REGS && !kv_loaded) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                kfrag[kk] = lds_read_chunk<D>(sK, 32 * kg + l32, 2 * kk + hi);
                vfrag[kk] = lds_read_chunk<D>(sV, 32 * kg + l32, 2 * kk + hi);
            }
            kv_loaded = true;
        }
    };

    typedef SliceStage<D, DKDV_THREADS> Stage;
    constexpr int CPT = Stage::CPT;
    // copy instructions per wave and tile: Q, dO, one of the small rows and (IDX) the row positions
    constexpr int NLOADS = 2 * CPT + 1 + (IDX ? 1 : 0);
    static_assert(NLOADS <= 2 * KK, "one copy per MFMA of the S / dP phase");
    Stage stQ, stDO;
    stQ.setup(SORTED ? 0 : 2 * p.q.ss, p.d / 8, tid);
    stDO.setup(SORTED ? 0 : 2 * p.dout.ss, p.d / 8, tid);
    const unsigned ldsQ = lds_addr(sQ), ldsDO = lds_addr(sDO);
    constexpr unsigned TILE_BYTES = DKDV_QT * NCH * 16;
    // small rows of a tile: lse, delta and the two halves of the 64 int64 bitfields, 64 dwords each;
    // wave w copies row w & 3 (waves 4..7 repeat what waves 0..3 write, so that every wave issues the same
    // number of copies)
    // (DENSE: rows 2 and 3 are the packed mask words of keys 0..63 / 64..127 of the tile, for the slice of the
    // copying wave's row stream; without packed bits, waves 2, 3, 6, 7 repeat lse / delta instead)
    const bool col_bits_on = DENSE && p.col_bits != nullptr;
    // (SORTED: waves 4..7 copy the row numbers of the tile behind, row 4)
    const int small = (DENSE && !col_bits_on) ? (wave & 1) : SORTED ? min(wave, 4) : (wave & 3);
    const unsigned ldsSmall = small == 0   ? lds_addr(sLse)
                              : small == 1 ? lds_addr(sDelta)
                              : SORTED && small == 4 ? lds_addr(sQpos)
                              : DENSE      ? lds_addr(sColBits) + (unsigned)(st * 128 + (small - 2) * 64) * 4u
                                           : lds_addr(sQbf) + (small - 2) * 256u;
    const unsigned smallBytes = small < 2 || (SORTED && small == 4) ? DKDV_QT * 4u : DENSE ? 2 * 128 * 4u : DKDV_QT * 8u;  // per buffer
    // Where the copies of a tile read.  The scalar unit is shared by the whole compute unit, so the address
    // arithmetic is kept short: descriptors of the head in work are carried along and moved when the head changes, a slice
    // costs one 32-bit product.  The slice that holds the end of the sequence is copied like the others: its rows past the
    // end are zeros, with an empty bitfield, and the list never calls such a slice "full".
    struct HeadViews {
        RowView<LONG> q, g;    // rows of the head in q and dout
        RowView<false> small;  // this wave's small row: lse / delta of the head, or the bitfields (head independent)
    };
    const int64_t small_head_step = small < 2 ? (int64_t)p.Sq_rounded * 4 : 0;
    auto head_views = [&](int h) {
        HeadViews hv;
        hv.q.init((const char*)p.q.ptr + 2 * ((int64_t)b * p.q.sb + (int64_t)h * p.q.sh), 2 * p.q.ss, Sq, 2 * p.d);
        hv.g.init((const char*)p.dout.ptr + 2 * ((int64_t)b * p.dout.sb + (int64_t)h * p.dout.sh), 2 * p.dout.ss, Sq, 2 * p.d);
        if (small < 2)
            hv.small.init((small == 0 ? (SCALED ? p.lse_scaled : p.lse) : p.delta) + (int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded, 4, Sq, 4);
        else if (DENSE)  // (one row per slice)
            hv.small.init(p.col_bits + (int64_t)b * p.col_bits_sb + nt * 128 + (small - 2) * 64, p.col_bits_ss * 4, (Sq + 31) >> 5, 256);
        else
            hv.small.init(bfrow, 8, Sq, 8);
        if (SORTED && small == 4) hv.small.init(p.rows + (int64_t)b * p.rows_sb, 4, p.Sq_rounded, 4);
        return hv;
    };
    auto next_head = [&](HeadViews& hv) {
        hv.q.move(2 * (int64_t)p.q.sh);
        hv.g.move(2 * (int64_t)p.dout.sh);
        hv.small.move(small_head_step);
    };
    RowView<false> pos_rows;
    if (IDX) pos_rows.init(p.posq, 4, Sq, 4);
    // lanes 32..63 of a copy of 2 x 32 consecutive floats / ints take the second slice: their byte offset moves
    // from "the rows after the first slice" to it
    const unsigned upper_lanes = lane >= 32 ? 0xFFFFFFFFu : 0u;
    struct TileSource {
        TileSrc q[CPT], g[CPT], small, pos;
        unsigned small_voff, pos_voff;
        unsigned q_voff[SORTED ? CPT : 1], g_voff[SORTED ? CPT : 1];
    };
    const unsigned q_rs = (unsigned)(2 * p.q.ss), g_rs = (unsigned)(2 * p.dout.ss);  // row strides in bytes
    // SORTED: the row numbers of a tile (waves 4..7)
    auto numbers_of = [&](TileSource& t, const HeadViews& hv, int row_lo, int row_hi) {
        t.small = hv.small.at(row_lo);
        t.small_voff = (unsigned)(lane * 4) + ((unsigned)((row_hi - row_lo - 32) * 4) & upper_lanes);
    };
    const int from_lo = __builtin_amdgcn_readfirstlane(small == 2 ? -1 : 0), from_hi = __builtin_amdgcn_readfirstlane(small == 3 ? -1 : 0),
              from_aft = __builtin_amdgcn_readfirstlane(small == 4 ? -1 : 0);
    // SORTED: the tile whose 64 row numbers are at pos; the rows past the last one are numbered Sq, beyond every descriptor.
    // (rows below 2^17, strides below 2^24 and products below 2^31: 24-bit products give the offsets).  aft_lo, aft_hi: the
    // slices of the tile behind it.
    auto gathered_source = [&](const HeadViews& hv, const int* pos, int row_lo, int row_hi, int aft_lo, int aft_hi) {
        TileSource t;
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const unsigned r = (unsigned)pos[Stage::row(i, tid) & (DKDV_QT - 1)];
            t.q[i].desc = hv.q.desc;
            t.g[i].desc = hv.g.desc;
            t.q_voff[SORTED ? i : 0] = __umul24(r, q_rs) + stQ.goff[i];
            t.g_voff[SORTED ? i : 0] = __umul24(r, g_rs) + stDO.goff[i];
        }
        t.small = hv.small.at((row_lo & from_lo) | (row_hi & from_hi) | (aft_lo & from_aft));
        const unsigned shift = (unsigned)((aft_hi - aft_lo - 32) * 4) & (unsigned)from_aft;
        t.small_voff = small < 2 ? 4u * (unsigned)pos[lane] : (unsigned)(lane * 4) + (shift & upper_lanes);
        return t;
    };
    // the 64-row tile made of the slices starting at rows row_lo (LDS rows 0..31) and row_hi (LDS rows 32..63)
    auto tile_source = [&](const HeadViews& hv, int row_lo, int row_hi) {
        TileSource t;
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int row = stQ.upper(i) ? row_hi : row_lo;
            t.q[i] = hv.q.at(row);
            t.g[i] = hv.g.at(row);
        }
        // lse / delta (small < 2): 32 floats of each slice.  Bitfields: 32 int64 = 64 dwords of slice lo
        // (small == 2) or hi (small == 3).  DENSE: the words of the slice this wave's row stream works on
        if (DENSE && small >= 2)
            t.small = hv.small.at((st ? row_hi : row_lo) >> 5);
        else
            t.small = hv.small.at(small == 3 ? row_hi : row_lo);
        const unsigned shift = (unsigned)((row_hi - row_lo - 32) * 4);
        t.pos_voff = (unsigned)(lane * 4) + (shift & upper_lanes);
        t.small_voff = small < 2 ? t.pos_voff : (unsigned)(lane * 4);
        if (IDX) t.pos = pos_rows.at(row_lo);
        return t;
    };
    // copy instruction j of a tile into buffer buf
    auto issue_copy = [&](int j, const TileSource& t, int buf, int pos_buf) {
        if (SORTED && j < CPT)
            stQ.template issue_gather<WAIT>(j, t.q[j].desc, t.q_voff[j], ldsQ + buf * TILE_BYTES);
        else if (SORTED && j < 2 * CPT)
            stDO.template issue_gather<WAIT>(j - CPT, t.g[j - CPT].desc, t.g_voff[j - CPT], ldsDO + buf * TILE_BYTES);
        else if (j < CPT)
            stQ.template issue_from<WAIT>(j, t.q[j], ldsQ + buf * TILE_BYTES);
        else if (j < 2 * CPT)
            stDO.template issue_from<WAIT>(j - CPT, t.g[j - CPT], ldsDO + buf * TILE_BYTES);
        else if (j == 2 * CPT)
            copy_b32<WAIT>(t.small, t.small_voff, ldsSmall + (SORTED ? (pos_buf & from_aft) | (buf & ~from_aft) : buf) * smallBytes);
        else  // 2 x 32 row positions; every wave writes the same values
            copy_b32<WAIT>(t.pos, t.pos_voff, lds_addr(sQpos) + pos_buf * (DKDV_QT * 4u));
    };

    // One 64-row tile held in buffer cur against this wave's 32 keys; the wave's 32 rows sit at sequence
    // rows myrow0.. and its class for them is cls.  The copies of the next tile into the other buffer
    // are issued one per MFMA of the S / dP phase, or back to back when this wave has nothing to compute.
    const int qr = 32 * st;  // this wave's rows inside the 64-row tile
    // The wave's flag class is extracted with a per-lane copy of the key group number on purpose: a branch
    // condition the compiler can prove wave-uniform makes it restructure the loop around that branch, and the
    // result needs far more registers than a wave has.
    const int kg_lane = (tid >> 6) & 3;
    // SAVE: where this lane's 32 bytes sit inside a 2 KiB block (key l32: 64 bytes, rows 4 hi + {0..3, 8..11, ...} first)
    const unsigned ds_lane_off = (unsigned)(kg * 2048 + l32 * 64 + hi * 32);
    // SAVE: the pairs (slice, this key tile) that have work are numbered consecutively from ds_base, by ascending slice,
    // i.e. in the order of the slice list: pair number = ds_base + position in the list
    int ds_base = 0;
    if (SAVE) ds_base = __builtin_amdgcn_readfirstlane(p.ds_tile_base[(int64_t)b * p.num_kt + nt]);
    // BIAS, per-key form (row stride 0): this lane's bias value for the head in work
    float bias_key = 0.f;
    int bias_head = -1;
    auto fetch_bias_key = [&](int h) {
        if (BIAS && p.bias_sm == 0 && h != bias_head) {
            bias_head = h;
            bias_key = kvalid ? load_bias1<T>(p.bias, (int64_t)b * p.bias_sb + (int64_t)h * p.bias_sh + key, p.bias_f32 != 0) : 0.f;
            asm volatile("" : "+v"(bias_key));  // arrives here, not at its first use between the tile copies
        }
    };
    // ds_pos: position of the wave's slice in the slice list.
    // returns true when the wave has issued its two dS stores (they may stay in flight over the end of the iteration)
    // pos_cur, pos_nxt: the buffers of the tile's positions and of those that are copied now
    auto tile_step = [&](int cur, int cls, int h_cur, int myrow0, int ds_pos, const TileSource& next, int nxt, int pos_cur, int pos_nxt) -> bool {
        if (cls == 0) {
#pragma unroll
            for (int j = 0; j < NLOADS; ++j) issue_copy(j, next, nxt, pos_nxt);
            return false;
        }
        const int ds_e = ds_base + ds_pos;
        const u32x4* tQ = sQ[cur];
        const u32x4* tG = sDO[cur];
        // ---- S = Q K^T and dP = dO V^T : 32 queries x 32 keys, two accumulator chains; both operands of
        // every MFMA come from LDS and are requested AHEAD MFMAs in front of their use
        // The V tile in LDS is NEGATED (see negate_v_tile), and the dP accumulator starts from delta instead of
        // zero: the chain then delivers delta - dO V^T = -(dP - delta) with no subtraction left for the VALU.
        // The sign is carried through dS into dK and taken back by the epilogue.
        f32x16 s, dp;
        {
            constexpr int NOP = 2 * KK, AHEAD = 3;  // MFMA j: S (j even) or dP (j odd), k-slice j / 2
            constexpr int FIRST = SORTED ? (NOP - NLOADS < 4 ? NOP - NLOADS : 4) : 0;  // the copies start behind MFMA FIRST - 1
            u32x4 a[NOP], bb[NOP];
            a[0] = lds_read_chunk<D>(tQ, qr + l32, hi);  // the operands of the first MFMA go first
            bb[0] = KV_REGS ? kfrag[0] : lds_read_chunk<D>(sK, 32 * kg + l32, hi);
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                const f32x4 d4 = *(const f32x4*)&sDelta[cur][qr + 8 * grp + 4 * hi];
#pragma unroll
                for (int x = 0; x < 4; ++x) dp[4 * grp + x] = d4[x];
            }
#pragma unroll
            for (int j = 1; j < AHEAD; ++j) {
                a[j] = lds_read_chunk<D>((j & 1) ? tG : tQ, qr + l32, 2 * (j >> 1) + hi);
                bb[j] = KV_REGS ? ((j & 1) ? vfrag[j >> 1] : kfrag[j >> 1])
                                : lds_read_chunk<D>((j & 1) ? sV : sK, 32 * kg + l32, 2 * (j >> 1) + hi);
            }
#pragma unroll
            for (int j = 0; j < NOP; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                if (j + AHEAD < NOP) {
                    a[j + AHEAD] = lds_read_chunk<D>(((j + AHEAD) & 1) ? tG : tQ, qr + l32, 2 * ((j + AHEAD) >> 1) + hi);
                    bb[j + AHEAD] = KV_REGS ? (((j + AHEAD) & 1) ? vfrag[(j + AHEAD) >> 1] : kfrag[(j + AHEAD) >> 1])
                                            : lds_read_chunk<D>(((j + AHEAD) & 1) ? sV : sK, 32 * kg + l32, 2 * ((j + AHEAD) >> 1) + hi);
                }
                if (j & 1)
                    dp = T::mfma(a[j], bb[j], dp);
                else
                    s = T::mfma(a[j], bb[j], j < 2 ? zero16 : s);
                if (j >= FIRST && j - FIRST < NLOADS) issue_copy(j - FIRST, next, nxt, pos_nxt);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- P = exp(scale s - lse) on allowed pairs, -dS/scale = P (delta - dP)   (the factor `-scale` of dS
        // is applied once to dK in the epilogue).  C fragment: register i <-> query row
        // 8*(i/4) + 4*hi + i%4 of this wave's 32 rows.
        if (BIAS && p.bias_sm == 0) {
            // the per-key ("vector") form: one value per key and head, fetched when the head changes
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = fmaf(s[i], p.scale, bias_key);
        } else if (BIAS) {
            // column `key` of the bias, one element per row of the C fragment
            const int64_t col = (int64_t)b * p.bias_sb + (int64_t)h_cur * p.bias_sh + key;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 8 * (i >> 2) + 4 * hi + (i & 3);
                const int row = SORTED ? sQpos[pos_cur][qr + r] : myrow0 + r;
                float bv = 0.f;
                if (kvalid && row < Sq) bv = load_bias1<T>(p.bias, col + (int64_t)row * p.bias_sm, p.bias_f32 != 0);
                s[i] = fmaf(s[i], p.scale, bv);
            }
        }
#pragma unroll
        for (int grp = 0; grp < 4; ++grp) {
            const f32x4 l4 = *(const f32x4*)&sLse[cur][qr + 8 * grp + 4 * hi];
#pragma unroll
            for (int x = 0; x < 4; ++x) s[4 * grp + x] = __builtin_amdgcn_exp2f(fmaf(s[4 * grp + x], c2, SCALED ? -l4[x] : l4[x] * -LOG2E));
        }
        if (DENSE) {
            if (cls == 1 && col_bits_on) {
                // (shifted by this lane's first row, 4 hi, once: the bit numbers tested are then constants)
                const unsigned w = sColBits[cur][st][32 * kg + l32] >> (4 * hi);
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = ((w >> (8 * (i >> 2) + (i & 3))) & 1u) ? s[i] : 0.f;
            } else if (cls == 1) {
                // mask bytes of this lane's key column, one per row of the C fragment
                const uint8_t* mcol = p.mask + ((int64_t)b * Sq + myrow0) * Sk + key;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int r = 8 * (i >> 2) + 4 * hi + (i & 3);
                    bool a = kvalid && myrow0 + r < Sq;
                    if (a && p.mask != nullptr) a = mcol[(int64_t)r * Sk] != 0;
                    s[i] = a ? s[i] : 0.f;
                }
            }
        } else if (cls == 1) {
            // Most partial tiles are partial only through causality: the 32 rows carry the same bitfield.
            // Then the bit test is a per-key constant and the rule reduces to one position compare.
            const int64_t mine = sQbf[cur][qr + l32];
            const unsigned mlo = (unsigned)mine, mhi = (unsigned)((uint64_t)mine >> 32);
            const unsigned flo = __builtin_amdgcn_readfirstlane(mlo), fhi = __builtin_amdgcn_readfirstlane(mhi);
            bool uniform = (mlo == flo) & (mhi == fhi);
            int qpos0 = myrow0;  // position of this wave's first row
            if (ROW_POS) {          // ... and the 32 rows must sit at consecutive positions
                const int rel0 = sQpos[pos_cur][qr + l32] - l32;
                qpos0 = __builtin_amdgcn_readfirstlane(rel0);
                uniform &= rel0 == qpos0;
            }
            if (__all(uniform)) {
                const QueryBits qu = make_query_bits(((int64_t)fhi << 32) | (int64_t)flo, 0);
                const bool ok = allow_bits(qu, klo, khi) & (qu.text | (qu.lim >= 0));
                // allowed iff krel <= 8 * grp + x  (text rows: key position <= row position)
                const int krel = !ok ? 0x7FFFFFFF : qu.text ? kpos - qpos0 - 4 * hi : (int)0x80000000;
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = (krel <= 8 * (i >> 2) + (i & 3)) ? s[i] : 0.f;
            } else {
                // rule constants of this wave's 32 rows, derived once per row (lane r < 32 takes row r) and
                // handed to all lanes through a wave-private LDS scratch
                {
                    const QueryBits qb = make_query_bits(mine, ROW_POS ? sQpos[pos_cur][qr + l32] : myrow0 + l32);
                    if (hi == 0) {
                        sWq[wave][0][l32] = qb.a_lo;
                        sWq[wave][1][l32] = qb.a_hi;
                        sWq[wave][2][l32] = qb.x_lo;
                        sWq[wave][3][l32] = qb.x_hi;
                        sWq[wave][4][l32] = (unsigned)qb.lim;
                    }
                }
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const int roff = 8 * grp + 4 * hi;
                    const u32x4 qalo = *(const u32x4*)&sWq[wave][0][roff];
                    const u32x4 qahi = *(const u32x4*)&sWq[wave][1][roff];
                    const u32x4 qxlo = *(const u32x4*)&sWq[wave][2][roff];
                    const u32x4 qxhi = *(const u32x4*)&sWq[wave][3][roff];
                    const u32x4 qlim = *(const u32x4*)&sWq[wave][4][roff];
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        QueryBits qb;
                        qb.a_lo = qalo[x];
                        qb.a_hi = qahi[x];
                        qb.x_lo = qxlo[x];
                        qb.x_hi = qxhi[x];
                        qb.lim = (int)qlim[x];
                        qb.text = qlim[x] < 0x7FFFFFFFu;  // text rows carry their position, modality rows INT_MAX or -1
                        s[4 * grp + x] = allow_pair(qb, klo, khi, kpos) ? s[4 * grp + x] : 0.f;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) dp[i] = s[i] * dp[i];  // -dS / scale
        u32x4 pb[2], dsb[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            pb[t] = pack8<T>(s, 8 * t);
            dsb[t] = pack8<T>(dp, 8 * t);
        }
        // ---- dV^T += dO^T P ; dK^T += Q^T dS -------------------------------------------------
        {
            u32x4 tg[2][DB], tq[2][DB];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    tg[t][db] = lds_read_transposed<D>(tG, lane, qr + 16 * t + 4 * hi, 32 * db + 16 * half16);
                    tq[t][db] = lds_read_transposed<D>(tQ, lane, qr + 16 * t + 4 * hi, 32 * db + 16 * half16);
                }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    dv[db] = T::mfma(tg[t][db], pb[t], dv[db]);
                    dk[db] = T::mfma(tq[t][db], dsb[t], dk[db]);
                }
            sched_pipeline_mfma_lds<4 * DB, 4, 2>();
        }
        if (SAVE) {
            // Issued after the MFMAs of the tile (in front of them they cost the kernel 2 % more).  Record number and
            // record address are wave-uniform (kept in scalar registers); the two 16-byte stores are inline asm so that
            // they take the scalar-base form and stay out of the compiler's load / store bookkeeping, like the tile
            // copies (the caller waits with explicit counts); non-temporal: the blocks are read once, by another
            // kernel, and should not push the Q / dO rows the other workgroups re-read out of L2
            const unsigned rec_no = (unsigned)__builtin_amdgcn_readfirstlane(h_cur * (int)p.ds_capacity + ds_e);
            const char* rec = (const char*)p.ds_ws + ((uint64_t)rec_no << 13);
            asm volatile("global_store_dwordx4 %0, %1, %3 nt\n\tglobal_store_dwordx4 %0, %2, %3 offset:16 nt"
                         :
                         : "v"(ds_lane_off), "v"(dsb[0]), "v"(dsb[1]), "s"(rec)
                         : "memory");
        }
        return SAVE;
    };

    // Sequences of more than MAX_SLICE_LIST slices are walked in several passes, from the end, each with a list
    // of its own; dK and dV live in registers and simply carry over.
    for (int s_end = ns_total;;) {
        lds_barrier();
        const int n = sCount;
        // Main loop: the listed slices are taken in pairs from the END of the list (the workgroups of one kv head
        // that are resident together then read the same Q / dO rows at about the same time, and all but the first
        // of them find them in L2); pair r = entries n - 2 - 2 r (row stream 0) and n - 1 - 2 r (row stream 1).
        // An odd count leaves the first entry alone: its pair repeats it with all classes cleared for stream 0.
        // The q heads of the group follow one another: tile t = (head t / npairs, pair t % npairs).
        const int npairs = (n + 1) >> 1;
        const int total = npairs * G;
        if (total > 0) {
            auto entry_hi = [&](int r) { return sList[n - 1 - 2 * r]; };
            auto entry_lo = [&](int r) { return sList[n - 2 - 2 * r]; };  // entry -1 where the count is odd
            // current tile (g_cur, entries e_*), next tile (g_nxt, r_nxt, entries n_*, head views hv_nxt); past the
            // last tile "next" keeps walking through pairs of the last head, whose copies nobody reads
            int g_cur = 0, g_nxt = 0, r_nxt = 0, r_cur = 0;
            HeadViews hv_nxt = head_views(hk * G);
            int e_lo = __builtin_amdgcn_readfirstlane(entry_lo(0)), e_hi = __builtin_amdgcn_readfirstlane(entry_hi(0));
            int a_lo = 0, a_hi = 0;  // SORTED: the entries of the tile after next
            auto after = [&](int r) { return r + 1 == npairs ? 0 : r + 1; };
            if constexpr (!SORTED) {
                const TileSource first = tile_source(hv_nxt, (e_lo >> 8) * 32, (e_hi >> 8) * 32);
#pragma unroll
                for (int j = 0; j < NLOADS; ++j) issue_copy(j, first, 0, 0);
            } else {  // the row numbers of the first two tiles, then the first tile
                const int r1 = after(0);
                const int lo1 = (__builtin_amdgcn_readfirstlane(entry_lo(r1)) >> 8) * 32, hi1 = (__builtin_amdgcn_readfirstlane(entry_hi(r1)) >> 8) * 32;
                if (small == 4) {
                    TileSource numbers;
                    numbers_of(numbers, hv_nxt, (e_lo >> 8) * 32, (e_hi >> 8) * 32);
                    issue_copy(2 * CPT, numbers, 0, 0);
                }
                wait_async();
                __syncthreads();
                const TileSource first = gathered_source(hv_nxt, sQpos[0], (e_lo >> 8) * 32, (e_hi >> 8) * 32, lo1, hi1);
#pragma unroll
                for (int j = 0; j < NLOADS; ++j) issue_copy(j, first, 0, 1);
                a_lo = __builtin_amdgcn_readfirstlane(entry_lo(after(r1)));
                a_hi = __builtin_amdgcn_readfirstlane(entry_hi(after(r1)));
            }
            auto advance = [&]() {
                if (++r_nxt == npairs) {
                    r_nxt = 0;
                    if (++g_nxt < G) next_head(hv_nxt);
                }
            };
            advance();
            int n_lo = __builtin_amdgcn_readfirstlane(entry_lo(r_nxt)), n_hi = __builtin_amdgcn_readfirstlane(entry_hi(r_nxt));
            // DEEP: two tiles are copied ahead, f_* is the one between the current tile and the one that is copied
            int f_lo = n_lo, f_hi = n_hi, f_g = g_nxt, f_r = r_nxt;
            if constexpr (DEEP) {
                const TileSource second = tile_source(hv_nxt, (n_lo >> 8) * 32, (n_hi >> 8) * 32);
#pragma unroll
                for (int j = 0; j < NLOADS; ++j) issue_copy(j, second, 1, 1);
                advance();
                n_lo = __builtin_amdgcn_readfirstlane(entry_lo(r_nxt));
                n_hi = __builtin_amdgcn_readfirstlane(entry_hi(r_nxt));
            }
            wait_async();
            asm volatile("" : "+v"(klo), "+v"(khi), "+v"(kpos));  // (see arrived())
            __syncthreads();
            if (!v_negated) {  // K, V and the first tile have landed
                negate_v_tile();
                v_negated = true;
                __syncthreads();
            }
            load_kv_operands();
            int pos_cur = 0;  // SORTED: it % 3
            for (int it = 0; it < total; ++it) {
                const int cur = it & (NB - 1), nxt = DEEP ? (it + 2) & (NB - 1) : cur ^ 1;
                // pair after next (SORTED: the one behind it): its list entries are requested now and picked up at the end of
                // the iteration
                const int r_req = SORTED ? after(after(r_nxt)) : after(r_nxt);
                const int x_lo = entry_lo(r_req), x_hi = entry_hi(r_req);
                TileSource next;
                const int p1 = SORTED ? (pos_cur == 2 ? 0 : pos_cur + 1) : nxt, p2 = SORTED ? (pos_cur == 0 ? 2 : pos_cur - 1) : nxt;
                if constexpr (SORTED) {
                    next = gathered_source(hv_nxt, sQpos[p1], (n_lo >> 8) * 32, (n_hi >> 8) * 32, (a_lo >> 8) * 32, (a_hi >> 8) * 32);
                } else {
                    next = tile_source(hv_nxt, (n_lo >> 8) * 32, (n_hi >> 8) * 32);
                }
                const int mine = st ? e_hi : e_lo;
                fetch_bias_key(hk * G + g_cur);
                const bool stored = tile_step(cur, (mine >> (2 * kg_lane)) & 3, hk * G + g_cur, (mine >> 8) * 32, n - 2 - 2 * r_cur + st,
                                              next, nxt, SORTED ? pos_cur : cur, p2);
                g_cur = DEEP ? f_g : g_nxt;
                r_cur = DEEP ? f_r : r_nxt;
                e_lo = DEEP ? f_lo : n_lo;
                e_hi = DEEP ? f_hi : n_hi;
                if (DEEP) {
                    f_lo = n_lo;
                    f_hi = n_hi;
                    f_g = g_nxt;
                    f_r = r_nxt;
                }
                advance();
                n_lo = SORTED ? a_lo : __builtin_amdgcn_readfirstlane(x_lo);
                n_hi = SORTED ? a_hi : __builtin_amdgcn_readfirstlane(x_hi);
                if (SORTED) {
                    a_lo = __builtin_amdgcn_readfirstlane(x_lo);
                    a_hi = __builtin_amdgcn_readfirstlane(x_hi);
                    pos_cur = p1;
                }
                // DEEP: after every second tile the next two have landed and their buffers are free again
                if (DEEP && (it & 1) == 0) continue;
                // the copies of the next tile must have landed; the two dS stores, issued after them, may stay in flight
                if (SAVE && stored)
                    asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
                else
                    wait_async();
                __syncthreads();
            }
        }
        if (!LONG) break;
        s_end = max(0, s_end - MAX_SLICE_LIST);
        if (s_end == 0) break;
        __syncthreads();  // everybody has read the list of the pass that just ended
        if (wave == 0) {
            const int s_begin = max(0, s_end - MAX_SLICE_LIST);
            build_slice_list(p, b, nt, lane, s_begin, s_end, load_slice_classes(p, b, nt, s_begin + lane, s_end), sList, &sCount);
        }
    }
    // every copy has landed and every wave is done with the tiles: the epilogue reuses the tile arrays
    wait_async();
    __syncthreads();

    // ---- epilogue.  The two waves of a key group hold partial sums of dK and dV.  The K, V, Q and dO tiles are dead now: through
    // tile array number kg (exactly the right size) the row stream 0 wave hands its dV over and the stream 1 wave its dK; then
    // the one finishes dK, the other dV.  This workgroup is the sole owner of these rows.
    f32x4* const park = (f32x4*)(kg == 0 ? sK : kg == 1 ? sV : kg == 2 ? &sQ[0][0] : &sDO[0][0]);
    auto hand_over = [&](const f32x16 (&acc)[DB], int half) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp)
                park[((half * DB + db) * 4 + grp) * 64 + lane] =
                    f32x4{acc[db][4 * grp], acc[db][4 * grp + 1], acc[db][4 * grp + 2], acc[db][4 * grp + 3]};
    };
    auto finish = [&](const f32x16 (&acc)[DB], int half, float factor, const Tensor4& t) {
        const int64_t at = (int64_t)b * t.sb + (int64_t)key * t.ss + (int64_t)hk * t.sh;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            f32x16 x = acc[db];
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                const f32x4 other = park[((half * DB + db) * 4 + grp) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) x[4 * grp + i] = (x[4 * grp + i] + other[i]) * factor;
            }
            if (p.grad_typed == 1) {  // overwrite mode: the input dtype
                store_block16<T>((char*)t.ptr + 2 * (at + 32 * db), p.d - 32 * db, hi, [&](int i) { return x[i]; });
                continue;
            }
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                if (32 * db + 8 * grp >= p.d) break;
                f32x4* dst = (f32x4*)((float*)t.ptr + at + 32 * db + 8 * grp + 4 * hi);
                const f32x4 y = {x[4 * grp], x[4 * grp + 1], x[4 * grp + 2], x[4 * grp + 3]};
                *dst = PARTS && p.grad_typed == 2 ? y : *dst + y;
            }
        }
    };
    if (st == 0)
        hand_over(dv, 1);
    else
        hand_over(dk, 0);
    __syncthreads();
    if (!kvalid) return;
    if (st == 0)
        finish(dk, 0, -p.scale, p.dk);  // (dk holds -dK / scale)
    else
        finish(dv, 1, 1.f, p.dv);
}

// ---------------------------------------------------------------------------------------
// dQ.  Same decomposition and S^T layout as the forward kernel: a lane owns one query, so
// lse and delta are per-lane scalars; dS^T feeds dQ^T = K^T dS^T from registers and K^T comes
// from the transposing LDS read of the K tile that also serves S^T = K Q^T.
constexpr int DQ_KT = 64;
constexpr int DQ_THREADS = 256;

// Forms of a bias: read from global memory group by group, or (one row of keys, its groups of four aligned) copied with the
// tiles.  The second takes a wave per SIMD of the head dims up to 64 (26 spilled registers otherwise), the first keeps it.  As
// one kernel with two waves the matrix form lost and both paid for the choice in the loop; dQ, 2 x 2048 tokens, 16 heads, bf16,
// one kernel -> two: matrix D 32 104.6 -> 96.6 us, D 64 108.0 -> 108.0, fp32 matrix D 32 92.8 -> 85.6, D 64 99.0 -> 97.1; one
// row of keys D 32 47.2 -> 43.1, D 64 59.9 -> 57.0; 2047 tokens (unaligned rows) D 32 88.8 -> 81.9, D 64 104.6 -> 103.1.
constexpr int BIAS_NONE = 0, BIAS_READ = 1, BIAS_TILES = 2;

// LONG: as in the dK/dV kernel, for more than MAX_LIST 64-key tiles.
// STREAMS: as in the forward.
template <typename T, int D, int MODE, int BIAS_FORM, bool LONG, int STREAMS>
__global__ __launch_bounds__(DQ_THREADS * STREAMS, D > 64 || BIAS_FORM == BIAS_TILES || STREAMS > 1 ? 2 : 3) void bwd_dq_kernel(const AttnParams p) {
    static_assert(STREAMS == 1 || !LONG, "streams and passes are not combined");
    constexpr bool BIAS = BIAS_FORM != BIAS_NONE, bias_lds = BIAS_FORM == BIAS_TILES;
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = MODE == MASK_DENSE;
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    __shared__ u32x4 sK_all[STREAMS][2][DQ_KT * NCH];
    __shared__ u32x4 sV_all[STREAMS][2][DQ_KT * NCH];
    __shared__ __attribute__((aligned(16))) int64_t sKbf_all[STREAMS][2][DQ_KT];  // raw bitfields of the tile's keys
    __shared__ __attribute__((aligned(16))) int sKpos_all[STREAMS][2][DQ_KT];     // their global positions (IDX only)
    __shared__ int sList[MAX_LIST];
    __shared__ int sCount[STREAMS];
    // DENSE with packed mask bits: per wave, the words of its 32 rows for the tile's two 32-key blocks
    __shared__ unsigned sRowBits_all[STREAMS][DENSE ? 2 : 1][4][DENSE ? 64 : 1];
    // BIAS in its per-key form: the 64 values of the tile (raw words; 16-bit elements fill half)
    __shared__ __attribute__((aligned(16))) unsigned sBias_all[STREAMS][bias_lds ? 2 : 1][bias_lds ? 64 : 1];

    // (tid and wave: inside the stream)
    const int tid = threadIdx.x % DQ_THREADS, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int stream = STREAMS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / DQ_THREADS) : 0;
    auto &sK = sK_all[stream], &sV = sV_all[stream];
    auto& sKbf = sKbf_all[stream];
    auto& sKpos = sKpos_all[stream];
    auto& sRowBits = sRowBits_all[stream];
    auto& sBias = sBias_all[stream];
    const int hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
    const int wave_lane = tid >> 6;
    const int Sq = p.Sq, Sk = p.Sk;
    const int G = p.Hq / p.Hkv;

    int ub, hk, g;
    head_unit_map(blockIdx.x, p.num_m * p.B, p.Hkv, G, ub, hk, g);
    constexpr bool MAY_SIDE = STREAMS > 1 && D > 32;
    int code = 0;
    bool side = false, idle = false;  // the streams take a unit each; ... and there is none left for this one
    if constexpr (MAY_SIDE) {
        if (p.group_order != nullptr) code = plan_word(p.group_order + ub);
        side = streams_side_by_side(p);
        if (__builtin_expect(side, 0)) {
            const int units = p.num_m * p.B * p.Hq, unit = side_unit(blockIdx.x, stream);
            if (side_unit(blockIdx.x, 0) >= units) return;
            idle = unit >= units;
            head_unit_map(idle ? 0 : unit, p.num_m * p.B, p.Hkv, G, ub, hk, g);
            code = plan_word(p.group_order + ub);
        }
    }
    int b = ub % p.B, grp = ub / p.B;
    if (p.group_order != nullptr) {  // with a plan: the groups of all sequences by falling length of their tile lists
        if constexpr (!MAY_SIDE) code = p.group_order[ub];
        b = code / p.num_m;
        grp = code - b * p.num_m;
    }
    const int h = hk * G + g;
    const WaveSlices ws = pick_wave_slices<!BIAS>(p, b, grp);  // group 0 is the heaviest

    const int slice = idle ? -1 : __builtin_amdgcn_readfirstlane(wave == 0 ? ws.slice[0] : wave == 1 ? ws.slice[1] : wave == 2 ? ws.slice[2] : ws.slice[3]);
    const int slot = (slice < 0 ? 0 : slice) * 32 + l32;
    const bool qvalid = slice >= 0 && slot < Sq;
    const int qrow = row_of_slot(p, ws, b, slot, qvalid);
    // (the class bytes are asked for ahead of the rows: loads arrive in order)
    const bool lists = wave == 0 && (stream == 0 || side);
    const int list_keys = idle ? 0 : Sk;
    TileClasses first_classes = {};
    if (lists) first_classes = load_tile_classes(ws, p.num_n, key_tiles(list_keys, 0), lane);
    u32x4 qreg[KK], greg[KK];
    {
        const char* qp = (const char*)p.q.ptr + 2 * ((int64_t)b * p.q.sb + (int64_t)qrow * p.q.ss + (int64_t)h * p.q.sh);
        const char* gp = (const char*)p.dout.ptr + 2 * ((int64_t)b * p.dout.sb + (int64_t)qrow * p.dout.ss + (int64_t)h * p.dout.sh);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            u32x4 zq = {0u, 0u, 0u, 0u}, zg = {0u, 0u, 0u, 0u};
            if (qvalid && 16 * kk + 8 * hi < p.d) {
                zq = *(const u32x4*)(qp + (16 * kk + 8 * hi) * 2);
                zg = *(const u32x4*)(gp + (16 * kk + 8 * hi) * 2);
            }
            qreg[kk] = zq;
            greg[kk] = zg;
        }
    }
    const int64_t qf = (!DENSE && qvalid) ? p.bfq[(int64_t)b * p.bfq_sb + qrow] : 0;
    float lse_row = 0.f, dlt = 0.f;
    if (qvalid) {
        const int64_t off = (int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded + qrow;
        lse_row = p.lse[off];
        if (D > 64 || p.o.ptr == nullptr) dlt = p.delta[off];
    }
    u32x4 oreg[D <= 64 ? KK : 1];
    const bool sums_delta = D <= 64 && p.o.ptr != nullptr;
    if (sums_delta) {
        const char* op = (const char*)p.o.ptr + 2 * ((int64_t)b * p.o.sb + (int64_t)qrow * p.o.ss + (int64_t)h * p.o.sh);
#pragma unroll
        for (int kk = 0; kk < (D <= 64 ? KK : 1); ++kk) {
            u32x4 zo = {0u, 0u, 0u, 0u};
            if (qvalid && 16 * kk + 8 * hi < p.d) zo = *(const u32x4*)(op + (16 * kk + 8 * hi) * 2);
            oreg[kk] = zo;
        }
    }
    const int qpos = (IDX && qvalid) ? p.posq[qrow] : qrow;
    // (the row loads above are in flight while wave 0 reads the class rows and the first tile is on its way)
    if (lists)  // first pass (usually the only one)
        build_key_tile_list<STREAMS>(ws, p.num_n, list_keys, lane, 0, first_classes, sList + stream * (MAX_LIST / 2), sCount + stream, !side);
    QueryBits qb = {};
    float lse2 = INFINITY;
    // With o given, this launch also is the delta pre-pass: it runs in front of the dK/dV kernel, has the rows of dO in
    // registers and covers every row once; a launch and a second reading of dO less (2 x 283 tokens: 3.4 us; 8 x 4096
    // tokens, 16 heads, D 64: 25 us for reading both).  Sums as the pre-pass does: chunk pairs, then the two half waves.
    auto rows_arrived = [&]() {
        arrived(qreg);
        arrived(greg);
        if (sums_delta) {
            float part[KK];
#pragma unroll
            for (int kk = 0; kk < (D <= 64 ? KK : 1); ++kk) part[kk] = chunk_dot<T>(oreg[kk], greg[kk]);
            dlt = half_swap_sum(KK == 4 ? (part[0] + part[2]) + (part[1] + part[KK - 1]) : part[0] + part[1]);
            if ((stream == 0 || side) && qvalid && hi == 0) {
                const int64_t at = (int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded + qrow;
                p.delta[at] = dlt;
                if (p.lse_scaled != nullptr) p.lse_scaled[at] = lse_row * LOG2E;
            }
        }
        qb = make_query_bits(qf, qpos);
        lse2 = (!qvalid || lse_row == -INFINITY) ? INFINITY : lse_row * LOG2E;
    };

    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dq[db][i] = 0.f;
    f32x16 zero16;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero16[i] = 0.f;
    // A per-key bias whose groups of four keys are aligned, in-range accesses travels with the tile copies, and with bf16
    // operands it is added by one more MFMA of the S phase, as in the forward.  (Read from global memory inside the loop,
    // every group of four waited, through the in-order vmcnt, for all tile copies in flight: 2 x 2048 tokens, 16 heads,
    // D 64: 75 us, now 63.)
    constexpr bool bias_fold = bias_lds && std::is_same<T, BF16>::value;
    const float c2 = (BIAS && !bias_fold) ? LOG2E : p.scale * LOG2E;  // otherwise the scores become scale * s + bias first
    const float inv_scale = 1.f / p.scale;
    const char* bias_row = nullptr;  // this lane's row of the bias
    if (BIAS)
        bias_row = (const char*)p.bias + (p.bias_f32 ? 4 : 2) * ((int64_t)b * p.bias_sb + (int64_t)h * p.bias_sh +
                                                                (int64_t)(qvalid ? qrow : 0) * p.bias_sm);

    RowView<LONG> k_rows, v_rows;
    RowView<false> bf_rows, pos_rows, bias_rows;  // key bitfields, (IDX) positions, per-key bias
    k_rows.init((const char*)p.k.ptr + 2 * ((int64_t)b * p.k.sb + (int64_t)hk * p.k.sh), 2 * p.k.ss, Sk, 2 * p.d);
    v_rows.init((const char*)p.v.ptr + 2 * ((int64_t)b * p.v.sb + (int64_t)hk * p.v.sh), 2 * p.v.ss, Sk, 2 * p.d);
    if (!DENSE) bf_rows.init(p.bfk + (int64_t)b * p.bfk_sb, 8, Sk, 8);
    if (IDX) pos_rows.init(p.posk, 4, Sk, 4);

    typedef TileStage<D, DQ_KT, DQ_THREADS, true> Stage;
    constexpr int CPT = Stage::CPT;
    // copy instructions per wave and tile: K, V, the key bitfields, (IDX) the key positions and (BIAS_TILES) the bias values
    constexpr int NLOADS = 2 * CPT + 1 + (IDX ? 1 : 0) + (bias_lds ? 1 : 0);
    static_assert(NLOADS <= 2 * KK + 1, "one copy per MFMA of the first S / dP block (and at most one behind it)");
    Stage stK;
    TileStage<D, DQ_KT, DQ_THREADS> stV;
    stK.setup(2 * p.k.ss, p.d / 8, tid);
    stV.setup(2 * p.v.ss, p.d / 8, tid);
    const unsigned ldsK = lds_addr(sK), ldsV = lds_addr(sV), ldsB = lds_addr(sKbf), ldsP = lds_addr(sKpos);
    const unsigned ldsR = lds_addr(sRowBits);
    // DENSE: the packed mask rows of this wave's slice (null: no plan, the mask bytes are read instead)
    const unsigned* row_bits_w = (DENSE && p.row_bits != nullptr)
                                     ? p.row_bits + (int64_t)b * p.row_bits_sb + (slice < 0 ? 0 : slice) * 32
                                     : nullptr;
    const unsigned row_bits_voff = DENSE ? (unsigned)(hi * (int)p.row_bits_sn * 4 + l32 * 4) : 0u;
    if (bias_lds) {
        const int esz = p.bias_f32 ? 4 : 2;
        bias_rows.init((const char*)p.bias + esz * ((int64_t)b * p.bias_sb + (int64_t)h * p.bias_sh), esz, Sk, esz);
    }
    const unsigned bias_voff = (unsigned)((p.bias_f32 ? lane : (lane & 31)) * 4);
    constexpr unsigned TILE_BYTES = DQ_KT * NCH * 16, BITS_BYTES = DQ_KT * 8;
    // copy instruction j of tile kt into buffer buf (key bitfields: 64 dwords per wave, waves 2, 3
    // repeat what waves 0, 1 write, so that every wave issues the same number of copies)
    auto issue_copy = [&](int j, int kt, int buf) {
        const int row = kt * DQ_KT;
        if (j < CPT)
            stK.template issue<WAIT>(j, k_rows.at(row), ldsK + buf * TILE_BYTES);
        else if (j < 2 * CPT)
            stV.template issue<WAIT>(j - CPT, v_rows.at(row), ldsV + buf * TILE_BYTES);
        else if (j == 2 * CPT) {
            if (DENSE) {  // lanes 0..31: block 2 kt, lanes 32..63: block 2 kt + 1, rows of this wave's slice
                if (row_bits_w != nullptr)
                    dma_b32(row_bits_w + (int64_t)(2 * kt) * p.row_bits_sn, row_bits_voff, ldsR + (unsigned)(buf * 4 + wave) * 256u);
            } else {
                copy_b32<WAIT>(bf_rows.at(row), (unsigned)((wave & 1) * 256 + lane * 4), ldsB + buf * BITS_BYTES + (wave & 1) * 256u);
            }
        }
        else if (IDX && j == 2 * CPT + 1)  // 64 positions; every wave writes the same values
            copy_b32<WAIT>(pos_rows.at(row), (unsigned)(lane * 4), ldsP + buf * (DQ_KT * 4u));
        else if (bias_lds)  // BIAS: the tile's 64 bias values; every wave writes the same values
            copy_b32<WAIT>(bias_rows.at(row), bias_voff, lds_addr(sBias) + buf * 256u);
    };

    // One 64-key tile held in buffer `cur`; the copies of tile kt_next into the other buffer
    // are issued one per MFMA of the first S / dP block.
    auto tile_step = [&](int cur, int entry, int kt_next) {
        // (the class is extracted with a per-lane copy of the wave number on purpose: a skip branch the compiler
        // can prove wave-uniform makes it restructure the loop around it at the price of ~90 spilled registers)
        const int kt = entry >> 8, cls = (entry >> (2 * wave_lane)) & 3;
        if (cls == 0) {  // nothing for this wave's slice in the tile: only keep the copies of the next one going
#pragma unroll
            for (int j = 0; j < NLOADS; ++j) issue_copy(j, kt_next, cur ^ 1);
            return;
        }
        const u32x4* tK = sK[cur];
        const u32x4* tV = sV[cur];
        // partial tile whose 64 keys all carry the same bitfield: the rule is one position compare
        bool uniform_keys = false;
        int rel = 0;
        if (!DENSE && cls == 1) {
            const int64_t mine = sKbf[cur][lane];
            const unsigned mlo = (unsigned)mine, mhi = (unsigned)((uint64_t)mine >> 32);
            const unsigned flo = __builtin_amdgcn_readfirstlane(mlo), fhi = __builtin_amdgcn_readfirstlane(mhi);
            bool uniform = (mlo == flo) & (mhi == fhi);
            int kt0 = kt * DQ_KT;  // position of the tile's first key
            if (IDX) {             // ... and the 64 keys must sit at consecutive positions
                const int rel0 = sKpos[cur][lane] - lane;
                kt0 = __builtin_amdgcn_readfirstlane(rel0);
                uniform &= rel0 == kt0;
            }
            uniform_keys = __all(uniform);
            // last allowed key, relative to the first key this lane holds (4 hi): what it is compared with are then
            // compile-time constants, which occupy no registers
            rel = allow_bits(qb, flo, fhi) ? qb.lim - kt0 - 4 * hi : -1;
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            // ---- S^T = K Q^T and dP^T = V dO^T : 32 keys x 32 queries, two accumulator chains
            f32x16 s, dp;
            u32x4 bias_a = {0u, 0u, 0u, 0u};  // bias_fold: this lane's key of the block, as an operand
            if (BIAS && bias_fold && hi == 0) {
                const float bv = p.bias_f32 ? ((const float*)sBias[cur])[32 * kb + l32]
                                            : T::to_float(((const unsigned short*)sBias[cur])[32 * kb + l32]);
                bias_a = split3_operand<T>(bv * inv_scale);
            }
            {
                constexpr int NOP = 2 * KK, AHEAD = 4;  // operand j: K chunk (j even) or V chunk (j odd) of k-slice j / 2
                u32x4 a[NOP];
#pragma unroll
                for (int j = 0; j < AHEAD; ++j) a[j] = lds_read_chunk<D>((j & 1) ? tV : tK, 32 * kb + l32, 2 * (j >> 1) + hi);
#pragma unroll
                for (int j = 0; j < NOP; ++j) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (j + AHEAD < NOP)
                        a[j + AHEAD] = lds_read_chunk<D>(((j + AHEAD) & 1) ? tV : tK, 32 * kb + l32, 2 * ((j + AHEAD) >> 1) + hi);
                    if (j & 1)
                        dp = T::mfma(a[j], greg[j >> 1], j < 2 ? zero16 : dp);
                    else
                        s = T::mfma(a[j], qreg[j >> 1], j < 2 ? zero16 : s);
                    if (kb == 0 && j < NLOADS) issue_copy(j, kt_next, cur ^ 1);
                }
                if (kb == 0) {
#pragma unroll
                    for (int j = NOP; j < NLOADS; ++j) issue_copy(j, kt_next, cur ^ 1);
                }
                if (BIAS && bias_fold) {
                    const u32x4 z = {0u, 0u, 0u, 0u};
                    s = T::mfma(bias_a, hi == 0 ? ones3_operand<T>() : z, s);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (BIAS && bias_fold) {
                // (added by the MFMA above)
            } else if (BIAS && bias_lds) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const int koff = 32 * kb + 8 * grp + 4 * hi;
                    f32x4 b4;
                    if (p.bias_f32) {
                        b4 = *(const f32x4*)&sBias[cur][koff];
                    } else {
                        const u32x2 w = *(const u32x2*)((const char*)sBias[cur] + 2 * koff);
                        b4[0] = T::to_float((unsigned short)(w[0] & 0xFFFFu));
                        b4[1] = T::to_float((unsigned short)(w[0] >> 16));
                        b4[2] = T::to_float((unsigned short)(w[1] & 0xFFFFu));
                        b4[3] = T::to_float((unsigned short)(w[1] >> 16));
                    }
#pragma unroll
                    for (int x = 0; x < 4; ++x) s[4 * grp + x] = fmaf(s[4 * grp + x], p.scale, b4[x]);
                }
            } else if (BIAS) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const f32x4 b4 = load_bias4<T>(bias_row, kt * DQ_KT + 32 * kb + 8 * grp + 4 * hi, Sk, p.bias_f32 != 0, p.bias_vec != 0);
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        s[4 * grp + x] = bias_fold ? fmaf(b4[x], inv_scale, s[4 * grp + x])  // (c2 holds the scale)
                                                   : fmaf(s[4 * grp + x], p.scale, b4[x]);
                }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float e = __builtin_amdgcn_exp2f(fmaf(s[i], c2, -lse2));
                dp[i] = e * (dp[i] - dlt);  // the factor `scale` of dS is applied to dQ in the epilogue
            }
            if (DENSE) {
                if (cls == 1 && row_bits_w != nullptr) {
                    // (shifted by this lane's first key, 4 hi, once: the bit numbers tested are then constants)
                    const unsigned w = sRowBits[cur][wave][32 * kb + l32] >> (4 * hi);
#pragma unroll
                    for (int i = 0; i < 16; ++i) dp[i] = ((w >> (8 * (i >> 2) + (i & 3))) & 1u) ? dp[i] : 0.f;
                } else if (cls == 1) {
                    const int kt0 = kt * DQ_KT;
                    const uint8_t* mrow = p.mask + ((int64_t)b * Sq + (qvalid ? qrow : 0)) * Sk + kt0;
                    const bool dwords = (Sk & 3) == 0;  // rows start 4-byte aligned
#pragma unroll
                    for (int grp = 0; grp < 4; ++grp) {
                        const int koff = 32 * kb + 8 * grp + 4 * hi;
                        unsigned m4 = 0;
                        if (p.mask == nullptr) {
                            m4 = 0x01010101u;
                        } else if (qvalid) {
                            if (dwords) {
                                if (kt0 + koff < Sk) m4 = *(const unsigned*)(mrow + koff);
                            } else {
#pragma unroll
                                for (int x = 0; x < 4; ++x)
                                    if (kt0 + koff + x < Sk) m4 |= (unsigned)mrow[koff + x] << (8 * x);
                            }
                        }
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            const bool a = ((m4 >> (8 * x)) & 0xFFu) != 0 && kt0 + koff + x < Sk;
                            dp[4 * grp + x] = a ? dp[4 * grp + x] : 0.f;
                        }
                    }
                }
            } else if (cls == 1) {
                if (uniform_keys) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) dp[i] = (32 * kb + 8 * (i >> 2) + (i & 3) <= rel) ? dp[i] : 0.f;
                } else {
                    // natural positions: the row's limit relative to the first key this lane holds
                    const int lim_rel = qb.lim - (kt * DQ_KT + 4 * hi);
#pragma unroll
                    for (int grp = 0; grp < 4; ++grp) {
                        const int koff = 32 * kb + 8 * grp + 4 * hi;
                        const u32x4 k01 = *(const u32x4*)&sKbf[cur][koff];      // lo0 hi0 lo1 hi1
                        const u32x4 k23 = *(const u32x4*)&sKbf[cur][koff + 2];  // lo2 hi2 lo3 hi3
                        const unsigned klo[4] = {k01[0], k01[2], k23[0], k23[2]};
                        const unsigned khi[4] = {k01[1], k01[3], k23[1], k23[3]};
                        u32x4 kp = {0u, 0u, 0u, 0u};
                        if (IDX) kp = *(const u32x4*)&sKpos[cur][koff];
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            const bool pos_ok = IDX ? (int)kp[x] <= qb.lim : 32 * kb + 8 * grp + x <= lim_rel;
                            dp[4 * grp + x] = (allow_bits(qb, klo[x], khi[x]) & pos_ok) ? dp[4 * grp + x] : 0.f;
                        }
                    }
                }
            }
            u32x4 dsb[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) dsb[t] = pack8<T>(dp, 8 * t);
            // ---- dQ^T += K^T dS^T
            {
                u32x4 ta[2][DB];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int db = 0; db < DB; ++db)
                        ta[t][db] = lds_read_transposed<D>(tK, lane, 32 * kb + 16 * t + 4 * hi, 32 * db + 16 * half16);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int db = 0; db < DB; ++db) dq[db] = T::mfma(ta[t][db], dsb[t], dq[db]);
                sched_pipeline_mfma_lds<2 * DB, 2, 2>();
            }
        }
    };

    // Sequences of more than MAX_LIST 64-key tiles are walked in several passes, each with a list of its own.
    const int nkt_total = (Sk + DQ_KT - 1) / DQ_KT;
    for (int kt_begin = 0;;) {
        lds_barrier();
        // (two streams: the even and the odd tiles, as in the forward)
        const int n = sCount[stream], rounds = STREAMS > 1 ? max(n, sCount[STREAMS - 1 - stream]) : n;
        const int* const list = sList + stream * (MAX_LIST / 2);
        auto list_at = [&](int i) {
            if (STREAMS == 1) return list[i < n ? i : n - 1];
            const int e = list[i < n ? i : max(n - 1, 0)];
            return i < n ? e : n > 0 ? e & ~0xFF : 0;
        };
        int entry = 0, next = 0;
        if (rounds > 0) {
            entry = __builtin_amdgcn_readfirstlane(list_at(0));
            next = __builtin_amdgcn_readfirstlane(list_at(1));
    #pragma unroll
            for (int j = 0; j < NLOADS; ++j) issue_copy(j, entry >> 8, 0);
        }
        if (!LONG || kt_begin == 0) rows_arrived();  // (also where there is no tile: somebody needs delta)
        if (rounds > 0) {
            wait_async();
            __syncthreads();
            for (int it = 0; it < rounds; ++it) {
                const int cur = it & 1;
                // entry after next, requested now and picked up at the end of the iteration
                const int after = list_at(it + 2);
                tile_step(cur, entry, next >> 8);
                entry = next;
                next = __builtin_amdgcn_readfirstlane(after);
                wait_async();
                __syncthreads();
            }
        }
        if (!LONG) break;
        kt_begin += MAX_LIST;
        if (kt_begin >= nkt_total) break;
        __syncthreads();  // everybody has read the list of the pass that just ended
        if (wave == 0) build_key_tile_list(ws, p.num_n, Sk, lane, kt_begin, load_tile_classes(ws, p.num_n, key_tiles(Sk, kt_begin), kt_begin + lane), sList, sCount);
    }

    // Two streams: each hands over the columns that the other one finishes, through the tile arrays, which nobody reads any more.
    constexpr int DB0 = STREAMS > 1 ? (DB + 1) / 2 : DB;
    f32x4* const park = (f32x4*)sK_all + wave * (DB * 4 * 64);
    const bool merged = STREAMS > 1 && !side;
    if (merged) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
            if ((db < DB0) == (stream == 1)) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp)
                    park[(4 * db + grp) * 64 + lane] = f32x4{dq[db][4 * grp], dq[db][4 * grp + 1], dq[db][4 * grp + 2], dq[db][4 * grp + 3]};
            }
        __syncthreads();
#pragma unroll
        for (int db = 0; db < DB; ++db)
            if ((db < DB0) == (stream == 0)) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const f32x4 other = park[(4 * db + grp) * 64 + lane];
#pragma unroll
                    for (int i = 0; i < 4; ++i) dq[db][4 * grp + i] += other[i];
                }
            }
    }
    if (qvalid && p.grad_typed) {  // overwrite mode: dq has the input dtype
        char* dqp = (char*)p.dq.ptr + 2 * ((int64_t)b * p.dq.sb + (int64_t)qrow * p.dq.ss + (int64_t)h * p.dq.sh);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (merged && (db < DB0) != (stream == 0)) continue;
            store_block16<T>(dqp + 64 * db, p.d - 32 * db, hi, [&](int i) { return dq[db][i] * p.scale; });
        }
    } else if (qvalid) {
        float* dqp = (float*)p.dq.ptr + ((int64_t)b * p.dq.sb + (int64_t)qrow * p.dq.ss + (int64_t)h * p.dq.sh);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (merged && (db < DB0) != (stream == 0)) continue;
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                if (32 * db + 8 * grp >= p.d) break;
                const int d0 = 32 * db + 8 * grp + 4 * hi;
                f32x4 a = *(f32x4*)(dqp + d0);
#pragma unroll
                for (int x = 0; x < 4; ++x) a[x] = fmaf(dq[db][4 * grp + x], p.scale, a[x]);
                *(f32x4*)(dqp + d0) = a;
            }
        }
    }
}


// ---------------------------------------------------------------------------------------
// Sorted rows: dK/dV of sequences whose rows have been moved and of the others are different instantiations.  As long as the host
// has not seen the plan builder's count word both are launched, and the workgroups of the wrong one end at once (a launch of 2048
// such workgroups: 16 us, their LDS keeps them from running beside each other).
inline bool rows_may_be_moved(const AttnParams& p) { return p.rows != nullptr && p.rows_known != BAM_ROWS_LEFT; }
inline bool rows_may_be_left(const AttnParams& p) { return p.rows == nullptr || p.rows_known != BAM_ROWS_MOVED; }
template <typename T, int D, bool BIAS, bool LONG, bool SAVE, bool SCALED>
static int launch_dkdv_m(const AttnParams& p, hipStream_t stream) {
    const int blocks = p.num_kt * p.B * p.Hkv;  // one workgroup per 128-key tile
    if (p.mask_mode == MASK_INDEXED)
        hipLaunchKernelGGL((bwd_dkdv_kernel<T, D, MASK_INDEXED, BIAS, LONG, SAVE, SCALED>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, p);
    else if (p.mask_mode == MASK_DENSE)
        hipLaunchKernelGGL((bwd_dkdv_kernel<T, D, MASK_DENSE, BIAS, LONG, SAVE, SCALED>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, p);
    else {
        if constexpr (!LONG) {  // (beyond, there are no sorted rows)
            if (rows_may_be_moved(p))
                hipLaunchKernelGGL((bwd_dkdv_kernel<T, D, MASK_SORTED, BIAS, LONG, SAVE, SCALED>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, p);
        }
        if (LONG || rows_may_be_left(p))
            hipLaunchKernelGGL((bwd_dkdv_kernel<T, D, MASK_BITFIELD, BIAS, LONG, SAVE, SCALED>), dim3(blocks), dim3(DKDV_THREADS), 0, stream, p);
    }
    return (int)hipGetLastError();
}
template <typename T, int D, bool BIAS, bool LONG, bool SAVE = false>
static int launch_dkdv_b(const AttnParams& p, hipStream_t stream) {
    if constexpr (!BIAS && !LONG && D <= 64)
        if (p.lse_scaled != nullptr) return launch_dkdv_m<T, D, BIAS, LONG, SAVE, true>(p, stream);
    return launch_dkdv_m<T, D, BIAS, LONG, SAVE, false>(p, stream);
}
template <typename T, int D, int BIAS, bool LONG, int STREAMS>
static int launch_dq_s(const AttnParams& p, hipStream_t stream) {
    const int blocks = p.num_m * p.B * p.Hq, threads = DQ_THREADS * STREAMS;
    if (p.mask_mode == MASK_INDEXED)
        hipLaunchKernelGGL((bwd_dq_kernel<T, D, MASK_INDEXED, BIAS, LONG, STREAMS>), dim3(blocks), dim3(threads), 0, stream, p);
    else if (p.mask_mode == MASK_DENSE)
        hipLaunchKernelGGL((bwd_dq_kernel<T, D, MASK_DENSE, BIAS, LONG, STREAMS>), dim3(blocks), dim3(threads), 0, stream, p);
    else
        hipLaunchKernelGGL((bwd_dq_kernel<T, D, MASK_BITFIELD, BIAS, LONG, STREAMS>), dim3(blocks), dim3(threads), 0, stream, p);
    return (int)hipGetLastError();
}
// Two streams where the forward takes them.  dQ alone, us, one stream -> two: D 64, 1000 tokens, 8 heads 27.1 -> 22.7, 1024, 32 heads
// 29.4 -> 25.1, 2 x 700 28.4 -> 27.2, 2048 (512 workgroups) 50.9 -> 49.8, 3001 (768) 77 -> 87; with a bias 2 x 2048, 16 heads 64.1 -> 59.2; D 32: 2048 46.4 -> 35.9, 3001 64.1 -> 52.9, 4096
// (1024) 84.3 -> 77.0, 8 x 300 (768) 18.8 -> 24.3.
template <typename T, int D, int BIAS, bool LONG>
static int launch_dq_f(const AttnParams& p, hipStream_t stream) {
    if constexpr (!LONG && D <= 64)  // (above, dQ is computed from the stored dS but for rare calls)
        if (two_streams(p)) return launch_dq_s<T, D, BIAS, false, 2>(p, stream);
    return launch_dq_s<T, D, BIAS, LONG, 1>(p, stream);
}
template <typename T, int D, bool LONG>
static int launch_dq_b(const AttnParams& p, hipStream_t stream) {
    if (p.bias == nullptr) return launch_dq_f<T, D, BIAS_NONE, LONG>(p, stream);
    return p.bias_sm == 0 && p.bias_vec ? launch_dq_f<T, D, BIAS_TILES, LONG>(p, stream) : launch_dq_f<T, D, BIAS_READ, LONG>(p, stream);
}

// fn<T, D>(p, stream) for the element type and head dimension of the call
#define BAM_DISPATCH(fn)                                       \
    if (dtype == 1) {                                          \
        if (p.D == 128) return fn<BF16, 128>(p, stream);       \
        if (p.D == 96) return fn<BF16, 96>(p, stream);         \
        if (p.D == 64) return fn<BF16, 64>(p, stream);         \
        return fn<BF16, 32>(p, stream);                        \
    }                                                          \
    if (p.D == 128) return fn<F16, 128>(p, stream);            \
    if (p.D == 96) return fn<F16, 96>(p, stream);              \
    if (p.D == 64) return fn<F16, 64>(p, stream);              \
    return fn<F16, 32>(p, stream);

}  // namespace bam
