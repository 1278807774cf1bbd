// Forward kernel of bitfield-masked attention for gfx950 (template; instantiated by fwd.hip and fwd_long.hip).
// Reference semantics: cornstarch/kernel/bitfield_attention.py:236-523 (+ the split-KV merge
// :1292-1436, which a single pass over the keys makes unnecessary).
//
// Work decomposition
//   workgroup  = four 32-row slices of one (batch, q head), one per wave: a 128-row block, or, with a plan,
//                four slices that need about the same keys (sorted slice order).
//   key loop   = 64-key tiles taken from the class rows of those slices: tiles no slice needs are never
//                touched; a wave skips the tiles its own slice does not need, skips the mask where every
//                pair of its slice is allowed, and evaluates the bitfield rule in registers otherwise.
//   K/V tiles  = double buffered in LDS; the next tile is copied global -> LDS directly while
//                the current one is consumed.
// Math layout
//   S^T = K Q^T on v_mfma_f32_32x32x16 with K rows as the A operand (LDS) and Q as the B
//   operand (registers).  In the C fragment a lane owns ONE query (lane & 31) and 16 of the
//   32 keys of a block, so the running max / sum / rescale factors are per-lane scalars and
//   the only cross-lane traffic is one exchange with lane ^ 32.  P^T then feeds
//   O^T = V^T P^T straight from registers as the B operand; V^T comes from the row-major V
//   tile through the transposing LDS read.
#pragma once
#include "bam_common.h"
#include "bam_launch.h"
#include "bam_tiles.h"
#include <type_traits>

namespace bam {

constexpr int FWD_KT = 64;
constexpr int FWD_THREADS = 256;

// MODE (MASK_*): where allow / deny comes from.  MASK_INDEXED: query rows and keys carry explicit global
// positions (p.posq, p.posk) and the bitfield arrays are already gathered per local row / key
// (context-parallel shards, reference bitfield_attention.py:71-81).  MASK_DENSE: a materialized bool mask
// (the reference's sibling kernel, cornstarch/kernel/attention.py:184-232), read from global memory in the
// tiles the flags call partial.
// BIAS: an additive bias p.bias (reference bitfield_attention.py:410-434) is added to scale * q.k.
// LONG: sequences of more than MAX_LIST 64-key tiles (131072 keys), walked in several passes; the short form has no
// pass loop at all (a loop around the main loop costs registers and a few per cent).
// STREAMS: how many tiles of the list are in work at a time, each by four waves of its own on the same four slices.
template <typename T, int D, int MODE, bool BIAS, bool LONG, int STREAMS>
__global__ __launch_bounds__(FWD_THREADS * STREAMS, D > 64 || STREAMS > 1 ? 2 : 3) void fwd_kernel(const AttnParams p) {
    static_assert(STREAMS == 1 || !LONG, "streams and passes are not combined");
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    __shared__ __attribute__((aligned(256))) u32x4 sK_all[STREAMS][2][FWD_KT * NCH];
    __shared__ __attribute__((aligned(256))) u32x4 sV_all[STREAMS][2][FWD_KT * NCH];
    __shared__ __attribute__((aligned(16))) int64_t sKbf_all[STREAMS][2][FWD_KT];  // raw bitfields of the tile's keys
    __shared__ __attribute__((aligned(16))) int sKpos_all[STREAMS][2][FWD_KT];     // their global positions (IDX only)
    __shared__ int sList[MAX_LIST];
    __shared__ int sCount[STREAMS];
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = MODE == MASK_DENSE;
    // DENSE with packed mask bits: per wave, the words of its 32 rows for the tile's two 32-key blocks
    __shared__ unsigned sRowBits_all[STREAMS][DENSE ? 2 : 1][4][DENSE ? 64 : 1];
    // BIAS in its per-key ("vector") form: the 64 values of the tile (raw words; 16-bit elements fill half)
    __shared__ __attribute__((aligned(16))) unsigned sBias_all[STREAMS][BIAS ? 2 : 1][BIAS ? 64 : 1];

    // (tid and wave: inside the stream)
    const int tid = threadIdx.x % FWD_THREADS, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int stream = STREAMS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / FWD_THREADS) : 0;
    auto &sK = sK_all[stream], &sV = sV_all[stream];
    auto& sKbf = sKbf_all[stream];
    auto& sKpos = sKpos_all[stream];
    auto& sRowBits = sRowBits_all[stream];
    auto& sBias = sBias_all[stream];
    const int hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
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

    // ---- per-lane query state -------------------------------------------------------
    const int slice = idle ? -1 : __builtin_amdgcn_readfirstlane(wave == 0 ? ws.slice[0] : wave == 1 ? ws.slice[1] : wave == 2 ? ws.slice[2] : ws.slice[3]);
    const int slot = (slice < 0 ? 0 : slice) * 32 + l32;
    const bool qvalid = slice >= 0 && slot < Sq;
    const int qrow = row_of_slot(p, ws, b, slot, qvalid);
    // (the class bytes are asked for ahead of the rows: loads arrive in order)
    const bool lists = wave == 0 && (stream == 0 || side);
    const int list_keys = idle ? 0 : Sk;
    TileClasses first_classes = {};
    if (lists) first_classes = load_tile_classes(ws, p.num_n, key_tiles(list_keys, 0), lane);
    u32x4 qreg[KK];
    {
        const char* qp = (const char*)p.q.ptr + 2 * ((int64_t)b * p.q.sb + (int64_t)qrow * p.q.ss + (int64_t)h * p.q.sh);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            u32x4 z = {0u, 0u, 0u, 0u};
            if (qvalid && 16 * kk + 8 * hi < p.d) z = *(const u32x4*)(qp + (16 * kk + 8 * hi) * 2);
            qreg[kk] = z;
        }
    }
    int64_t qf = (!DENSE && qvalid) ? p.bfq[(int64_t)b * p.bfq_sb + qrow] : 0;
    int qpos = (IDX && qvalid) ? p.posq[qrow] : qrow;
    QueryBits qb = {};  // of qf and qpos, once they have arrived
    // (the row loads above are in flight while the class rows are read and the first tile is on its way)
    if (lists)  // first pass (usually the only one)
        build_key_tile_list<STREAMS>(ws, p.num_n, list_keys, lane, 0, first_classes, sList + stream * (MAX_LIST / 2), sCount + stream, !side);

    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    // Online softmax state.  m_i is the reference maximum the exponentials are taken against;
    // it is only moved (and O, l rescaled) when a tile raises a row's maximum by more than
    // RESCALE_LOG2 in the exponent, so most tiles skip the rescale entirely.  Until then the
    // probabilities are at most 2^RESCALE_LOG2, harmless in fp32 / bf16 and cancelled by the
    // final division by l.
    constexpr float RESCALE_LOG2 = 8.f;
    float m_i = -INFINITY, l_i = 0.f, nb = 0.f;  // nb = -m_i * c2 (0 while m_i is -inf); l_i: this lane's half of the row's sum
    // with a bias the scores are turned into scale * s + bias right after the S phase, and only log2(e) is left
    // to fold into the exponent
    // A per-key bias whose groups of four keys are aligned, in-range accesses travels with the tile copies: 64 values
    // per tile, one word per lane (16-bit elements: lanes 32..63 repeat lanes 0..31).
    const bool bias_lds = BIAS && p.bias_sm == 0 && p.bias_vec != 0;
    // ... and with bf16 operands it is added by the matrix cores: bias / scale, split into three bf16 values, rides in
    // one more MFMA of the S phase against an operand of ones, so that the scores come out as q.k + bias / scale and
    // the exponent is taken exactly as without a bias (no multiply-add per score, no bias reads per score).
    const bool bias_fold = bias_lds && std::is_same<T, BF16>::value;
    const float c2 = (BIAS && !bias_fold) ? LOG2E : p.scale * LOG2E;
    const float inv_scale = 1.f / p.scale;
    const char* bias_row = nullptr;  // this lane's row of the bias
    if (BIAS)
        bias_row = (const char*)p.bias + (p.bias_f32 ? 4 : 2) * ((int64_t)b * p.bias_sb + (int64_t)h * p.bias_sh +
                                                                (int64_t)(qvalid ? qrow : 0) * p.bias_sm);
    const float rescale_thr = RESCALE_LOG2 / c2;
    f32x16 zero16;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero16[i] = 0.f;

    RowView<LONG> k_rows, v_rows;
    RowView<false> bf_rows, pos_rows, bias_rows;  // key bitfields, (IDX) positions, per-key bias
    k_rows.init((const char*)p.k.ptr + 2 * ((int64_t)b * p.k.sb + (int64_t)hk * p.k.sh), 2 * p.k.ss, Sk, 2 * p.d);
    v_rows.init((const char*)p.v.ptr + 2 * ((int64_t)b * p.v.sb + (int64_t)hk * p.v.sh), 2 * p.v.ss, Sk, 2 * p.d);
    if (!DENSE) bf_rows.init(p.bfk + (int64_t)b * p.bfk_sb, 8, Sk, 8);
    if (IDX) pos_rows.init(p.posk, 4, Sk, 4);

    typedef TileStage<D, FWD_KT, FWD_THREADS, true> Stage;
    constexpr int CPT = Stage::CPT;
    // copy instructions per wave and tile: K, V, the key bitfields (DENSE: the mask bits of the wave's rows) and
    // (IDX) the key positions
    constexpr int NLOADS = 2 * CPT + 1 + (IDX ? 1 : 0) + (BIAS ? 1 : 0);
    static_assert(NLOADS <= 2 * KK + 1, "one copy per MFMA of the S phase (and at most one behind it)");
    Stage stK, stV;
    stK.setup(2 * p.k.ss, p.d / 8, tid);
    stV.setup(2 * p.v.ss, p.d / 8, tid);
    const unsigned ldsK = lds_addr(sK), ldsV = lds_addr(sV), ldsB = lds_addr(sKbf), ldsP = lds_addr(sKpos);
    const unsigned ldsR = lds_addr(sRowBits);
    if (BIAS) {
        const int esz = p.bias_f32 ? 4 : 2;
        bias_rows.init((const char*)p.bias + esz * ((int64_t)b * p.bias_sb + (int64_t)h * p.bias_sh), esz, Sk, esz);
    }
    const unsigned bias_voff = (unsigned)((p.bias_f32 ? lane : (lane & 31)) * 4);
    // DENSE: the packed mask rows of this wave's slice (null: no plan, the mask bytes are read instead)
    const unsigned* row_bits_w = (DENSE && p.row_bits != nullptr)
                                     ? p.row_bits + (int64_t)b * p.row_bits_sb + (slice < 0 ? 0 : slice) * 32
                                     : nullptr;
    const unsigned row_bits_voff = DENSE ? (unsigned)(hi * (int)p.row_bits_sn * 4 + l32 * 4) : 0u;
    constexpr unsigned TILE_BYTES = FWD_KT * NCH * 16, BITS_BYTES = FWD_KT * 8;
    // Copy instruction j (0 <= j < NLOADS) of tile kt into buffer buf.  The 128 dwords of key
    // bitfields are copied 64 dwords per wave (waves 2, 3 repeat what waves 0, 1 write), so that every
    // wave issues the same number of copies.
    auto issue_copy = [&](int j, int kt, int buf) {
        const int row = kt * FWD_KT;
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
            copy_b32<WAIT>(pos_rows.at(row), (unsigned)(lane * 4), ldsP + buf * (FWD_KT * 4u));
        else if (bias_lds)  // BIAS: the tile's 64 bias values; every wave writes the same values
            copy_b32<WAIT>(bias_rows.at(row), bias_voff, lds_addr(sBias) + buf * 256u);
    };

    // Where this lane reads in buffer 0, as byte addresses (forward alone, 24 problems of 512 to 8192 tokens, head dims 64 to 128, 1.01x of indices
    // computed per read: 512 to 1024 tokens 1.02x, 8192 1.005x): the K operand of k-slice 0 and the transposed V operand of column block 0.  What
    // a k-slice or a block of columns adds is a constant, XORed (the swizzle takes bits 0 to 3 of the row, the tiles start at multiples
    // of 256), rows are in the instruction.
    constexpr unsigned ROW_BYTES = NCH * 16;
    const int lane16 = lane & 15;
    const unsigned k_lane = ldsK + 16u * (unsigned)chunk_slot<D>(l32, hi);
    const unsigned v_lane =
        ldsV + 16u * (unsigned)chunk_slot<D>(4 * hi + (lane16 >> 2), 2 * half16 + ((lane16 & 3) >> 1)) + 8u * (lane16 & 1);
    // keys 32 kb .., k-slice kk
    auto k_operand = [&](unsigned at, int kb, int kk) { return lds_read16<u32x4>((at ^ (32u * kk)) + 32u * kb * ROW_BYTES); };
    // keys 32 kb + 16 t .., columns 32 db ..
    auto v_operand = [&](unsigned at, int kb, int t, int db) {
        const unsigned row = (32u * kb + 16u * t) * ROW_BYTES;
        return lds_read_transposed_at((at ^ (64u * db)) + row, (at ^ (64u * db + 16u)) + row + 8u * ROW_BYTES);
    };

    // One 64-key tile held in buffer `cur`.  The copies of tile `kt_next` into the other
    // buffer are issued one per MFMA of the S phase, where the wave has nothing else to wait for.
    auto tile_step = [&](int cur, int entry, int kt_next) {
        // (One `if` after the other that the compiler does not take for `else`, and none that leaves: the accumulators then stay in their
        // registers.  With a return for the skipped tile, or classes it takes for divergent, it copied all of O to and fro in every tile.)
        const int kt = entry >> 8, cls = (entry >> (2 * wave)) & 3;
        if (cls == 0) {  // nothing for this wave's slice in the tile: only keep the copies of the next one going
#pragma unroll
            for (int j = 0; j < NLOADS; ++j) issue_copy(j, kt_next, cur ^ 1);
        }
        int work = cls;
        asm volatile("" : "+s"(work));
        if (work != 0) {
            const unsigned k_at = k_lane + cur * TILE_BYTES;

            // ---- S^T = K Q^T : 64 keys x 32 queries per wave ----------------------------------
            // two independent accumulator chains (key blocks 0 and 1) alternate; operand reads run AHEAD
            // MFMAs in front of their use; the first MFMA of a chain takes C = 0
            // (the MFMA phases run at raised wave priority: when the SIMD's other wave is in its softmax phase, this
            // wave's next MFMA is picked first and the MFMA pipe does not idle behind a queue of VALU instructions)
            f32x16 s[2];
            u32x4 bias_a[2];  // bias_fold: this lane's key of either 32-key block, as an operand (keys are the rows of S^T)
            if (BIAS && bias_fold) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const float bv = p.bias_f32 ? ((const float*)sBias[cur])[32 * kb + l32]
                                                : T::to_float(((const unsigned short*)sBias[cur])[32 * kb + l32]);
                    const u32x4 z = {0u, 0u, 0u, 0u};
                    bias_a[kb] = hi == 0 ? split3_operand<T>(bv * inv_scale) : z;
                }
            }
            __builtin_amdgcn_s_setprio(1);
            {
                constexpr int NOP = 2 * KK, AHEAD = 4;
                u32x4 ka[NOP];
#pragma unroll
                for (int j = 0; j < AHEAD; ++j) ka[j] = k_operand(k_at, j & 1, j >> 1);
#pragma unroll
                for (int j = 0; j < NOP; ++j) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (j + AHEAD < NOP)
                        ka[j + AHEAD] = k_operand(k_at, (j + AHEAD) & 1, (j + AHEAD) >> 1);
                    s[j & 1] = T::mfma(ka[j], qreg[j >> 1], j < 2 ? zero16 : s[j & 1]);
                    if (j < NLOADS) issue_copy(j, kt_next, cur ^ 1);
                }
#pragma unroll
                for (int j = NOP; j < NLOADS; ++j) issue_copy(j, kt_next, cur ^ 1);
                if (BIAS && bias_fold) {
                    const u32x4 z = {0u, 0u, 0u, 0u};
                    const u32x4 ones = hi == 0 ? ones3_operand<T>() : z;
                    s[0] = T::mfma(bias_a[0], ones, s[0]);
                    s[1] = T::mfma(bias_a[1], ones, s[1]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);

            if (BIAS && bias_fold) {
                // (added by the MFMA above)
            } else if (BIAS && bias_lds) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
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
                        for (int x = 0; x < 4; ++x) s[kb][4 * grp + x] = fmaf(s[kb][4 * grp + x], p.scale, b4[x]);
                    }
            } else if (BIAS) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int grp = 0; grp < 4; ++grp) {
                        const f32x4 b4 = load_bias4<T>(bias_row, kt * FWD_KT + 32 * kb + 8 * grp + 4 * hi, Sk, p.bias_f32 != 0, p.bias_vec != 0);
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            s[kb][4 * grp + x] = bias_fold ? fmaf(b4[x], inv_scale, s[kb][4 * grp + x])  // (c2 holds the scale)
                                                           : fmaf(s[kb][4 * grp + x], p.scale, b4[x]);
                    }
            }

            // ---- bitfield rule in registers (partial tiles only) ------------------------------
            // two_kinds: every row of the slice sees all keys of the tile or none.  The latter's scores stay as they are (they may be NaN), and their
            // packed probabilities are cleared: 17 instructions for 64.  A slice with text and modality rows, or with padding, has such
            // tiles all the way back, and its workgroup is often the longest of a launch: 3001 tokens with two segments, 32 / 8
            // heads, D 128 80.6 -> 78.6 us, 4096 rows of a zigzag shard against 8192 keys 272 -> 263; text only and nothing hidden alike.
            bool two_kinds = false, sees = true;
            if (DENSE) {
                if (cls == 1 && row_bits_w != nullptr) {
                    unsigned w01[2] = {sRowBits[cur][wave][l32], sRowBits[cur][wave][32 + l32]};
                    sees = (w01[0] & w01[1]) == ~0u;
                    two_kinds = __all(sees | ((w01[0] | w01[1]) == 0u));
                    if (!two_kinds) {
                        sees = true;
                        // (shifted by this lane's first key, 4 hi, once: the bit numbers tested are then constants)
                        w01[0] >>= 4 * hi;
                        w01[1] >>= 4 * hi;
#pragma unroll
                        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                            for (int i = 0; i < 16; ++i)
                                s[kb][i] = ((w01[kb] >> (8 * (i >> 2) + (i & 3))) & 1u) ? s[kb][i] : -INFINITY;
                    }
                } else if (cls == 1) {
                    // mask bytes of this lane's query row: 4 consecutive keys per C-fragment group
                    const int kt0 = kt * FWD_KT;
                    const uint8_t* mrow = p.mask + ((int64_t)b * Sq + (qvalid ? qrow : 0)) * Sk + kt0;
                    const bool dwords = (Sk & 3) == 0;  // rows start 4-byte aligned
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
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
                                s[kb][4 * grp + x] = a ? s[kb][4 * grp + x] : -INFINITY;
                            }
                        }
                }
            } else if (cls == 1) {
                // Most partial tiles are partial only through causality: all 64 keys carry the same bitfield (and,
                // with index tensors, sit at consecutive positions).  Then the bit test is a per-query constant and
                // the rule reduces to one position compare.
                const int64_t mine = sKbf[cur][lane];
                const unsigned mlo = (unsigned)mine, mhi = (unsigned)((uint64_t)mine >> 32);
                const unsigned flo = __builtin_amdgcn_readfirstlane(mlo), fhi = __builtin_amdgcn_readfirstlane(mhi);
                bool uniform = (mlo == flo) & (mhi == fhi);
                int kt0 = kt * FWD_KT;  // position of the tile's first key
                if (IDX) {
                    const int rel0 = sKpos[cur][lane] - lane;
                    kt0 = __builtin_amdgcn_readfirstlane(rel0);
                    uniform &= rel0 == kt0;
                }
                if (__all(uniform)) {
                    // last allowed key, relative to the first key this lane holds (4 hi): what it is compared with are
                    // then compile-time constants, which occupy no registers
                    const int rel = allow_bits(qb, flo, fhi) ? qb.lim - kt0 - 4 * hi : -1;
                    sees = rel >= 59;  // (the last key of a lane: 32 + 24 + 3)
                    two_kinds = __all(sees | (rel < 0));
                    if (!two_kinds) {
                        sees = true;
#pragma unroll
                        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                            for (int i = 0; i < 16; ++i)
                                s[kb][i] = (32 * kb + 8 * (i >> 2) + (i & 3) <= rel) ? s[kb][i] : -INFINITY;
                    }
                } else {
                    // natural positions: the row's limit relative to the first key this lane holds, so that the position
                    // test compares with compile-time constants
                    const int lim_rel = qb.lim - (kt * FWD_KT + 4 * hi);
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
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
                                const bool a = allow_bits(qb, klo[x], khi[x]) & pos_ok;
                                s[kb][4 * grp + x] = a ? s[kb][4 * grp + x] : -INFINITY;
                            }
                        }
                }
            }

            // ---- online softmax (per-lane scalars) ----------------------------------------------
            // (The maximum is looked at before any exponential.  Exponentials of one 32-key half beside the MFMAs of the other against the maximum of
            // the tiles before, and the tile done again where one came out too large, gave 3 % with standard normal q and k where a launch's
            // second round is half empty (3001 tokens, 32 / 8 heads, D 128), nothing elsewhere, and lost 4 to 19 % with scores of deviation 3
            // to 8, as trained models have them; with the probabilities scaled afterwards instead it still lost 1 to 7 %.)
            // (four short chains instead of one long one: the wave issues in order and would sit out the latency of
            // every link)
            float mx[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                mx[c] = fmaxf(s[0][4 * c], s[1][4 * c]);
#pragma unroll
                for (int i = 1; i < 4; ++i) mx[c] = fmaxf(fmaxf(mx[c], s[0][4 * c + i]), s[1][4 * c + i]);
            }
            float mloc = half_swap_max(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])));
            mloc = sees ? mloc : -INFINITY;
            if (__any(mloc > m_i + rescale_thr)) {  // wave-uniform; rare after the first tiles
                const float mnew = fmaxf(m_i, mloc);
                const float muse = (mnew == -INFINITY) ? 0.f : mnew;
                const float alpha = __builtin_amdgcn_exp2f((m_i - muse) * c2);  // 0 when m_i = -inf
                m_i = mnew;
                nb = -muse * c2;
                l_i *= alpha;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[0][i] = __builtin_amdgcn_exp2f(fmaf(s[0][i], c2, nb));
                s[1][i] = __builtin_amdgcn_exp2f(fmaf(s[1][i], c2, nb));
            }
            u32x4 pb[2][2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int t = 0; t < 2; ++t) pb[kb][t] = pack8<T>(s[kb], 8 * t);
            if (__builtin_expect(two_kinds, 0)) {
                const unsigned keep = sees ? ~0u : 0u;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int t = 0; t < 2; ++t) pb[kb][t] &= u32x4{keep, keep, keep, keep};
            }
            // row sum of the probabilities as the P V product sees them (rounded to T), two per instruction; a tile's are added up by
            // themselves and meet the running sum once
            {
                float ps[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int x = 0; x < 4; ++x) ps[kb][t] = T::add_pair(pb[kb][t][x], ps[kb][t]);
                l_i += (ps[0][0] + ps[0][1]) + (ps[1][0] + ps[1][1]);
            }

            // ---- O^T += V^T P^T -------------------------------------------------------------------
            __builtin_amdgcn_s_setprio(1);
            constexpr int PV = 2 * DB, VAHEAD = 3 < PV ? 3 : PV;
            const unsigned v_at = v_lane + cur * TILE_BYTES;
            u32x4 va[2 * PV];
            auto read_v = [&](int j) { va[j] = v_operand(v_at, j / PV, j % PV / DB, j % DB); };
#pragma unroll
            for (int j = 0; j < VAHEAD; ++j) read_v(j);
#pragma unroll
            for (int j = 0; j < 2 * PV; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                if (j + VAHEAD < 2 * PV) read_v(j + VAHEAD);
                o[j % DB] = T::mfma(va[j], pb[j / PV][j % PV / DB], o[j % DB]);
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(0);
        }
    };

    // Sequences of more than MAX_LIST 64-key tiles are walked in several passes, each with a list of its own; the
    // softmax state lives in registers and simply carries over.
    const int nkt_total = (Sk + FWD_KT - 1) / FWD_KT;
    for (int kt_begin = 0;;) {
        lds_barrier();
        // With two streams, one takes the even tiles and the other the odd ones.  Past the end of its list a stream copies its
        // last tile again, for nobody to read or, where the other list is longer, with all classes cleared.
        const int n = sCount[stream], rounds = STREAMS > 1 ? max(n, sCount[STREAMS - 1 - stream]) : n;
        if (rounds > 0) {
            const int* const list = sList + stream * (MAX_LIST / 2);
            auto list_at = [&](int i) {
                if (STREAMS == 1) return list[i < n ? i : n - 1];
                const int e = list[i < n ? i : max(n - 1, 0)];
                return i < n ? e : n > 0 ? e & ~0xFF : 0;
            };
            int entry = __builtin_amdgcn_readfirstlane(list_at(0));
            int next = __builtin_amdgcn_readfirstlane(list_at(1));
    #pragma unroll
            for (int j = 0; j < NLOADS; ++j) issue_copy(j, entry >> 8, 0);
            wait_async();
            arrived(qreg);
            if (!LONG || kt_begin == 0) qb = make_query_bits(qf, qpos);
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

    // ---- epilogue: normalize, write O (q dtype) and LSE (natural log) -------------------
    float ltot = half_swap_sum(l_i), mine = 1.f, theirs = 0.f;
    // With two streams, a row's two partial results meet through the tile arrays, which nobody reads any more: each stream
    // hands over the columns that the other one finishes.
    constexpr int DB0 = STREAMS > 1 ? (DB + 1) / 2 : DB;  // stream 0 finishes the column blocks below DB0, stream 1 the others
    f32x4* const park = (f32x4*)sK_all + wave * (DB * 4 * 64);
    float* const park_ml = (float*)sV_all;
    auto meet = [&]() {
#pragma unroll
        for (int db = 0; db < DB; ++db)
            if ((db < DB0) == (stream == 1)) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp)
                    park[(4 * db + grp) * 64 + lane] = f32x4{o[db][4 * grp], o[db][4 * grp + 1], o[db][4 * grp + 2], o[db][4 * grp + 3]};
            }
        park_ml[(8 * stream + 2 * wave) * 64 + lane] = m_i;
        park_ml[(8 * stream + 2 * wave + 1) * 64 + lane] = ltot;
        __syncthreads();
        const float m_other = park_ml[(8 * (1 - stream) + 2 * wave) * 64 + lane];
        const float l_other = park_ml[(8 * (1 - stream) + 2 * wave + 1) * 64 + lane];
        const float m = fmaxf(m_i, m_other), muse = m == -INFINITY ? 0.f : m;
        mine = __builtin_amdgcn_exp2f((m_i - muse) * c2);  // 0 for a stream that has seen no key of this row
        theirs = __builtin_amdgcn_exp2f((m_other - muse) * c2);
        ltot = stream == 0 ? fmaf(ltot, mine, l_other * theirs) : fmaf(l_other, theirs, ltot * mine);
        m_i = m;
    };
    if constexpr (STREAMS > 1)
        if (!side) meet();
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
    if ((stream == 0 || side) && hi == 0 && slice >= 0)
        p.lse[(int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded + qrow] =
            ltot > 0.f ? (m_i * c2 + __builtin_amdgcn_logf(ltot)) * LN2 : -INFINITY;
    // A wave without a slice (plan: slot 4 grp + wave of the order lies past the last slice) owns the 32 padding rows
    // of that slot, so that every row of the rounded lse is written whether or not a plan is given.
    if ((stream == 0 || side) && !idle && hi == 0 && slice < 0 && 32 * (4 * grp + wave) + 31 < p.Sq_rounded)
        p.lse[(int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded + 32 * (4 * grp + wave) + l32] = -INFINITY;
    if (qvalid) {
        char* op = (char*)p.o.ptr + 2 * ((int64_t)b * p.o.sb + (int64_t)qrow * p.o.ss + (int64_t)h * p.o.sh);
        if constexpr (MAY_SIDE)
            if (__builtin_expect(side, 0)) {  // (a loop of its own: the other one reads the partner's blocks together)
#pragma unroll
                for (int db = 0; db < DB; ++db) store_block16<T>(op + 64 * db, p.d - 32 * db, hi, [&](int i) { return o[db][i] * inv; });
                return;
            }
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (STREAMS > 1 && (db < DB0) != (stream == 0)) continue;
            f32x16 x = o[db];
            if constexpr (STREAMS > 1) {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const f32x4 other = park[(4 * db + grp) * 64 + lane];
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[4 * grp + i] = fmaf(x[4 * grp + i], mine, other[i] * theirs);
                }
            }
            store_block16<T>(op + 64 * db, p.d - 32 * db, hi, [&](int i) { return x[i] * inv; });
        }
    }
}


// Launches every (mask mode, bias) instantiation of one (element type, head dim, LONG) combination.
template <typename T, int D, bool BIAS, bool LONG, int STREAMS>
static int launch_fwd_s(const AttnParams& p, hipStream_t stream) {
    const int blocks = p.num_m * p.B * p.Hq, threads = FWD_THREADS * STREAMS;
    if (p.mask_mode == MASK_INDEXED)
        hipLaunchKernelGGL((fwd_kernel<T, D, MASK_INDEXED, BIAS, LONG, STREAMS>), dim3(blocks), dim3(threads), 0, stream, p);
    else if (p.mask_mode == MASK_DENSE)
        hipLaunchKernelGGL((fwd_kernel<T, D, MASK_DENSE, BIAS, LONG, STREAMS>), dim3(blocks), dim3(threads), 0, stream, p);
    else
        hipLaunchKernelGGL((fwd_kernel<T, D, MASK_BITFIELD, BIAS, LONG, STREAMS>), dim3(blocks), dim3(threads), 0, stream, p);
    return (int)hipGetLastError();
}
// Two streams halve the chain of tiles a workgroup walks and double the waves of a compute unit that has one workgroup; the price
// is a workgroup that fills the unit (D = 64 and above), so that nothing runs beside its first loads and its stores.  Forward
// kernel alone, bf16, us, one stream -> two (workgroups in brackets; lists of a causal mask with a few segments):
//   D 128:  60 tokens (64) 8.3 -> 9.9;  120 (288) 14.5 -> 21.9;  250 (256) 17.4 -> 16.3, (384) 19.7 -> 25.6;  640 (240) 24.0 ->
//           21.0, (320) 26.2 -> 28.3;  1000 (384) 36.2 -> 34.5, (512) 37.7 -> 42.5;  1500 (384) 45.9 -> 36.6, (480) 47.8 -> 47.5;  2000 (384) 53.5 ->
//           42.8, (512) 55.1 -> 54.7
//   D 64:   60 (256) 7.6 -> 8.7;  250 (256) 14.0 -> 12.4, (384) 15.3 -> 19.4;  640 (320) 21.8 -> 22.3, (480) 23.0 -> 26.8;  900
//           (384) 26.9 -> 25.6, (512) 28.7 -> 30.6;  1500 (480) 37.1 -> 33.1;  1000 (640) 32.2 -> 40.3
//   D 32 (two such workgroups fit a unit):  60 (64) 6.9 -> 7.5;  120 (288) 9.9 -> 10.7;  250 (384) 13.3 -> 12.1, (512) 13.8 ->
//           14.1;  500 (512) 18.1 -> 16.8;  2048 (512) 37.8 -> 28.2, 3001 (768) 52.4 -> 40.7, 4096 (1024) 69 -> 61, but with short
//           lists 8 x 300 (768) 16.0 -> 19.5, 4 x 1024 (1024) 27.8 -> 30.4;  with a bias 4096 (640) 82 -> 77, (1024) 85 -> 107;
//           nothing hidden: 2048 (512) 34.4 -> 32.3, 3001 (768) 69.1 -> 66.9, 4096 (1024) 118 -> 112
// Above 512 workgroups and D 32 the mask decides: text only / 4 / 10 segments / nothing hidden, D 128, 5000 tokens (640) 119 -> 128 /
// 118 -> 108 / 128 -> 99 / 234 -> 241;  3200 (600) 79 -> 89 / 82 -> 80 / 92 -> 71 / 158 -> 165;  8192 (768) 220 -> 240 / 205 -> 205 /
// 198 -> 151 / 409 -> 415;  D 64, 6500 (765) 109 -> 124 / 120 -> 111 / 136 -> 94 / 204 -> 219.  The host launches before anybody
// has seen the lists, and the plainest mask is the one that loses: one stream.
template <typename T, int D, bool BIAS, bool LONG>
static int launch_fwd_b(const AttnParams& p, hipStream_t stream) {
    if constexpr (!LONG)
        if (two_streams(p)) return launch_fwd_s<T, D, BIAS, false, 2>(p, stream);
    return launch_fwd_s<T, D, BIAS, LONG, 1>(p, stream);
}
template <typename T, int D, bool LONG>
static int launch_fwd_t(const AttnParams& p, hipStream_t stream) {
    return p.bias != nullptr ? launch_fwd_b<T, D, true, LONG>(p, stream) : launch_fwd_b<T, D, false, LONG>(p, stream);
}
template <bool LONG>
static int launch_fwd_all(const AttnParams& p, int dtype, hipStream_t stream) {
    if (dtype == 1) {
        if (p.D == 128) return launch_fwd_t<BF16, 128, LONG>(p, stream);
        if (p.D == 96) return launch_fwd_t<BF16, 96, LONG>(p, stream);
        if (p.D == 64) return launch_fwd_t<BF16, 64, LONG>(p, stream);
        return launch_fwd_t<BF16, 32, LONG>(p, stream);
    }
    if (p.D == 128) return launch_fwd_t<F16, 128, LONG>(p, stream);
    if (p.D == 96) return launch_fwd_t<F16, 96, LONG>(p, stream);
    if (p.D == 64) return launch_fwd_t<F16, 64, LONG>(p, stream);
    return launch_fwd_t<F16, 32, LONG>(p, stream);
}

}  // namespace bam
