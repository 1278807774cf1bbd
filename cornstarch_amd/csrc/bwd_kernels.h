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
    if (valid && c == 0) {
        const int64_t at = (int64_t)b * p.lse_sb + (int64_t)h * p.Sq_rounded + i;
        p.delta[at] = acc;
        if (D <= 64 && p.lse_scaled != nullptr) p.lse_scaled[at] = p.lse[at] * LOG2E;
    }
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
// The two waves that share a key group hold partial sums; at the end one hands its dV over through LDS, the other its dK, and each
// adds up and stores what it has received: deterministic and atomic free.  (Four-wave form: a wave takes both rows of slices, and
// holds the whole sums.)
constexpr int DKDV_QT = 64;
constexpr int DKDV_THREADS = 512, DKDV_NARROW_THREADS = 256;

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
// A tile is 16 MFMAs per wave at head dims up to 64, half of what it is above, and there is room for four buffers: two tiles
// are copied ahead and the workgroup meets after every second one.  dK/dV alone, us, a meeting per tile -> per two: D 64, 3001
// tokens, 32 / 8 heads 190 -> 180, 2 x 700 57.7 -> 54.9, 8 x 4096, 16 heads 555 -> 532; D 32: 3001 148.8 -> 139.8.
// (Sorted rows have row numbers to copy one tile earlier still.)
template <int D, int MODE, bool LONG>
constexpr bool DKDV_DEEP = D <= 64 && MODE != MASK_SORTED && !LONG;

// LDS of dkdv_work.  (The kernels declare the same arrays one by one.)
template <int D, int MODE>
struct DkdvShared {
    static constexpr int NB = DKDV_DEEP<D, MODE, false> ? 4 : 2;  // tile buffers
    static constexpr int NCH = LDS_COLS<D> / 8;
    __attribute__((aligned(256))) u32x4 k[128 * NCH];
    u32x4 v[128 * NCH];
    u32x4 q[NB][DKDV_QT * NCH];
    u32x4 dout[NB][DKDV_QT * NCH];
    __attribute__((aligned(16))) float lse[NB][DKDV_QT];    // natural-log lse of the rows
    __attribute__((aligned(16))) float delta[NB][DKDV_QT];
    __attribute__((aligned(16))) int64_t qbf[NB][DKDV_QT];  // raw bitfields of the rows
    __attribute__((aligned(16))) int qpos[NB][DKDV_QT];     // their positions (MASK_INDEXED)
    __attribute__((aligned(16))) unsigned wq[DKDV_THREADS / 64][5][32];  // per-wave rule constants
    // MASK_DENSE with packed mask bits: for the two slices of the tile, one word per key of the workgroup's 128 keys
    unsigned col_bits[MODE == MASK_DENSE ? NB : 1][2][MODE == MASK_DENSE ? 128 : 1];
    int list[MAX_SLICE_LIST + 1];  // entry -1: partner of the first entry of an odd count
    int count;
};

template <typename T, int D, int MODE, bool BIAS, bool LONG, bool SAVE = false, bool SCALED = false>
__global__ __launch_bounds__(DKDV_THREADS, 2) void bwd_dkdv_kernel(const AttnParams p) {
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = MODE == MASK_DENSE, SORTED = MODE == MASK_SORTED;
    constexpr bool ROW_POS = IDX || SORTED;  // the rows' positions travel with the tiles
    static_assert(!(SORTED && LONG), "no plan for so many rows");
    constexpr bool NARROW = false, KEY_BIAS = false, DEEP = DKDV_DEEP<D, MODE, LONG>;
    constexpr int NB = DEEP ? 4 : 2;  // tile buffers
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    __shared__ __attribute__((aligned(256))) u32x4 sTiles[(2 * 128 + 2 * NB * DKDV_QT) * NCH];
    u32x4* const sK = sTiles;
    u32x4* const sV = sTiles + 128 * NCH;
    u32x4 (*const sQ)[DKDV_QT * NCH] = (u32x4 (*)[DKDV_QT * NCH])(sTiles + 256 * NCH);
    u32x4 (*const sDO)[DKDV_QT * NCH] = sQ + NB;
    __shared__ __attribute__((aligned(16))) float sRowNumbers[2 * NB][DKDV_QT];
    float (*const sLse)[DKDV_QT] = sRowNumbers;  // natural-log lse of the rows
    float (*const sDelta)[DKDV_QT] = sRowNumbers + NB;
    __shared__ __attribute__((aligned(16))) int64_t sQbf[NB][DKDV_QT];    // raw bitfields of the rows
    // their positions (ROW_POS).  SORTED: a tile's rows are gathered, so their numbers have to be here a tile earlier
    __shared__ __attribute__((aligned(16))) int sQpos[SORTED ? 3 : NB][DKDV_QT];
    __shared__ __attribute__((aligned(16))) unsigned sWq[DKDV_THREADS / 64][5][32];  // per-wave rule constants
    // DENSE with packed mask bits: for the two slices of the tile, one word per key of the workgroup's 128 keys
    __shared__ unsigned sColBits[MODE == MASK_DENSE ? NB : 1][2][MODE == MASK_DENSE ? 128 : 1];
    __shared__ int sListStore[MAX_SLICE_LIST + 1];  // entry -1: partner of the first entry of an odd count
    int* const sList = sListStore + 1;
    __shared__ int sCount;

    const int block = blockIdx.x;
#include "bwd_dkdv_body.h"
}

// The same work for head dims up to 64 by four waves, one for each 32 keys, that take both slices of a pair one after the other: three
// workgroups fit a unit, so a third wave per SIMD fills the gaps of MFMAs, arithmetic and LDS reads (each 450 to 550 cycles of a 32 x 32
// block's 1050 at head dim 64 with two), and a workgroup's start and end pass behind the others' work.  168 registers: every wave
// holds its K and V operands, and nothing lies in LDS but Q, dO and the small rows; what derives from the lane is derived anew for
// every block (75 vector instructions a block beside the MFMAs); the rule constants of a block are read one row at a time.  (Spilled K and V operands, read back between
// the tile copies, wait for those: step 1.26 -> 1.42 ms at 8 x 4096.)  No partial sums to add at the end.
// Step through the public entry points, us, eight waves -> four, both in turn in one process, D 64: 8 x 4096, 16 heads, segments of 256
// to 512 tokens 1290 -> 1246, of 256 to 1024 1072 -> 1038 (replayed as a graph 1087 -> 1003), 8 x 2048 389 -> 367, 32 x 512, 32 heads 445 -> 412,
// 8 x 4096, 32 / 8 heads 2388 -> 2350, 16384, 16 heads, nothing hidden 5192 -> 5195; D 32: 8 x 2048, 16 heads 282 -> 239, 16 x 512, 32 heads
// 168 -> 137, 2 x 8192, 16 heads 821 -> 744.
template <typename T, int D, int MODE, bool BIAS, bool SCALED>
__global__ __launch_bounds__(DKDV_NARROW_THREADS, 3) void bwd_dkdv_narrow_kernel(const AttnParams p) {
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = false, SORTED = false, ROW_POS = IDX, LONG = false, SAVE = false;
    constexpr bool NARROW = true, KEY_BIAS = false, DEEP = false;
    constexpr int NB = 2;
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    __shared__ __attribute__((aligned(256))) u32x4 sTiles[2 * NB][DKDV_QT * NCH];
    u32x4 (*const sQ)[DKDV_QT * NCH] = sTiles;
    u32x4 (*const sDO)[DKDV_QT * NCH] = sTiles + NB;
    u32x4* const sK = sTiles[0];  // (not in LDS: named by code that is not compiled for this kernel)
    u32x4* const sV = sTiles[0];
    __shared__ __attribute__((aligned(16))) float sRowNumbers[2 * NB][DKDV_QT];
    float (*const sLse)[DKDV_QT] = sRowNumbers;
    float (*const sDelta)[DKDV_QT] = sRowNumbers + NB;
    __shared__ __attribute__((aligned(16))) int64_t sQbf[NB][DKDV_QT];
    __shared__ __attribute__((aligned(16))) int sQpos[NB][DKDV_QT];
    __shared__ __attribute__((aligned(16))) unsigned sWq[4][5][32];
    __shared__ unsigned sColBits[1][2][1];
    __shared__ int sListStore[MAX_SLICE_LIST + 1];
    int* const sList = sListStore + 1;
    __shared__ int sCount;

    const int block = blockIdx.x;
#include "bwd_dkdv_body.h"
}

// The work of workgroup `block` of a dK/dV launch, in LDS of the caller's: rows in natural order, one pass, no dS kept.
template <typename T, int D, int MODE, bool BIAS, bool SCALED>
__device__ __forceinline__ void dkdv_work(const AttnParams& p, const int block, DkdvShared<D, MODE>& sh) {
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = MODE == MASK_DENSE, ROW_POS = IDX;
    constexpr bool NARROW = false, SORTED = false, LONG = false, SAVE = false;
    constexpr bool KEY_BIAS = BIAS;  // (both_in_one_launch refuses a bias with rows of its own)
    constexpr bool DEEP = DKDV_DEEP<D, MODE, LONG>;
    constexpr int NB = DEEP ? 4 : 2;  // tile buffers
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    typedef DkdvShared<D, MODE> Shared;
    static_assert(alignof(Shared) % 256 == 0 && offsetof(Shared, k) % 256 == 0 && offsetof(Shared, q) % 256 == 0 &&
                      offsetof(Shared, v) - offsetof(Shared, k) == sizeof(Shared::k) && offsetof(Shared, dout) - offsetof(Shared, q) == sizeof(Shared::q) &&
                      offsetof(Shared, delta) - offsetof(Shared, lse) == sizeof(Shared::lse),
                  "the second array of each pair is read at a constant behind the first, and addresses below 256 are XORed");
    auto &sK = sh.k, &sV = sh.v;
    auto &sQ = sh.q, &sDO = sh.dout;
    auto &sLse = sh.lse, &sDelta = sh.delta;
    auto& sQbf = sh.qbf;
    auto& sQpos = sh.qpos;
    auto& sWq = sh.wq;
    auto& sColBits = sh.col_bits;
    int* const sList = sh.list + 1;
    int& sCount = sh.count;
#include "bwd_dkdv_body.h"
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
template <int D, int MODE, int BIAS_FORM, int STREAMS>
struct DqShared {
    static constexpr int NCH = LDS_COLS<D> / 8;
    static constexpr bool DENSE = MODE == MASK_DENSE, bias_lds = BIAS_FORM == BIAS_TILES;
    __attribute__((aligned(256))) u32x4 k[STREAMS][2][DQ_KT * NCH];
    u32x4 v[STREAMS][2][DQ_KT * NCH];
    __attribute__((aligned(16))) int64_t kbf[STREAMS][2][DQ_KT];  // raw bitfields of the tile's keys
    __attribute__((aligned(16))) int kpos[STREAMS][2][DQ_KT];     // their global positions (MASK_INDEXED only)
    int list[MAX_LIST];
    int count[STREAMS];
    // MASK_DENSE with packed mask bits: per wave, the words of its 32 rows for the tile's two 32-key blocks
    unsigned row_bits[STREAMS][DENSE ? 2 : 1][4][DENSE ? 64 : 1];
    // BIAS_TILES: the 64 bias values of the tile
    __attribute__((aligned(16))) unsigned bias[STREAMS][bias_lds ? 2 : 1][bias_lds ? 64 : 1];
};

// The work of workgroup `block` of a dQ launch.
template <typename T, int D, int MODE, int BIAS_FORM, bool LONG, int STREAMS>
__device__ __forceinline__ void dq_work(const AttnParams& p, const int block, DqShared<D, MODE, BIAS_FORM, STREAMS>& sh) {
    static_assert(STREAMS == 1 || !LONG, "streams and passes are not combined");
    constexpr bool BIAS = BIAS_FORM != BIAS_NONE, bias_lds = BIAS_FORM == BIAS_TILES;
    constexpr bool IDX = MODE == MASK_INDEXED, DENSE = MODE == MASK_DENSE;
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32;
    constexpr int WAIT = COPY_WAIT<BIAS, LONG>;
    auto &sK_all = sh.k, &sV_all = sh.v;
    auto& sKbf_all = sh.kbf;
    auto& sKpos_all = sh.kpos;
    auto& sList = sh.list;
    auto& sCount = sh.count;
    auto& sRowBits_all = sh.row_bits;
    auto& sBias_all = sh.bias;

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
    head_unit_map(block, p.num_m * p.B, p.Hkv, G, ub, hk, g);
    constexpr bool MAY_SIDE = STREAMS > 1 && D > 32;
    int code = 0;
    bool side = false, idle = false;  // the streams take a unit each; ... and there is none left for this one
    if constexpr (MAY_SIDE) {
        if (p.group_order != nullptr) code = plan_word(p.group_order + ub);
        side = streams_side_by_side(p);
        if (__builtin_expect(side, 0)) {
            const int units = p.num_m * p.B * p.Hq, unit = side_unit(block, stream);
            if (side_unit(block, 0) >= units) return;
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
    // Up to head dim 64 there are registers (without a bias 119 to 125 and 165 to 168 of 168) to start the dP chain from -delta, as dK/dV does:
    // 16 of some 73 vector instructions a block less.  Step, us, D 32: 8 x 2048 tokens, 16 heads 249.0 -> 243.3, 2 x 8192 779 -> 760, 1 x 2048 93.6 -> 92.7.
    // D 64, since the LDS addresses are XORed (160 registers before): dQ of 8 x 4096, 16 heads 314 -> 299, with a bias, in one launch with
    // dK/dV, 2 x 2048 89.7 -> 87.3.
    // At head dim 64 the 16 (equal) values are written anew for every block where a bias is read group by group, or where the keys take several passes
    // without a bias in the tiles (whose form may have 256 registers): no register is left there to hold them.  dQ, us, held -> written
    // anew: 133120 tokens, 2 heads, one segment 6643 -> 6173 (spilled registers 62 -> 31), with such a bias 13368 -> 11088 (97 -> 45); a bias per row, 4 x 2048,
    // 16 heads 178 either way (3 -> 0).  Masks gain from them in several passes all the same (7564 held, 7842 without any start values), and so
    // does a bias in the tiles (7208, 7463).  All forms have the same sums.
    constexpr bool DELTA_FIRST = D <= 64;
    constexpr bool DELTA_HELD = D <= 32 || (DELTA_FIRST && BIAS_FORM != BIAS_READ && !(LONG && BIAS_FORM == BIAS_NONE && MODE != MASK_DENSE));
    f32x16 minus_delta;
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
        if (DELTA_HELD)
#pragma unroll
            for (int i = 0; i < 16; ++i) minus_delta[i] = -dlt;
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

    // Where this lane reads in buffer 0, as byte addresses, as in the forward: the K operand of k-slice 0 (V: V_AT behind it) and the
    // transposed K operand of column block 0.
    constexpr unsigned ROW_BYTES = NCH * 16, V_AT = STREAMS * 2 * TILE_BYTES;
    static_assert(alignof(decltype(sh)) % 256 == 0, "addresses below 256 are XORed");
    const int lane16 = lane & 15;
    const unsigned k_lane = ldsK + 16u * (unsigned)chunk_slot<D>(l32, hi);
    const unsigned kt_lane =
        ldsK + 16u * (unsigned)chunk_slot<D>(4 * hi + (lane16 >> 2), 2 * half16 + ((lane16 & 3) >> 1)) + 8u * (lane16 & 1);

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
        const unsigned k_at = k_lane + cur * TILE_BYTES, kt_at = kt_lane + cur * TILE_BYTES;
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
                auto operand = [&](int j) {
                    return lds_read16<u32x4>((k_at ^ (32u * (j >> 1))) + 32u * kb * ROW_BYTES + ((j & 1) ? V_AT : 0u));
                };
#pragma unroll
                for (int j = 0; j < AHEAD; ++j) a[j] = operand(j);
#pragma unroll
                for (int j = 0; j < NOP; ++j) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (j + AHEAD < NOP) a[j + AHEAD] = operand(j + AHEAD);
                    if (DELTA_FIRST && !DELTA_HELD && j == 1) {
                        float here = -dlt;
                        asm volatile("" : "+v"(here));
#pragma unroll
                        for (int i = 0; i < 16; ++i) dp[i] = here;
                    }
                    if (j & 1)
                        dp = T::mfma(a[j], greg[j >> 1], j < 2 ? (DELTA_HELD ? minus_delta : DELTA_FIRST ? dp : zero16) : dp);
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
                dp[i] = e * (DELTA_FIRST ? dp[i] : dp[i] - dlt);  // the factor `scale` of dS is applied to dQ in the epilogue
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
                        ta[t][db] = lds_read_transposed_at((kt_at ^ (64u * db)) + (32u * kb + 16u * t) * ROW_BYTES,
                                                           (kt_at ^ (64u * db + 16u)) + (32u * kb + 16u * t + 8u) * ROW_BYTES);
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
template <typename T, int D, int MODE, int BIAS_FORM, bool LONG, int STREAMS>
__global__ __launch_bounds__(DQ_THREADS * STREAMS, D > 64 || BIAS_FORM == BIAS_TILES || STREAMS > 1 ? 2 : 3) void bwd_dq_kernel(const AttnParams p) {
    __shared__ DqShared<D, MODE, BIAS_FORM, STREAMS> sh;
    dq_work<T, D, MODE, BIAS_FORM, LONG, STREAMS>(p, blockIdx.x, sh);
}

// dK/dV and dQ in one launch, for small problems: the workgroups of one kernel take the units that the other leaves idle at its
// end.  The first `dkdv_blocks` workgroups are dK/dV's (`kv`: its parameters, which differ from dQ's where the q heads of a kv head
// are dealt to parts), the others dQ's.  Delta (and the scaled lse) come from the pre-pass.
template <typename T, int D, int MODE, int BIAS_FORM>
__global__ __launch_bounds__(DKDV_THREADS, 2) void bwd_both_kernel(const AttnParams kv, const AttnParams p, const int dkdv_blocks) {
    static_assert(DKDV_THREADS == 2 * DQ_THREADS, "dQ with two streams");
    constexpr bool BIAS = BIAS_FORM != BIAS_NONE;
    __shared__ union {
        DkdvShared<D, MODE> dkdv;
        DqShared<D, MODE, BIAS_FORM, 2> dq;
    } sh;
    if ((int)blockIdx.x < dkdv_blocks)
        dkdv_work<T, D, MODE, BIAS, !BIAS && D <= 64>(kv, blockIdx.x, sh.dkdv);
    else
        dq_work<T, D, MODE, BIAS_FORM, false, 2>(p, blockIdx.x - dkdv_blocks, sh.dq);
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
    // Four waves (bwd_dkdv_narrow_kernel) where there are more than four workgroups a unit.  Few leave the units a wave or two per SIMD: step,
    // us, D 32, 512 workgroups (2 x 2048, 16 heads) 107 -> 110, 576 (4 x 3000, 6 heads) 156 -> 160; D 64, 512 (8192, 32 / 8 heads) 1045 -> 1196.
    // The line at 1024 is not one of speed: from 768 on they win (8 x 700, 16 heads, D 32 91 -> 83, D 64 3 x 2048 179 -> 176).  But their sums come
    // in another order, and the test of level lists holds a call of 1024 workgroups (2 x 2048 tokens, 32 heads) to the bits of one of 512.  Across the
    // line the bits of dK and dV change with the size of the call.
    // A bias takes registers that head dim 64 does not have: 8192, 16 heads 648 -> 672 (D 32: 8 x 2048 330 -> 282).
    if constexpr (D <= 64 && !LONG && !SAVE && !(BIAS && D > 32)) {
        if (p.rows == nullptr && blocks > 1024 && p.mask_mode != MASK_DENSE) {
            if (p.mask_mode == MASK_INDEXED)
                hipLaunchKernelGGL((bwd_dkdv_narrow_kernel<T, D, MASK_INDEXED, BIAS, SCALED>), dim3(blocks), dim3(DKDV_NARROW_THREADS), 0, stream, p);
            else
                hipLaunchKernelGGL((bwd_dkdv_narrow_kernel<T, D, MASK_BITFIELD, BIAS, SCALED>), dim3(blocks), dim3(DKDV_NARROW_THREADS), 0, stream, p);
            return (int)hipGetLastError();
        }
    }
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
