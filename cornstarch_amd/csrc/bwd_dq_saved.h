// dQ from saved dS: the second half of the backward that does NOT recompute S and dP for dQ.
// Reference semantics: cornstarch/kernel/bitfield_attention.py:877-898 (ds rounded to the input dtype, dq += ds k); the
// reference adds every 128 x 32 tile's contribution to dq with fp32 atomics, here the dK/dV kernel (SAVE form) leaves
// its 32 x 32 blocks of -dS / scale in a workspace and this kernel, which owns whole query rows, sums them up:
// dQ^T = K^T dS^T over the key tiles that have work for the slice.  One GEMM instead of three, no exponentials, no
// mask logic (masked pairs were stored as zeros); the price is reading the workspace once.
//
// Work decomposition: as the forward -- a workgroup is four 32-row slices of one (batch, q head), one per wave (taken
// from the plan's slice order), and walks the 64-key tiles any of them needs; K tiles are shared through LDS (double
// buffered), every wave copies its own dS blocks (two 2 KiB blocks per tile, one per 32-key half) into a wave-private
// LDS area, two tiles ahead: a buffer is refilled as soon as its operands are in registers.  Both MFMA operands come
// from transposing LDS reads: K^T (d x keys) from the row-major K tile, dS^T (keys x rows) from the block, which the
// dK/dV lanes wrote key by key.
#pragma once
#include "bam_common.h"
#include "bam_launch.h"
#include "bam_tiles.h"
#include <type_traits>

namespace bam {

constexpr int DQS_KT = 64;
constexpr int DQS_THREADS = 256;

// List, in ascending order, the 64-key tiles the four slices of a workgroup have to visit (at most MAX_LIST).
// entry = (tile << 16) | sum_w (c0_w | c1_w << 2) << (4 w), c0 / c1 = class of the tile's two 32-key halves for wave
// w's slice.  first: load_tile_classes of this lane's first tile.  Executed by wave 0; the caller synchronizes before reading.
__device__ __forceinline__ void build_key_half_list(const WaveSlices& ws, int num_n, int S, int lane, const TileClasses& first, int* list,
                                                    int* count_out) {
    const int nkt = key_tiles(S, 0);
    int count = 0;
    TileClasses cur = first;
    for (int base = 0; base < nkt; base += 64) {
        const TileClasses next = load_tile_classes(ws, num_n, nkt, base + 64 + lane);
        const int kt = base + lane;
        const bool second = 2 * kt + 1 < num_n;
        int packed = 0;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int f0 = cur.f[x][0] & 3, f1 = second ? cur.f[x][1] & 3 : 0;
            packed |= ws.cls_row[x] != nullptr ? (f0 | (f1 << 2)) << (4 * x) : 0;
        }
        if (kt >= nkt) packed = 0;
        const unsigned long long bal = __ballot(packed != 0);
        if (packed) list[count + __popcll(bal & ((1ull << lane) - 1ull))] = (kt << 16) | packed;
        count += __popcll(bal);
        cur = next;
    }
    if (lane == 0) *count_out = count;
    wait_lds();
}

template <typename T, int D>
__global__ __launch_bounds__(DQS_THREADS, 2) void bwd_dq_saved_kernel(const AttnParams p) {
    constexpr int NCH = LDS_COLS<D> / 8, DB = D / 32;
    __shared__ u32x4 sK[2][DQS_KT * NCH];
    __shared__ __attribute__((aligned(256))) u32x4 sDS[DQS_THREADS / 64][2][256];  // per wave and buffer: two 2 KiB blocks (key halves 0 and 1)
    __shared__ int sList[MAX_LIST];
    __shared__ int sCount;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
    const int wave_lane = tid >> 6;
    const int Sq = p.Sq, Sk = p.Sk;
    const int G = p.Hq / p.Hkv;

    int ub, hk, g;
    // (dQ alone, us, falling -> mirrored: D 128, 2 x 2003 tokens, 16 heads 41.6 -> 37.8, 8192, 8 heads 139.8 -> 129.5; D 96, 2 x 2003,
    // 16 heads 36.1 -> 33.6.  The forward gains nothing: there a workgroup takes the same time with or without a second one.)
    head_unit_map(mirror_second(blockIdx.x, gridDim.x), p.num_m * p.B, p.Hkv, G, ub, hk, g);
    int b = ub % p.B, grp = ub / p.B;
    if (p.group_order != nullptr) {  // with a plan: the groups of all sequences by falling length of their tile lists
        const int code = p.group_order[ub];
        b = code / p.num_m;
        grp = code - b * p.num_m;
    }
    const int h = hk * G + g;
    const WaveSlices ws = pick_wave_slices(p, b, grp);  // the plan's order (the launcher requires a plan)

    TileClasses first_classes = {};
    if (wave == 0) first_classes = load_tile_classes(ws, p.num_n, key_tiles(Sk, 0), lane);

    const int slice = __builtin_amdgcn_readfirstlane(wave == 0 ? ws.slice[0] : wave == 1 ? ws.slice[1] : wave == 2 ? ws.slice[2] : ws.slice[3]);
    // column n of a dS block holds query row 8 * ((n & 15) >> 2) + 4 * (n >> 4) + (n & 3) of the slice
    const int slot = (slice < 0 ? 0 : slice) * 32 + 8 * ((l32 & 15) >> 2) + 4 * (l32 >> 4) + (l32 & 3);
    const bool qvalid = slice >= 0 && slot < Sq;
    const int qrow = row_of_slot(p, ws, b, slot, qvalid);
    // Record numbers of the slice's pairs, 64 key tiles at a time: lane j holds the one of 128-key tile 64 ent_chunk + j.  The first
    // 64 are asked for together with the classes, before anybody knows which of them are needed.
    // The loaded value is handed on through an instruction of its own, so that the compiler's wait for the load sits
    // right here (once per 128 tiles) and not in front of every later use: a wait for this load is a wait for every
    // tile copy in flight.
    const int* entry_row = p.ds_entry + (int64_t)b * p.ds_entry_sb + (int64_t)(slice < 0 ? 0 : slice) * p.num_kt;
    int ent_vec = 0, ent_chunk = 0;
    auto load_entries = [&](int chunk) {
        const int e = entry_row[min(64 * chunk + lane, p.num_kt - 1)];
        ent_chunk = chunk;
        return e;
    };
    auto keep_entries = [&](int e) { asm volatile("v_mov_b32 %0, %1" : "=v"(ent_vec) : "v"(e)); };
    const int first_entries = load_entries(0);
    if (wave == 0) build_key_half_list(ws, p.num_n, Sk, lane, first_classes, sList, &sCount);

    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dq[db][i] = 0.f;

    RowView<false> k_rows;
    k_rows.init((const char*)p.k.ptr + 2 * ((int64_t)b * p.k.sb + (int64_t)hk * p.k.sh), 2 * p.k.ss, Sk, 2 * p.d);
    typedef TileStage<D, DQS_KT, DQS_THREADS> Stage;
    constexpr int CPT = Stage::CPT;
    Stage stK;
    stK.setup(2 * p.k.ss, p.d / 8, tid);
    const unsigned ldsK = lds_addr(sK), ldsDS = lds_addr(sDS) + wave * 8192u;
    constexpr unsigned TILE_BYTES = DQS_KT * NCH * 16;
    // records of this q head; record e (a slice x 128-key tile pair) is 8 KiB = four 2 KiB blocks
    const char* ds_head = (const char*)p.ds_ws + (((int64_t)h * p.ds_capacity) << 13);
    // record number of the pair of list entry `entry` (64-key tile kt -> 128-key tile kt / 2; the entries come in ascending order)
    auto entry_number = [&](int entry) {
        const int tile = entry >> 17;
        if ((tile >> 6) != ent_chunk) keep_entries(load_entries(tile >> 6));
        return __builtin_amdgcn_readlane(ent_vec, tile & 63);
    };

    // copy of the K tile of list entry `entry` into buffer buf (shared by the four waves)
    auto issue_k = [&](int entry, int buf) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) stK.template issue<0>(j, k_rows.at((entry >> 16) * DQS_KT), ldsK + buf * TILE_BYTES);
    };
    // copies of this wave's dS blocks of tile `entry` (record e), the halves that have work, into its buffer buf;
    // returns the number of copy instructions issued (wave-uniform)
    auto issue_ds = [&](int entry, int e, int buf) -> int {
        const int kt = entry >> 16;
        const int c = (entry >> (4 * wave)) & 15;  // wave-uniform
        const char* rec = ds_head + ((int64_t)e << 13) + (kt & 1) * 4096;
        int issued = 0;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
            if ((c >> (2 * kb)) & 3) {
                dma_b128_stream<1>(rec + kb * 2048, (unsigned)(lane * 16), ldsDS + buf * 4096u + kb * 2048u);
                dma_b128_stream<2>(rec + kb * 2048, (unsigned)(lane * 16 + 1024), ldsDS + buf * 4096u + kb * 2048u + 1024u);
                issued += 2;
            }
        return issued;
    };

    // Where this lane reads in the first block of buffer 0: column 16 half16 + (lane & 15) of keys 4 hi + {0,1,2,3}.  16 keys further are 256
    // bytes, 8 keys a bit of the address.  (The layout: bwd_dkdv_body.h, ds_first.)
    const int lane16 = lane & 15, upper = (lane16 >> 1) & 1;
    const unsigned ds_lane = ldsDS + (unsigned)(upper * 1024 + half16 * 512 + ((4 * hi + (lane16 >> 2)) ^ (4 * upper) ^ (8 * half16)) * 16 + (lane16 & 1) * 8);

    // One 64-key tile.  The dS operands are read first; the wave's buffer is then free again and takes the blocks of
    // the tile after next (`entry2`, record `e2`; negative entry2 = nothing left), so that two tiles' worth of
    // workspace reads are in flight per wave: the kernel waits for HBM, not for the MFMAs.  Returns the number of
    // copies issued.
    auto tile_step = [&](int cur, int entry, int entry2, int e2) -> int {
        // (per-lane copy of the wave number: a skip branch the compiler can prove wave-uniform makes it restructure the loop)
        const int c = (entry >> (4 * wave_lane)) & 15;
        const u32x4* tK = sK[cur];
        const unsigned ds_at = ds_lane + cur * 4096u;
        u32x4 bop[2][2];
        if (c != 0) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    if ((c >> (2 * kb)) & 3) {
                        const unsigned x = ds_at + 2048u * kb + 256u * t;
                        bop[kb][t] = lds_read_transposed_at(x, x ^ 128u);
                    }
            wait_lds();  // the copies below overwrite what was just read
        }
        const int issued = entry2 >= 0 ? issue_ds(entry2, e2, cur) : 0;
        if (c == 0) return issued;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            if (((c >> (2 * kb)) & 3) == 0) continue;
            u32x4 ta[2][DB];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int db = 0; db < DB; ++db)
                    ta[t][db] = lds_read_transposed<D>(tK, lane, 32 * kb + 16 * t + 4 * hi, 32 * db + 16 * half16);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int db = 0; db < DB; ++db) dq[db] = T::mfma(ta[t][db], bop[kb][t], dq[db]);
        }
        return issued;
    };

    __syncthreads();
    const int n = sCount;
    if (n > 0) {
        keep_entries(first_entries);
        int entry = __builtin_amdgcn_readfirstlane(sList[0]);
        int next = __builtin_amdgcn_readfirstlane(sList[n > 1 ? 1 : 0]);
        issue_k(entry, 0);
        issue_ds(entry, entry_number(entry), 0);
        if (n > 1) issue_ds(next, entry_number(next), 1);
        wait_async();
        __syncthreads();
        for (int it = 0; it < n; ++it) {
            const int cur = it & 1;
            // the K tile of the next entry (past the end the last tile is copied again: nobody reads it)
            issue_k(next, cur ^ 1);
            // the dS blocks of the entry after next
            const int i2 = it + 2;
            int entry2 = -1, e2 = 0;
            if (i2 < n) {
                entry2 = __builtin_amdgcn_readfirstlane(sList[i2]);
                e2 = entry_number(entry2);
            }
            const int issued = tile_step(cur, entry, entry2, e2);
            entry = next;
            next = entry2 >= 0 ? entry2 : next;
            // everything but the copies of the entry after next has to have landed: copies complete in order
            if (issued == 4)
                asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else if (issued == 2)
                asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
            else
                wait_async();
            __syncthreads();
        }
    }
    // ---- epilogue: dq holds -dQ / scale (C fragment: lane = query column, registers = head dims 8 g + 4 hi + x)
    const float factor = -p.scale;
    if (qvalid && p.grad_typed) {
        char* dqp = (char*)p.dq.ptr + 2 * ((int64_t)b * p.dq.sb + (int64_t)qrow * p.dq.ss + (int64_t)h * p.dq.sh);
#pragma unroll
        for (int db = 0; db < DB; ++db)
            store_block16<T>(dqp + 64 * db, p.d - 32 * db, hi, [&](int i) { return dq[db][i] * factor; });
    } else if (qvalid) {
        float* dqp = (float*)p.dq.ptr + ((int64_t)b * p.dq.sb + (int64_t)qrow * p.dq.ss + (int64_t)h * p.dq.sh);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                if (32 * db + 8 * grp >= p.d) break;
                const int d0 = 32 * db + 8 * grp + 4 * hi;
                f32x4 a = *(f32x4*)(dqp + d0);
#pragma unroll
                for (int x = 0; x < 4; ++x) a[x] = fmaf(dq[db][4 * grp + x], factor, a[x]);
                *(f32x4*)(dqp + d0) = a;
            }
    }
}

}  // namespace bam
