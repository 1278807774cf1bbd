// Global -> LDS tile staging and the flag-driven tile lists shared by the
// forward and backward kernels.
#pragma once
#include "bam_common.h"
#include "bam_launch.h"

namespace bam {

// LDS byte address of a __shared__ object (what the LDS-DMA base register M0 wants).
__device__ __forceinline__ unsigned lds_addr(const void* p) {
    return (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)p;
}

// LDS reads at a byte address: 16 bytes, and the two halves of a transposed operand (see lds_read_transposed)
template <typename V>
__device__ __forceinline__ V lds_read16(unsigned at) {
    return *(const __attribute__((address_space(3))) V*)at;
}
__device__ __forceinline__ u32x4 lds_read_transposed_at(unsigned a, unsigned b) {
    typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr;
    const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)a));
    const u32x2 y = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)b));
    return u32x4{x[0], x[1], y[0], y[1]};
}

// One direct global -> LDS copy instruction.  Lane l fetches `bytes` (16 or 4) from
// sbase + voff and the hardware writes them to LDS byte address lds_base + l * bytes;
// sbase and lds_base must be wave-uniform.  The LDS base travels in M0: it is handed to the asm
// statement as an input operand bound to that register, so the compiler writes M0 itself and knows
// it is occupied; the s_nop is the wait state the hardware wants between an M0 write and its use.  Issued as inline asm on purpose: the compiler
// then neither tracks the copy in vmcnt nor makes later LDS reads wait for it, which is what
// lets a tile load stay in flight across a whole loop iteration.  The price is that the
// caller owns the synchronization: wait_async() (or wait_async_but<N>()) + a workgroup
// barrier before anyone reads the destination.
// SITE only labels the instruction (as an assembler comment): copies issued from different places of a
// kernel get different labels, which keeps the compiler from merging them into one hoisted copy and so
// keeps each where the schedule wants it.
template <int SITE = 0>
__device__ __forceinline__ void dma_b128(const void* sbase, unsigned voff, unsigned lds_base) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 ; site %3" ::"v"(voff), "s"(sbase), "{m0}"(lds_base),
                 "n"(SITE)
                 : "memory");
}
// The same with the non-temporal hint: data that is read once (it should not displace what other workgroups re-read
// from the L2).
template <int SITE = 0>
__device__ __forceinline__ void dma_b128_stream(const void* sbase, unsigned voff, unsigned lds_base) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt ; site %3" ::"v"(voff), "s"(sbase), "{m0}"(lds_base),
                 "n"(SITE)
                 : "memory");
}
// The 16-byte copy through a buffer descriptor over [base, base + DMA_RANGE): a lane whose offset lies beyond reads nothing
// and the hardware writes zeros to its LDS slot.  For the K tiles of the decode step (8 x 8192 keys: 48.7 us either way); the other
// kernels copy through RowView.
constexpr unsigned DMA_RANGE = 0x80000000u, DMA_ZERO = 0xC0000000u;  // (room below for 31 rows of 2^24 bytes: decode steps back)
// The same for RowView, whose descriptors end below 2^31 and whose copies add a scalar offset below 2^31: beyond any of them, and
// the sum stays below 2^32.
constexpr unsigned ROW_ZERO = 0x80000000u;
template <int SITE = 0>
__device__ __forceinline__ void dma_b128_ranged(const void* sbase, unsigned voff, unsigned lds_base) {
    const unsigned long long base = reinterpret_cast<unsigned long long>(sbase);  // (48 bits: no stride in the second word)
    const u32x4 desc = {(unsigned)base, (unsigned)(base >> 32), DMA_RANGE, 0x00020000u};
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds ; site %3" ::"v"(voff), "s"(desc), "{m0}"(lds_base),
                 "n"(SITE)
                 : "memory");
}
template <int SITE = 0>
__device__ __forceinline__ void dma_b32(const void* sbase, unsigned voff, unsigned lds_base) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1 ; site %3" ::"v"(voff), "s"(sbase), "{m0}"(lds_base),
                 "n"(SITE)
                 : "memory");
}

// Consecutive rows of one head of one sequence (or of any array) that tiles are copied from: a buffer descriptor over exactly
// these rows, and where a tile starts in it.  Whatever a copy addresses past the last row becomes zeros in LDS (the hardware's
// range check covers the scalar offset too), so the tile that holds the end of a sequence is copied like any other.  The
// descriptor stays in scalar registers over the key loop and a tile costs one 32-bit product: with a 64-bit base per tile and
// the end of the sequence staged by a second instance of the loop body, dK/dV at D = 128 needed 88 bytes of scratch per lane.
// (Where rows overlap in memory -- a stride below the row's own bytes, 0 for a broadcast -- rows past the end may repeat bytes of
// the rows before them instead.)
// FAR: views of 2^31 bytes and more; the descriptor is built per tile around a 64-bit base.
constexpr unsigned BUFFER_WORD3 = 0x00020000u;
struct TileSrc {
    u32x4 desc;
    unsigned off;  // bytes, wave-uniform
};
template <bool FAR>
struct RowView {
    u32x4 desc;
    unsigned stride;  // bytes from row to row, below 2^24 by the host checks
    int rows;
    unsigned row_bytes;

    __device__ __forceinline__ static u32x4 describe(const void* ptr, unsigned range) {
        const unsigned long long base = reinterpret_cast<unsigned long long>(ptr);  // (48 bits: no stride in the second word)
        return u32x4{(unsigned)base, (unsigned)(base >> 32), range, BUFFER_WORD3};
    }
    __device__ __forceinline__ void init(const void* ptr, int64_t stride_bytes, int n_rows, int bytes_per_row) {
        stride = (unsigned)stride_bytes;
        rows = n_rows;
        row_bytes = (unsigned)bytes_per_row;
        desc = describe(ptr, (unsigned)(n_rows - 1) * stride + row_bytes);
    }
    // moves the view to another head of the same tensor
    __device__ __forceinline__ void move(int64_t bytes) {
        const unsigned long long base = (((unsigned long long)desc[1] << 32) | desc[0]) + (unsigned long long)bytes;
        desc[0] = (unsigned)base;
        desc[1] = (unsigned)(base >> 32);
    }
    __device__ __forceinline__ TileSrc at(int row) const {
        if (!FAR) return TileSrc{desc, (unsigned)row * stride};
        const unsigned long long base = (((unsigned long long)desc[1] << 32) | desc[0]) + (uint64_t)(unsigned)row * stride;
        const int left = rows - row;  // (a tile has up to 128 rows)
        return TileSrc{u32x4{(unsigned)base, (unsigned)(base >> 32), left >= 128 ? DMA_RANGE : (unsigned)(left - 1) * stride + row_bytes, BUFFER_WORD3}, 0u};
    }
};
// Lane l fetches 16 (4) bytes at src + voff and the hardware writes them to LDS byte address lds_base + 16 l (4 l).
// WAIT: wait states in front of the copy, less one.  A scalar register that a vector instruction has written (the reload of a
// spilled one) must not be read by a memory instruction within five wait states, and the compiler does not look into an asm
// statement.  Instantiations whose scalar registers spill in the loop pass 4 (COPY_WAIT); the others need the one state after
// the write of M0: waiting five everywhere costs 1.2 % (forward + backward of 1 x 8192 tokens, 32 / 8 heads, D 128: 1769 ->
// 1791 us).  tests/test_copy_hazard.py looks at every copy of the built library.
template <int WAIT>
__device__ __forceinline__ void copy_b128(const TileSrc& src, unsigned voff, unsigned lds_base) {
    asm volatile("s_nop %4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(src.desc), "s"(src.off),
                 "{m0}"(lds_base), "n"(WAIT)
                 : "memory");
}
template <int WAIT>
__device__ __forceinline__ void copy_b32(const TileSrc& src, unsigned voff, unsigned lds_base) {
    asm volatile("s_nop %4\n\tbuffer_load_dword %0, %1, %2 offen lds" ::"v"(voff), "s"(src.desc), "s"(src.off),
                 "{m0}"(lds_base), "n"(WAIT)
                 : "memory");
}
template <bool BIAS, bool LONG>
constexpr int COPY_WAIT = LONG || BIAS ? 4 : 0;

// All direct global-to-LDS copies this wave has issued have landed (pair with a barrier).
__device__ __forceinline__ void wait_async() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// All LDS accesses this wave has issued are complete.  The compiler puts this wait in front of a barrier by itself --
// except, as the generated code showed, in front of a barrier at the head of a loop that is reached over the back
// edge with LDS stores still in flight (the list rebuilt for the next pass over a long sequence: other waves then
// read the old count or old entries).  So whoever writes LDS ahead of such a barrier states the wait.
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// ROWS x D tile of 2-byte elements copied global -> LDS by THREADS threads, 16 bytes per lane.
// Full tiles use the direct global-to-LDS load (no staging registers, no LDS write
// instructions): a wave's 64 lanes fill 64 consecutive chunk slots of the LDS tile, so the
// XOR swizzle is applied on the SOURCE side -- lane `id` fetches the chunk that belongs in
// slot `id`.  `setup` fixes those source offsets once per kernel; `issue(i, ...)` emits copy
// instruction i of CPT so that callers can spread a tile's copies between other work.
// Row strides are limited to 2^23 elements by the host checks, so the offsets fit 32 bits.
// ZERO_PAD: chunks past the head dim become zero in LDS (whoever multiplies along the head dim has zeros in the other operand
// there, but zero times an infinity of chunk 0 would be a NaN in the score of a key whose weight is 0); otherwise their lanes
// fetch chunk 0 again.
template <int D, int ROWS, int THREADS, bool ZERO_PAD = false>
struct TileStage {
    static constexpr int NCH = LDS_COLS<D> / 8;
    static constexpr int CHUNKS = ROWS * NCH;
    static constexpr int CPT = (CHUNKS + THREADS - 1) / THREADS;
    static constexpr bool EXACT = (CHUNKS % THREADS) == 0;
    unsigned goff[CPT];
    int wave_first;  // first chunk slot this wave fills with instruction 0

    // chunks: how many 16-byte chunks a row has in global memory (d / 8); zero: the offset that reads zeros
    __device__ __forceinline__ void setup(int64_t row_stride_bytes, int chunks, int tid, unsigned zero = ROW_ZERO) {
        wave_first = __builtin_amdgcn_readfirstlane(tid & ~63);
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int id = tid + THREADS * i;
            const int row = id / NCH, pc = id % NCH;
            const int c = pc ^ swz<D>(row);
            goff[i] = ZERO_PAD && c >= chunks ? zero : (unsigned)(row * row_stride_bytes + (c < chunks ? c : 0) * 16);
        }
    }
    // tile_base: first row of the tile in global memory, tile_lds: lds_addr() of the LDS tile
    // (both wave-uniform)
    template <int SITE = 0>
    __device__ __forceinline__ void issue(int i, const char* tile_base, unsigned tile_lds) const {
        if (EXACT || wave_first + THREADS * i < CHUNKS) copy<SITE>(tile_base, goff[i], tile_lds + (unsigned)(THREADS * i + wave_first) * 16u);
    }
    template <int SITE = 0>
    static __device__ __forceinline__ void copy(const char* base, unsigned voff, unsigned lds_base) {
        if (ZERO_PAD)
            dma_b128_ranged<SITE>(base, voff, lds_base);
        else
            dma_b128<SITE>(base, voff, lds_base);
    }
    template <int WAIT>
    __device__ __forceinline__ void issue(int i, const TileSrc& src, unsigned tile_lds) const {
        if (EXACT || wave_first + THREADS * i < CHUNKS) copy_b128<WAIT>(src, goff[i], tile_lds + (unsigned)(THREADS * i + wave_first) * 16u);
    }
    __device__ __forceinline__ void load_full(const char* tile_base, unsigned tile_lds) const {
#pragma unroll
        for (int i = 0; i < CPT; ++i) issue(i, tile_base, tile_lds);
    }
    template <int WAIT>
    __device__ __forceinline__ void load(const TileSrc& src, unsigned tile_lds) const {
#pragma unroll
        for (int i = 0; i < CPT; ++i) issue<WAIT>(i, src, tile_lds);
    }
};

// 64-row tile made of two 32-row slices that sit anywhere in global memory: LDS rows [0, 32) come from slice
// `lo`, rows [32, 64) from slice `hi` (the LDS layout is that of TileStage<D, 64, THREADS>).  Every copy
// instruction of a wave covers 64 / (D / 8) <= 16 consecutive rows starting at a multiple of that, so it stays
// inside one slice and only its (wave-uniform) base pointer depends on which.
template <int D, int THREADS>
struct SliceStage {
    static constexpr int NCH = LDS_COLS<D> / 8;
    static constexpr int CHUNKS = 64 * NCH;
    static constexpr int CPT = (CHUNKS + THREADS - 1) / THREADS;
    static constexpr bool EXACT = (CHUNKS % THREADS) == 0;
    unsigned goff[CPT];
    int wave_first;  // first chunk slot this wave fills with instruction 0

    // chunks: how many 16-byte chunks a row has in global memory (d / 8)
    __device__ __forceinline__ void setup(int64_t row_stride_bytes, int chunks, int tid) {
        wave_first = __builtin_amdgcn_readfirstlane(tid & ~63);
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int id = tid + THREADS * i;
            const int row = id / NCH, pc = id % NCH;
            const int c = pc ^ swz<D>(row);
            goff[i] = (unsigned)((row & 31) * row_stride_bytes + (c < chunks ? c : 0) * 16);
        }
    }
    // Does copy instruction i of this wave fill LDS rows 32..63 (slice `hi`)?  Wave-uniform, and a compile-time
    // constant where every instruction covers whole 32-row halves (D = 128 with 512 threads).
    __device__ __forceinline__ bool upper(int i) const {
        if ((THREADS * (i + 1)) / NCH <= 32) return false;
        if ((THREADS * i) / NCH >= 32) return true;
        return (wave_first + THREADS * i) / NCH >= 32;
    }
    // Which row of the 64-row tile this lane copies with instruction i, and that copy with an offset of the caller's (sorted
    // rows: any row of the head; `setup` with a row stride of 0 leaves the offset inside a row in goff).
    static __device__ __forceinline__ int row(int i, int tid) { return (tid + THREADS * i) / NCH; }
    template <int WAIT>
    __device__ __forceinline__ void issue_gather(int i, const u32x4& desc, unsigned voff, unsigned tile_lds) const {
        if (EXACT || wave_first + THREADS * i < CHUNKS)
            copy_b128<WAIT>(TileSrc{desc, 0u}, voff, tile_lds + (unsigned)(THREADS * i + wave_first) * 16u);
    }
    // Copy instruction i from the first row of the slice it belongs to (see upper()).
    template <int WAIT>
    __device__ __forceinline__ void issue_from(int i, const TileSrc& slice, unsigned tile_lds) const {
        if (EXACT || wave_first + THREADS * i < CHUNKS)
            copy_b128<WAIT>(slice, goff[i], tile_lds + (unsigned)(THREADS * i + wave_first) * 16u);
    }
};

// Workgroup barrier that publishes LDS writes and leaves loads from memory in flight (the compiler's own barrier waits for them).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// The arrival of a load is pinned where this stands.  Left alone, the compiler waits for it at its first use inside the key
// loop, with a vmcnt that also (and every time round) drains the tile copies it does not know about.
template <int N>
__device__ __forceinline__ void arrived(u32x4 (&regs)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(regs[i]));
}

// The 32-row slice each of the four waves of a forward / dQ workgroup works on, and the row of tile classes
// (one byte per 32-key column tile: 0 empty, 1 partial, 2 full) that says which keys that slice needs.
// Without a plan the workgroup is a 128-row block in natural order and every wave reads the block's flag row;
// with one, group `grp` takes the next four slices of the sorted order and every slice has a class row of its own.
struct WaveSlices {
    int slice[4];             // -1: no slice (the wave idles through the key loop)
    bool moved;               // the rows of the slices are those of AttnParams::rows
    const int8_t* cls_row[4]; // null where slice is -1
};

// The query row at a place of the slice order's slices: the place itself, or with sorted rows whatever row was sorted there.
__device__ __forceinline__ int row_of_slot(const AttnParams& p, const WaveSlices& ws, int b, int slot, bool valid) {
    return ws.moved && valid ? p.rows[(int64_t)b * p.rows_sb + slot] : slot;
}

// A word of the plan at a wave-uniform address, by a scalar load (whatever stands in front of it).
__device__ __forceinline__ int plan_word(const int* at) {
    return *(const __attribute__((address_space(4))) int*)(unsigned long long)at;
}

// ONE_LOAD: the four codes in one load; left alone, the compiler waits for each before it asks for the next (0.5 us of a launch).
// Not with a bias, whose kernels spill scalars: dQ at D 32 over a bias matrix got 2 % slower.
template <bool ONE_LOAD = true>
__device__ __forceinline__ WaveSlices pick_wave_slices(const AttnParams& p, int b, int grp) {
    WaveSlices w;
    w.moved = false;
    if (p.fine != nullptr) {
        const int* ord = p.order + (int64_t)b * p.order_sb + 4 * grp;
        int code[4];
        if constexpr (ONE_LOAD) {
#pragma unroll
            for (int x = 0; x < 4; ++x) code[x] = plan_word(ord + x);
            asm volatile("" ::"s"(code[0]), "s"(code[1]), "s"(code[2]), "s"(code[3]));
        }
        w.moved = order_moved(ONE_LOAD ? code[0] : ord[0]);  // (a group has a first slice)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            w.slice[x] = order_slice(ONE_LOAD ? code[x] : ord[x]);
            w.cls_row[x] = w.slice[x] >= 0
                               ? (const int8_t*)p.fine + (int64_t)b * p.fine_sb + (int64_t)w.slice[x] * p.fine_ss
                               : nullptr;
        }
    } else {
        const int m = p.num_m - 1 - grp;  // late query blocks (most keys under causality) first
        const int8_t* row = p.flags + (int64_t)b * p.flags_sb + (int64_t)m * p.flags_sm;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            w.slice[x] = 4 * m + x;
            w.cls_row[x] = row;
        }
    }
    return w;
}

// Two streams, more workgroups than compute units: whether the streams take a unit each (level_heads).
__device__ __forceinline__ bool streams_side_by_side(const AttnParams& p) {
    const int groups = p.num_m * p.B;
    return p.group_order != nullptr && groups * p.Hq > 256 && p.Hq >= plan_word(p.group_order + groups);
}
// (units 8 apart are on the same XCD and, in head_unit_map, heads that read the same rows)
__device__ __forceinline__ int side_unit(int block, int stream) { return 16 * (block >> 3) + (block & 7) + 8 * stream; }

// The class bytes of 64-key tile kt (< nkt, or one that does not matter) for the four slices.  Without branches: the eight loads
// are on their way together, where each waited for the one before as long as slices that are not there were skipped.
struct TileClasses {
    int f[4][2];
};
__device__ __forceinline__ TileClasses load_tile_classes(const WaveSlices& ws, int num_n, int nkt, int kt) {
    TileClasses c;
    const int at = 2 * max(min(kt, nkt - 1), 0), second = min(at + 1, num_n - 1);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const int8_t* row = ws.cls_row[x] != nullptr ? ws.cls_row[x] : ws.cls_row[0];  // (a group has a first slice)
        c.f[x][0] = row[at];
        c.f[x][1] = row[second];
    }
    return c;
}
__device__ __forceinline__ int key_tiles(int S, int kt_begin) { return min((S + 63) >> 6, kt_begin + MAX_LIST); }

// List, in ascending order, the 64-key tiles the four slices of a workgroup have to visit, among the (at most
// MAX_LIST) tiles starting at tile kt_begin; longer sequences are walked in several passes.
// entry = (tile << 8) | c0 | c1 << 2 | c2 << 4 | c3 << 6 ; c_w is the class of the tile for wave w's slice:
// 0 nothing to do, 1 evaluate the mask, 2 every pair allowed.
// A tile is "full" for a slice only when both of its 32-column classes say so AND it has no column past
// the end of the sequence (those columns must still be masked out of the softmax).
// Executed by wave 0; the caller synchronizes before reading.
// first: load_tile_classes of this lane's first tile.  The classes of the next 64 tiles are asked for before those at hand are
// looked at.
// STREAMS = 2: the even and the odd tiles make a list each (the second at list + MAX_LIST / 2, its length in count_out[1]).  Which
// list a tile is in does not depend on what else is listed, so the tiles of a slice are added up in the same order whatever group or
// plan it is in.  (split false: one list all the same.)
template <int STREAMS = 1>
__device__ __forceinline__ void build_key_tile_list(const WaveSlices& ws, int num_n, int S, int lane, int kt_begin, const TileClasses& first,
                                                    int* list, int* count_out, bool split = STREAMS > 1) {
    const int nkt = key_tiles(S, kt_begin);
    int count[STREAMS] = {};
    const int mine = STREAMS > 1 && split ? lane & 1 : 0;  // (kt_begin is even)
    const unsigned long long even = split ? 0x5555555555555555ull : ~0ull;
    TileClasses cur = first;
    for (int base = kt_begin; base < nkt; base += 64) {
        const TileClasses next = load_tile_classes(ws, num_n, nkt, base + 64 + lane);
        const int kt = base + lane;
        const bool second = 2 * kt + 1 < num_n, inside = (kt + 1) * 64 <= S;
        int packed = 0;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int f0 = cur.f[x][0], f1 = second ? cur.f[x][1] : 0;
            int cls = 0;
            if (f0 > 0 || f1 > 0) cls = (f0 == 2 && f1 == 2 && inside) ? 2 : 1;
            packed |= ws.cls_row[x] != nullptr ? cls << (2 * x) : 0;
        }
        if (kt >= nkt) packed = 0;
        unsigned long long bal = __ballot(packed != 0), own = bal;
        if (STREAMS > 1) own &= mine ? ~even : even;
        const int at = (mine ? MAX_LIST / 2 + count[STREAMS - 1] : count[0]) + __popcll(own & ((1ull << lane) - 1ull));
        if (packed) list[at] = (kt << 8) | packed;
#pragma unroll
        for (int x = 0; x < STREAMS; ++x)
            count[x] += __popcll(STREAMS == 1 ? bal : bal & (x ? ~even : even));
        cur = next;
    }
#pragma unroll
    for (int x = 0; x < STREAMS; ++x)
        if (lane == 0 && (x == 0 || split)) count_out[x] = count[x];
    wait_lds();
}

// The four class bytes (key columns 4 nt ..) of slice s (< s_end, or one that does not matter), low byte first.
__device__ __forceinline__ unsigned load_slice_classes(const AttnParams& p, int b, int nt, int s, int s_end) {
    s = max(min(s, s_end - 1), 0);
    const int8_t* f = p.fine != nullptr ? (const int8_t*)p.fine + (int64_t)b * p.fine_sb + (int64_t)s * p.fine_ss
                                        : p.flags + (int64_t)b * p.flags_sb + (int64_t)(s >> 2) * p.flags_sm;
    if (p.fine_words) return *(const unsigned*)(f + 4 * nt);
    unsigned c = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) c |= (unsigned)(f[min(4 * nt + w, p.num_n - 1)] & 3) << (8 * w);
    return c;
}

// List, in ascending order, the 32-row slices among [s_begin, s_end) (at most MAX_SLICE_LIST of them; longer
// sequences are walked in several passes) that have work for a 128-key tile (4 class columns).
// entry = (slice << 8) | c0 | c1 << 2 | c2 << 4 | c3 << 6, c_w = class of (slice, key column 4 nt + w).
// With a plan the classes are those of the 32 x 32 tiles; without one a slice inherits the flags of its
// 128-row block.
// first: load_slice_classes of this lane's first slice.
__device__ __forceinline__ void build_slice_list(const AttnParams& p, int b, int nt, int lane, int s_begin, int s_end, unsigned first,
                                                 int* list, int* count_out) {
    const int ns = s_end;
    int count = 0;
    unsigned cur = first;
    for (int base = s_begin; base < ns; base += 64) {
        const unsigned next = load_slice_classes(p, b, nt, base + 64 + lane, ns);
        const int s = base + lane;
        int packed = 0;
        if (s < ns) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                int fw = (4 * nt + w < p.num_n) ? (int)(cur >> (8 * w)) & 3 : 0;
                if ((s + 1) * 32 > p.Sq) fw = min(fw, 1);  // rows past the end have to be masked out
                packed |= fw << (2 * w);
            }
        }
        const unsigned long long bal = __ballot(packed != 0);
        if (packed) list[count + __popcll(bal & ((1ull << lane) - 1ull))] = (s << 8) | packed;
        count += __popcll(bal);
        cur = next;
    }
    // list[-1] (the caller leaves room for it) repeats the first entry with all classes cleared: a consumer that
    // takes the entries in pairs from the end finds a harmless partner for the first entry of an odd count there.
    if (lane == 0) {
        *count_out = count;
        if (count > 0) list[-1] = list[0] & ~0xFF;
    }
    wait_lds();
}

}  // namespace bam
