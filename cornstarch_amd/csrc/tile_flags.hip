// Tile-summary kernel: int64 bitfields -> int8 flag per (128-row, 32-column) tile, and the
// dense-mask utility.  Integer work only; results are bit exact by construction.
// Reference: cornstarch/kernel/bitfield_attention.py:60-156.
#include "bam_common.h"
#include "bam_launch.h"
#include <type_traits>

namespace bam {

// One workgroup = one 128-row block x FLAG_COLS_PER_BLOCK key tiles.  Each wave takes one
// 128x32 tile at a time: lane l owns key column (l & 31) and the 64 query rows of half
// (l >> 5); the per-lane counts are summed over the wave.
// Shortcut: when the 128 rows carry one bitfield and the 32 columns carry one bitfield (and the
// tile lies inside the sequence) the class follows from one evaluation of the bit test plus the
// position of the tile relative to the diagonal; long runs of equal bitfields are the common case.
constexpr int FLAG_WAVES = 4;
constexpr int FLAG_TILES_PER_WAVE = 2;  // few tiles per wave: the grid, not the wave, covers the row of tiles
constexpr int FLAG_COLS_PER_BLOCK = FLAG_WAVES * FLAG_TILES_PER_WAVE;
constexpr int FLAG_MAX_BLOCKS_X = 64;  // workgroups per 128-row block; longer rows of tiles are walked in a loop

// ---------------------------------------------------------------------------------------------------------
// Slice order.  The forward and dQ kernels give each of the four waves of a workgroup one 32-row slice and walk
// the union of the key tiles those slices need, so four slices that need the same keys should sit together:
//   * slices holding a text row first, by descending position (they see their whole past; the latest see most),
//   * then the slices made of modality rows only, grouped by the OR of their bitfields (equal value = same
//     modality = same keys), by ascending position inside a group.
// Every slice gets a two-word sort key and is ranked against all others of its sequence (at most
// MAX_PLAN_SLICES of them); slots past the last slice are set to -1.  The work rides in the launch of the flag
// kernel, as extra workgroups of its grid (it needs the bitfields only): workgroup `part` of sequence b ranks
// slices [64 part, +64).
// Ranks the slices [64 part, +64) of one sequence among all `ns` slices by two-word keys (distinct for distinct
// slices; slices >= ns get the largest key) and writes order_row[rank] = slice; the slots past the last slice are set
// to -1.  `fill(base, sk)` puts the keys of slices [base, min(base + 256, ns)) into sk[2 i], sk[2 i + 1] (all 256 threads
// take part).  Four threads share a slice and compare it with a quarter of every chunk each, eight keys per step, so that
// the loop runs at the rate of the LDS and not at its latency.  (With one thread per slice and whole chunks of 256 keys
// whatever the length, this column of workgroups was what the launch waited for: 11 us of it at 283 tokens.)
constexpr int RANKED_PER_GROUP = 64;
typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
template <typename FillFn>
__device__ __forceinline__ void slice_order_ranked(FillFn fill, int ns, int slots, int part, int* __restrict__ order_row, int mark = 0) {
    __shared__ __attribute__((aligned(16))) unsigned long long sk[2 * 256];
    const int tid = threadIdx.x, s = part * RANKED_PER_GROUP + (tid >> 2), sub = tid & 3;
    unsigned long long my1 = 0, my2 = 0;
    int rank = 0;
    // the chunk that holds this workgroup's own slices first (their keys are what the others are compared with)
    const int own = part * RANKED_PER_GROUP / 256, nchunks = max(own + 1, (ns + 255) / 256);
    for (int c = 0; c < nchunks; ++c) {
        const int base = 256 * (c == 0 ? own : c <= own ? c - 1 : c), n = min(256, ns - base);
        __syncthreads();
        fill(base, sk);
        // the last step of eight reads past the last key
        if (tid < 32 && n + tid < 256 && n + tid < ((max(n, 0) + 31) & ~31)) sk[2 * (n + tid)] = sk[2 * (n + tid) + 1] = ~0ull;
        __syncthreads();
        if (c == 0) {
            my1 = sk[2 * (s & 255)];
            my2 = sk[2 * (s & 255) + 1];
        }
        for (int j0 = 8 * sub; j0 < n; j0 += 32) {  // entries past the last slice hold the largest key: never smaller
            u64x2 o[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) o[u] = *(const u64x2*)&sk[2 * (j0 + u)];
#pragma unroll
            for (int u = 0; u < 8; ++u) rank += (o[u][0] < my1 || (o[u][0] == my1 && o[u][1] < my2)) ? 1 : 0;
        }
    }
    rank += __shfl_xor(rank, 1);
    rank += __shfl_xor(rank, 2);
    if (sub != 0) return;
    if (s < ns)
        order_row[rank] = s | mark;
    else if (s < slots)
        order_row[s] = -1;
}

// OR over the 16 lanes of a DPP row, result in every lane (quad swaps, then the two mirror patterns).
__device__ __forceinline__ unsigned row_or(unsigned x) {
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, false);  // row_half_mirror
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x140, 0xF, 0xF, false);  // row_mirror
    return x;
}

// Keys of slices [base, base + 256) from the bitfields (k1 = 0 for a slice with a text row, else bit 62 + the OR of
// its bitfields; k2 = the position rank inside the class), read in order: 16 lanes take the 32 rows of one slice (two
// each) and OR them together; bit 0 of the OR says whether the slice holds a text row.
__device__ __forceinline__ void slice_keys_chunk(const int64_t* __restrict__ row, int S, int ns, int base,
                                                 unsigned long long* sk) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t M = (((int64_t)1) << 62) - 1;
    const int n = min(256, ns - base);
    for (int s0 = 0; s0 < n; s0 += 128) {  // eight slices per 16 lanes at a time: one memory latency for 128 slices
        uint64_t f[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = (base + s0 + 16 * u + 4 * wave + (lane >> 4)) * 32 + 2 * (lane & 15);
            f[u] = (uint64_t)((i < S ? row[i] : 0) | (i + 1 < S ? row[i + 1] : 0));
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int local = s0 + 16 * u + 4 * wave + (lane >> 4), s = base + local;  // local: slice within the chunk
            const unsigned lo = row_or((unsigned)f[u]), hi = row_or((unsigned)(f[u] >> 32));
            if ((lane & 15) == 0 && local < n) {
                const bool text = (lo & 1u) != 0;
                const unsigned long long sig = (((unsigned long long)hi << 32) | lo) & (unsigned long long)M;
                sk[2 * local] = text ? 0ull : (1ull << 62) | sig;
                sk[2 * local + 1] = text ? (unsigned long long)(ns - 1 - s) : (unsigned long long)s;
            }
        }
    }
}

__device__ __forceinline__ void slice_order_part(const int64_t* __restrict__ row, int S, int part,
                                                 int* __restrict__ order_row) {
    const int ns = (S + 31) / 32, slots = 4 * ((S + BLOCK_M - 1) / BLOCK_M);
    slice_order_ranked([&](int base, unsigned long long* sk) { slice_keys_chunk(row, S, ns, base, sk); }, ns, slots, part,
                       order_row);
}

// The same ordering idea for index-tensor attention, where a local row's position is pos[row]: slices holding a
// text row first, by descending largest position; then modality-only slices grouped by the OR of their bitfields,
// by ascending smallest position.  The slice number in the low bits keeps the keys distinct whatever the positions.
__device__ __forceinline__ int row_max(int x) {  // over the 16 lanes of a DPP row, result in every lane
    x = max(x, __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false));
    x = max(x, __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false));
    return max(x, __builtin_amdgcn_mov_dpp(x, 0x140, 0xF, 0xF, false));
}
// Bitfields and positions of the local rows (or keys): gathered arrays, or -- for the launch that does the gathering --
// the global bitfields seen through an index tensor.
struct GatheredRows {
    const int64_t* bits;
    const int* positions;
    __device__ __forceinline__ void get(int i, int64_t& f, int& pos) const {
        f = bits[i];
        pos = positions != nullptr ? positions[i] : i;
    }
};
struct IndexedRows {
    const int64_t* bf;
    const int64_t* idx;
    int L;
    __device__ __forceinline__ void get(int i, int64_t& f, int& pos) const {
        const int64_t p = idx[i];
        f = (p >= 0 && p < L) ? bf[p] : 0;
        pos = (int)(p < 0 ? 0 : p > 0x7FFFFFFE ? 0x7FFFFFFE : p);
    }
};

template <typename Rows>
__device__ __forceinline__ void slice_keys_chunk_indexed(const Rows& rows, int S, int ns, int base, unsigned long long* sk) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t M = (((int64_t)1) << 62) - 1;
    const int n = min(256, ns - base);
    for (int s0 = 0; s0 < n; s0 += 64) {
        int64_t f[4][2];
        int p[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int i = (base + s0 + 16 * u + 4 * wave + (lane >> 4)) * 32 + 2 * (lane & 15) + x;
                f[u][x] = 0;
                p[u][x] = -1;  // no such row
                if (i < S) rows.get(i, f[u][x], p[u][x]);
            }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int local = s0 + 16 * u + 4 * wave + (lane >> 4), s = base + local;
            const uint64_t both = (uint64_t)(f[u][0] | f[u][1]);
            const unsigned lo = row_or((unsigned)both), hi = row_or((unsigned)(both >> 32));
            const int hi_pos = max(0, row_max(max(p[u][0], p[u][1])));
            const int first = p[u][0] < 0 ? 0x7FFFFFFF : p[u][1] < 0 ? p[u][0] : min(p[u][0], p[u][1]);
            const int lo_pos = -row_max(-first);
            if ((lane & 15) == 0 && local < n) {
                const bool text = (lo & 1u) != 0;
                const unsigned long long sig = (((unsigned long long)hi << 32) | lo) & (unsigned long long)M;
                sk[2 * local] = text ? 0ull : (1ull << 62) | sig;
                sk[2 * local + 1] = ((unsigned long long)(text ? 0x7FFFFFFF - hi_pos : lo_pos) << 20) | (unsigned long long)s;
            }
        }
    }
}

// Sorted rows: text rows by position, then the modality rows grouped by their bitfield, by position inside a group, then
// padding.  A counting sort over 64 classes; different bitfields may share a class (only the packing of the slices suffers).  A
// workgroup of 256 threads places 1024 rows of one sequence; it counts the classes of all rows for itself (512 KiB of bitfields out
// of L2 for 65536 rows, eight loads in flight per thread) instead of waiting for the others, beside the workgroups that compute
// the flags, which take longer (17000 rows: 20.3 us with and 19.6 without; 28.8 when it took 64 rows of one bitfield one by one).
// Rows are only moved where at least one slice in SORT_MIXED holds text and modality rows: dK/dV gathers moved rows one by one,
// which costs it 3 %.  Training step, 32 / 8 heads, D 128, natural -> sorted: 65536 tokens, 200 segments (20 % of the slices
// mixed) 64.3 -> 48.2 ms; 8192 tokens, 30 segments (23 %) 1.87 -> 1.68 ms, 4 segments (3 %) 1.717 -> 1.722 ms; 16384 tokens, 4
// segments (1.6 %) 7.36 -> 7.46 ms.
constexpr int SORT_CHUNK = 1024, SORT_CLASSES = 64, SORT_MIXED = 32;
struct SortedRows {
    int* rows;           // null: not asked for
    int64_t* rows_bits;
    int64_t rows_sb;
    int* rows_moved;
};
__device__ __forceinline__ int sort_class(int64_t f) {
    const uint64_t bits = (uint64_t)f & ((1ull << 62) - 1ull);
    if (bits & 1) return 0;
    if (bits == 0) return SORT_CLASSES - 1;
    if ((bits & (bits - 1)) == 0) return 1 + (__ffsll((long long)bits) - 1) % (SORT_CLASSES - 2);
    return 1 + (int)((bits * 0x9E3779B97F4A7C15ull) >> 40) % (SORT_CLASSES - 2);
}
// f(class, lanes that hold it) for every class among the wave's lanes (cls < 0: none)
template <typename F>
__device__ __forceinline__ void each_class(int cls, F f) {
    unsigned long long left = __ballot(cls >= 0);
    while (left != 0) {  // wave-uniform
        const int c = __builtin_amdgcn_readlane(cls, __builtin_ctzll(left));
        const unsigned long long same = __ballot(cls == c);
        f(c, same);
        left &= ~same;
    }
}
__device__ void sort_rows_part(const int64_t* __restrict__ row, int S, int S_rounded, int part, int b, const SortedRows& out) {
    constexpr int THREADS = FLAG_WAVES * 64, GROUPS = SORT_CHUNK / 64;
    __shared__ int s_mixed, s_total[SORT_CLASSES], s_before[SORT_CLASSES], s_base[SORT_CLASSES];
    __shared__ int s_group[GROUPS][SORT_CLASSES];  // rows of a class in each run of 64 rows, then in front of it
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int first = part * SORT_CHUNK;
    if (tid == 0) s_mixed = 0;
    if (tid < SORT_CLASSES) s_total[tid] = s_before[tid] = 0;
    for (int i = tid; i < GROUPS * SORT_CLASSES; i += THREADS) s_group[0][i] = 0;
    __syncthreads();
    int mixed = 0;  // slices (in natural order) that hold text and modality rows, among those this wave has looked at
    // 64 rows of one bitfield (most of them are) only add to the counts of the run they belong to
    int64_t run_bits = 0;
    int run_total = 0, run_before = 0;
    auto end_run = [&]() {
        if (run_total > 0 && lane == 0) {
            const int c = sort_class(run_bits);
            atomicAdd(&s_total[c], run_total);
            if (run_before > 0) atomicAdd(&s_before[c], run_before);
        }
        run_total = run_before = 0;
    };
    constexpr int AHEAD = 8;
    for (int i0 = 0; i0 < S; i0 += AHEAD * THREADS) {
        int64_t f[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int i = i0 + u * THREADS + tid;
            f[u] = i < S ? row[i] : 0;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int run = i0 + u * THREADS, i = run + tid;
            const int64_t f0 = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)f[u]) |
                               (int64_t)__builtin_amdgcn_readfirstlane((int)(f[u] >> 32)) << 32;
            if (run + wave * 64 + 64 <= S && __all(f[u] == f0)) {
                if (f0 != run_bits) {
                    end_run();
                    run_bits = f0;
                }
                run_total += 64;
                run_before += run < first ? 64 : 0;
                continue;
            }
            const int cls = i < S ? sort_class(f[u]) : -1;
            const unsigned long long text = __ballot(cls == 0), modal = __ballot(cls > 0 && cls < SORT_CLASSES - 1);
            mixed += ((unsigned)text != 0 && (unsigned)modal != 0) + ((text >> 32) != 0 && (modal >> 32) != 0);
            each_class(cls, [&](int c, unsigned long long same) {
                if (lane == 0) {
                    atomicAdd(&s_total[c], __popcll(same));
                    if (run < first) atomicAdd(&s_before[c], __popcll(same));
                }
            });
        }
    }
    end_run();
    if (lane == 0) atomicAdd(&s_mixed, mixed);
    int64_t f[GROUPS / FLAG_WAVES];
    int cls[GROUPS / FLAG_WAVES], earlier[GROUPS / FLAG_WAVES];
#pragma unroll
    for (int u = 0; u < GROUPS / FLAG_WAVES; ++u) {
        const int mine = first + u * THREADS + tid;
        f[u] = mine < S ? row[mine] : 0;
        cls[u] = mine < S ? sort_class(f[u]) : -1;
        earlier[u] = 0;  // rows of my class in front of me in the run of 64
        each_class(cls[u], [&](int c, unsigned long long same) {
            if (lane == 0) s_group[u * FLAG_WAVES + wave][c] = __popcll(same);
            if (cls[u] == c) earlier[u] = __popcll(same & ((1ull << lane) - 1ull));
        });
    }
    __syncthreads();
    if (tid < SORT_CLASSES) {
        int base = 0;
        for (int c = 0; c < tid; ++c) base += s_total[c];
        s_base[tid] = base + s_before[tid];
        int before = 0;
        for (int g = 0; g < GROUPS; ++g) {
            const int n = s_group[g][tid];
            s_group[g][tid] = before;
            before += n;
        }
    }
    __syncthreads();
    const bool move = s_mixed * SORT_MIXED >= (S + 31) / 32;
    if (part == 0 && tid == 0) out.rows_moved[b] = move ? 1 : 0;
#pragma unroll
    for (int u = 0; u < GROUPS / FLAG_WAVES; ++u) {
        const int mine = first + u * THREADS + tid;
        if (mine < S) {
            const int64_t at = (int64_t)b * out.rows_sb + (move ? s_base[cls[u]] + s_group[u * FLAG_WAVES + wave][cls[u]] + earlier[u] : mine);
            out.rows[at] = mine;
            out.rows_bits[at] = f[u];
        } else if (mine < S_rounded) {
            out.rows[(int64_t)b * out.rows_sb + mine] = S;
            out.rows_bits[(int64_t)b * out.rows_sb + mine] = 0;
        }
    }
}

// FINE: also write the class of every 32-row x 32-column tile (the four row slices of each flag tile) to
// fine[b][4 m + w][n]; same 0 / 1 / 2 meaning, "full" again over the in-range cells only.
template <bool FINE>
__global__ __launch_bounds__(FLAG_WAVES * 64) void tile_flags_kernel(const int64_t* __restrict__ bf,
                                                                    int64_t bf_stride_b,
                                                                    int8_t* __restrict__ flags,
                                                                    int64_t flags_stride_b,
                                                                    int64_t flags_stride_m, int S, int num_n,
                                                                    uint8_t* __restrict__ fine, int64_t fine_sb,
                                                                    int64_t fine_ss, int* __restrict__ order,
                                                                    int64_t order_sb, int flag_blocks_x,
                                                                    int flag_groups, int* __restrict__ pair_count,
                                                                    SortedRows sorted) {
    // (the pair counter of the numbering kernel that follows in the stream starts from zero)
    if (FINE && pair_count != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0)
        *pair_count = 0;
    if (FINE && (int)blockIdx.x > flag_blocks_x) {  // the workgroups that sort the rows
        const int S_rounded = (int)gridDim.y * BLOCK_M;
        if ((int)blockIdx.y * SORT_CHUNK < S_rounded)
            sort_rows_part(bf + (int64_t)blockIdx.z * bf_stride_b, S, S_rounded, blockIdx.y, blockIdx.z, sorted);
        return;
    }
    if (FINE && (int)blockIdx.x >= flag_blocks_x) {  // the workgroups that sort the slices (see slice_order_part)
        const int part = blockIdx.y;
        if (part * RANKED_PER_GROUP < 4 * (int)gridDim.y)
            slice_order_part(bf + (int64_t)blockIdx.z * bf_stride_b, S, part, order + (int64_t)blockIdx.z * order_sb);
        return;
    }
    __shared__ int64_t q_bits[BLOCK_M];
    // classes of this workgroup's eight column tiles: row 0 the flag, rows 1..4 the four row slices; written out
    // together at the end (eight bytes per row in one store where the layout guarantees alignment)
    // (two copies: a workgroup that takes several groups of column tiles fills one while the other is stored)
    __shared__ __attribute__((aligned(8))) uint8_t s_out_buf[2][5][FLAG_COLS_PER_BLOCK];
    const int b = blockIdx.z, m = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t* row = bf + (int64_t)b * bf_stride_b;
    // the key bitfields of both tiles of this wave, requested together (one memory latency instead of one per tile), and
    // for the first group before the workgroup waits for its row bitfields
    const int half = lane >> 5, l32 = lane & 31;
    int64_t kfs[FLAG_TILES_PER_WAVE];
    auto request_keys = [&](int bx) {
#pragma unroll
        for (int t = 0; t < FLAG_TILES_PER_WAVE; ++t) {
            const int j = (bx * FLAG_COLS_PER_BLOCK + wave * FLAG_TILES_PER_WAVE + t) * BLOCK_N + l32;
            kfs[t] = (j < S) ? row[j] : 0;
        }
    };
    request_keys(blockIdx.x);
    if (tid < BLOCK_M) {
        const int i = m * BLOCK_M + tid;
        q_bits[tid] = (i < S) ? row[i] : 0;  // out-of-range positions read 0 (reference :86-87)
    }
    __syncthreads();
    const int rows_in_range = min(BLOCK_M, S - m * BLOCK_M);
    // Runs of equal bitfields inside each of the four 32-row slices: bit r of slice_starts[w] = row r starts a run
    // (rows past the end of the sequence read 0 and make a run of their own).  The count of a column over a run
    // follows from one evaluation of the bit test, so a tile costs one evaluation per run, not one per row.
    int64_t slice_q[4];
    unsigned slice_starts[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        slice_q[w] = q_bits[32 * w];
        slice_starts[w] = (unsigned)__ballot(l32 == 0 || q_bits[32 * w + l32] != q_bits[32 * w + max(l32, 1) - 1]);
    }
    const int64_t q0 = slice_q[0];
    const bool rows_uniform = rows_in_range == BLOCK_M && slice_starts[0] == 1u && slice_starts[1] == 1u &&
                              slice_starts[2] == 1u && slice_starts[3] == 1u && slice_q[1] == q0 && slice_q[2] == q0 &&
                              slice_q[3] == q0;
    // A workgroup takes the groups of eight column tiles bx = blockIdx.x, blockIdx.x + flag_blocks_x, ...: one group
    // for sequences of up to 16384 keys, several for longer ones (the setup above is then paid once).
    int it = 0;
    for (int bx = blockIdx.x; bx < flag_groups; bx += flag_blocks_x, ++it) {
        uint8_t (*s_out)[FLAG_COLS_PER_BLOCK] = s_out_buf[it & 1];
        if (tid < 5 * FLAG_COLS_PER_BLOCK) s_out[0][tid] = 0;
        __syncthreads();
        static_assert(FLAG_TILES_PER_WAVE == 2, "the counting path gives each half of a wave one tile");
        if (it > 0) request_keys(bx);
        bool counted[FLAG_TILES_PER_WAVE];  // wave-uniform: the tile still needs the counting path
#pragma unroll
        for (int t = 0; t < FLAG_TILES_PER_WAVE; ++t) {
            const int n = bx * FLAG_COLS_PER_BLOCK + wave * FLAG_TILES_PER_WAVE + t;
            counted[t] = n < num_n;
            if (n >= num_n) continue;  // wave-uniform
            const int64_t kf = kfs[t];
            if (rows_uniform && (n + 1) * BLOCK_N <= S) {
                const unsigned klo = __builtin_amdgcn_readfirstlane((unsigned)kf);
                const unsigned khi = __builtin_amdgcn_readfirstlane((unsigned)((uint64_t)kf >> 32));
                const int64_t k0 = (int64_t)(((uint64_t)khi << 32) | klo);
                if (__all(kf == k0)) {
                    const int64_t M = (((int64_t)1) << 62) - 1;
                    const int64_t qb = q0 & M, kb = k0 & M;
                    int8_t f;
                    const int r0 = m * BLOCK_M, c0 = n * BLOCK_N;
                    if (q0 & 1) {  // text rows: causal over keys that share a bit
                        f = (qb & kb) == 0 ? 0 : r0 >= c0 + BLOCK_N - 1 ? 2 : r0 + BLOCK_M - 1 < c0 ? 0 : 1;
                    } else {
                        f = (qb == kb && qb != 0) ? 2 : 0;
                    }
                    const int col = wave * FLAG_TILES_PER_WAVE + t;
                    if (lane == 0) s_out[0][col] = (uint8_t)f;
                    if (FINE && lane < 4) {  // the same closed form for the 32 rows of slice `lane`
                        const int rs = r0 + 32 * lane;
                        int8_t fw = f;
                        if (q0 & 1) fw = (qb & kb) == 0 ? 0 : rs >= c0 + BLOCK_N - 1 ? 2 : rs + 31 < c0 ? 0 : 1;
                        s_out[1 + lane][col] = (uint8_t)fw;
                    }
                    counted[t] = false;
                }
            }
        }
        if (counted[0] || counted[1]) {
            // Counting path, both tiles at once: lanes [0, 32) own the columns of tile 0, lanes [32, 64) those of tile 1.
            const int t = half;
            const int n = bx * FLAG_COLS_PER_BLOCK + wave * FLAG_TILES_PER_WAVE + t;
            const int j = n * BLOCK_N + l32;
            const int64_t kf = half ? kfs[1] : kfs[0];
            const int64_t M = (((int64_t)1) << 62) - 1;
            const int64_t kb = kf & M;
            int cnt[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int r0 = m * BLOCK_M + 32 * w;
                unsigned starts = slice_starts[w];  // wave-uniform, bit 0 set
                int c = 0;
                while (starts != 0u) {
                    const int a = __builtin_ctz(starts);
                    starts &= starts - 1u;
                    const int e = starts != 0u ? __builtin_ctz(starts) : 32;  // the run is rows [a, e) of the slice
                    const int64_t qf = q_bits[32 * w + a];
                    const int64_t qb = qf & M;
                    if (qf & 1)  // text rows: those at or after column j (reference :93-97)
                        c += (qb & kb) != 0 ? min(e - a, max(0, r0 + e - max(r0 + a, j))) : 0;
                    else
                        c += (qb == kb && qb != 0) ? e - a : 0;
                }
                cnt[w] = c;
            }
#pragma unroll
            for (int off = 16; off > 0; off >>= 1)  // over the 32 columns, inside each half of the wave
#pragma unroll
                for (int w = 0; w < 4; ++w) cnt[w] += __shfl_xor(cnt[w], off);
            const bool mine = half ? counted[1] : counted[0];
            if (l32 == 0 && mine) {
                const int cols_in_range = min(BLOCK_N, S - n * BLOCK_N);
                const int col = wave * FLAG_TILES_PER_WAVE + t;
                if (FINE) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int rows = max(0, min(32, S - (m * BLOCK_M + 32 * w)));
                        s_out[1 + w][col] = (uint8_t)(cnt[w] == 0 ? 0 : cnt[w] == rows * cols_in_range ? 2 : 1);
                    }
                }
                const int total = cnt[0] + cnt[1] + cnt[2] + cnt[3];
                // full over in-range cells (:149-153)
                s_out[0][col] = (uint8_t)(total == 0 ? 0 : total == rows_in_range * cols_in_range ? 2 : 1);
            }
        }
        __syncthreads();
        const int n0 = bx * FLAG_COLS_PER_BLOCK;
        if (tid < FLAG_COLS_PER_BLOCK && n0 + tid < num_n)  // the flag row may start anywhere: single bytes
            flags[(int64_t)b * flags_stride_b + (int64_t)m * flags_stride_m + n0 + tid] = (int8_t)s_out[0][tid];
        if (FINE && tid >= 64 && tid < 68) {  // rows of the class matrix are padded to 16 bytes: one 8-byte store
            static_assert(FLAG_COLS_PER_BLOCK == 8, "one 64-bit word per row");
            const int w = tid - 64;
            *(unsigned long long*)(fine + (int64_t)b * fine_sb + (int64_t)(4 * m + w) * fine_ss + n0) =
                *(const unsigned long long*)s_out[1 + w];
        }
    }
}

__global__ __launch_bounds__(256) void materialize_mask_kernel(const int64_t* __restrict__ bf,
                                                               int64_t bf_stride_b,
                                                               uint8_t* __restrict__ out, int S) {
    const int b = blockIdx.z, i = blockIdx.y;
    const int64_t* row = bf + (int64_t)b * bf_stride_b;
    const int64_t qf = row[i];
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < S; j += gridDim.x * blockDim.x)
        out[((int64_t)b * S + i) * S + j] = allow_rule(qf, row[j], i, j) ? 1 : 0;
}

// Index-tensor attention, step 0: the bitfield and the 32-bit position of every local row (or key),
// out_bits[b][i] = bf[b][idx[i]] (0 when idx[i] is outside [0, L)), out_pos[i] = idx[i].
// Restates the index branch of the reference's mask block (bitfield_attention.py:71-87), hoisted out
// of the attention kernels so that they read both with unit stride.
__global__ __launch_bounds__(256) void gather_bitfields_kernel(const int64_t* __restrict__ bf, int64_t bf_stride_b,
                                                               int L, const int64_t* __restrict__ idx, int n,
                                                               int64_t* __restrict__ out_bits,
                                                               int64_t out_stride_b, int* __restrict__ out_pos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (i >= n) return;
    const int64_t pos = idx[i];
    const bool inside = pos >= 0 && pos < L;
    out_bits[(int64_t)b * out_stride_b + i] = inside ? bf[(int64_t)b * bf_stride_b + pos] : 0;
    if (b == 0) out_pos[i] = (int)(pos < 0 ? 0 : pos > 0x7FFFFFFE ? 0x7FFFFFFE : pos);
}

int launch_gather_bitfields(const int64_t* bf, int64_t bf_stride_b, int L, const int64_t* idx, int n, int64_t* out_bits,
                            int64_t out_stride_b, int* out_pos, int B, hipStream_t stream) {
    dim3 grid((n + 255) / 256, B);
    hipLaunchKernelGGL(gather_bitfields_kernel, grid, dim3(256), 0, stream, bf, bf_stride_b, L, idx, n, out_bits,
                       out_stride_b, out_pos);
    return (int)hipGetLastError();
}

// Tile flags of a materialized bool mask (B, Sq, Sk), one byte per pair: the same 0 / 1 / 2 classification
// over 128 x 32 tiles that the bitfield path uses, so that the attention kernels skip empty tiles and
// read the mask only in partial ones.  (The reference's materialized-mask kernel decides per tile, inside
// the attention loop, whether anything is unmasked: cornstarch/kernel/attention.py:188-200.)
// One workgroup = one row block x 8 column tiles; thread = one column, 128 rows, coalesced byte reads.
__global__ __launch_bounds__(256) void mask_tile_flags_kernel(const uint8_t* __restrict__ mask, int8_t* __restrict__ flags,
                                                              int64_t flags_stride_b, int64_t flags_stride_m, int Sq,
                                                              int Sk, int num_n) {
    const int b = blockIdx.z, m = blockIdx.y, tid = threadIdx.x;
    const int col = blockIdx.x * 256 + tid;
    const int r0 = m * BLOCK_M, r1 = min(r0 + BLOCK_M, Sq);
    int count = 0;
    if (col < Sk) {
        const uint8_t* pcol = mask + (int64_t)b * Sq * Sk + col;
        for (int r = r0; r < r1; ++r) count += pcol[(int64_t)r * Sk] != 0;
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) count += __shfl_xor(count, off);  // over the 32 columns of a tile
    const int n = blockIdx.x * 8 + (tid >> 5);
    if ((tid & 31) == 0 && n < num_n) {
        const int cells = (r1 - r0) * min(BLOCK_N, Sk - n * BLOCK_N);
        flags[(int64_t)b * flags_stride_b + (int64_t)m * flags_stride_m + n] = count == 0 ? 0 : count == cells ? 2 : 1;
    }
}

int launch_mask_tile_flags(const uint8_t* mask, int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m, int B,
                           int Sq, int Sk, hipStream_t stream) {
    const int num_m = (Sq + BLOCK_M - 1) / BLOCK_M, num_n = (Sk + BLOCK_N - 1) / BLOCK_N;
    dim3 grid((num_n + 7) / 8, num_m, B);
    hipLaunchKernelGGL(mask_tile_flags_kernel, grid, dim3(256), 0, stream, mask, flags, flags_stride_b, flags_stride_m,
                       Sq, Sk, num_n);
    return (int)hipGetLastError();
}

// Work per 128-row block for the makespan-minimizing sequence split: the number of non-empty 128x32
// tiles of each row block, summed over the batch -- `torch.sum(compressed_mask > 0, dim=(0, 2))` of
// the reference (shardformer/layers/utils.py:161-166), computed where the flags already are instead
// of after a copy to the host.  One workgroup per row block, no atomics.
__global__ __launch_bounds__(256) void flag_row_workloads_kernel(const int8_t* __restrict__ flags, int64_t flags_stride_b,
                                                                 int64_t flags_stride_m, int B, int num_n,
                                                                 int* __restrict__ out) {
    __shared__ int partial[4];
    const int m = blockIdx.x, tid = threadIdx.x;
    int count = 0;
    for (int b = 0; b < B; ++b) {
        const int8_t* row = flags + (int64_t)b * flags_stride_b + (int64_t)m * flags_stride_m;
        for (int n = tid; n < num_n; n += 256) count += row[n] > 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) count += __shfl_xor(count, off);
    if ((tid & 63) == 0) partial[tid >> 6] = count;
    __syncthreads();
    if (tid == 0) out[m] = partial[0] + partial[1] + partial[2] + partial[3];
}

int launch_flag_row_workloads(const int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m, int B, int num_m,
                              int num_n, int* out, hipStream_t stream) {
    hipLaunchKernelGGL(flag_row_workloads_kernel, dim3(num_m), dim3(256), 0, stream, flags, flags_stride_b,
                       flags_stride_m, B, num_n, out);
    return (int)hipGetLastError();
}

// Plan for index-tensor attention: the class of every 32-row x 32-key tile of the LOCAL score matrix (rows and keys are
// subsets of a global sequence) and a slice order.  Same counting as the flag kernel: a run is a stretch of rows of one
// slice with equal bitfields at consecutive positions, and a column's count over a run follows from one evaluation of the
// bit test.  The extra column of workgroups ranks the slices.
// GATHER: rows and keys are read through index tensors, and the gathered bitfields and positions are left in out_* for the
// attention kernels (restates the index branch of the reference's mask block, bitfield_attention.py:71-87): the
// workgroups of column 0 write the rows, those of row 0 the keys.  One launch instead of three: with every pair evaluated and
// two gathers before it, 4096 rows against 8192 keys took 45 us; now 8.
template <bool GATHER>
__global__ __launch_bounds__(FLAG_WAVES * 64) void indexed_plan_kernel(
    const int64_t* __restrict__ bf, int64_t bf_sb, int L, const int64_t* __restrict__ idx_q, const int64_t* __restrict__ idx_k,
    int64_t* __restrict__ qbits, int64_t qbits_sb, int64_t* __restrict__ kbits, int64_t kbits_sb, int* __restrict__ qpos,
    int64_t qpos_sb, int* __restrict__ kpos, int Sq, int Sk, int num_n, uint8_t* __restrict__ fine, int64_t fine_sb,
    int64_t fine_ss, int* __restrict__ order, int64_t order_sb, int flag_blocks_x, int flag_groups, const int* __restrict__ rows_moved, int* __restrict__ pair_count) {
    typedef typename std::conditional<GATHER, IndexedRows, GatheredRows>::type Rows;
    const int b = blockIdx.z;
    if (rows_moved != nullptr && rows_moved[b] == 0) return;  // the plan in natural order stays
    Rows q_rows, k_rows;
    if constexpr (GATHER) {
        q_rows = IndexedRows{bf + (int64_t)b * bf_sb, idx_q, L};
        k_rows = IndexedRows{bf + (int64_t)b * bf_sb, idx_k, L};
    } else {
        q_rows = GatheredRows{qbits + (int64_t)b * qbits_sb, qpos + (int64_t)b * qpos_sb};
        k_rows = GatheredRows{kbits + (int64_t)b * kbits_sb, kpos};
    }
    if (pair_count != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0) *pair_count = 0;
    if ((int)blockIdx.x >= flag_blocks_x) {
        const int part = blockIdx.y;
        const int ns = (Sq + 31) / 32, slots = 4 * (int)gridDim.y;
        if (part * RANKED_PER_GROUP < slots)
            slice_order_ranked([&](int base, unsigned long long* sk) { slice_keys_chunk_indexed(q_rows, Sq, ns, base, sk); }, ns,
                               slots, part, order + (int64_t)b * order_sb,
                               rows_moved != nullptr ? ORDER_MOVED : 0);
        return;
    }
    __shared__ int64_t q_bits[BLOCK_M];
    __shared__ int q_pos[BLOCK_M];
    __shared__ __attribute__((aligned(8))) uint8_t s_out_buf[2][4][FLAG_COLS_PER_BLOCK];
    const int m = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5, l32 = lane & 31;
    // lanes [0, 32) own the columns of the wave's first tile, lanes [32, 64) those of the second
    static_assert(FLAG_TILES_PER_WAVE == 2, "each half of a wave takes one tile");
    int64_t kf = 0;
    int kp = 0;
    auto request_keys = [&](int bx) {
        const int j = (bx * FLAG_COLS_PER_BLOCK + wave * FLAG_TILES_PER_WAVE + half) * BLOCK_N + l32;
        kf = 0;
        kp = 0;
        if (j < Sk) {
            k_rows.get(j, kf, kp);
            if (GATHER && m == 0) {
                kbits[(int64_t)b * kbits_sb + j] = kf;
                if (b == 0) kpos[j] = kp;
            }
        }
    };
    request_keys(blockIdx.x);
    if (tid < BLOCK_M) {
        const int i = m * BLOCK_M + tid;
        int64_t f = 0;
        int pos = 0;
        if (i < Sq) {
            q_rows.get(i, f, pos);
            if (GATHER && blockIdx.x == 0) {
                qbits[(int64_t)b * qbits_sb + i] = f;
                if (b == 0) qpos[i] = pos;
            }
        }
        q_bits[tid] = f;  // rows past the end carry no bits: they see nothing
        q_pos[tid] = pos;
    }
    __syncthreads();
    const int64_t M = (((int64_t)1) << 62) - 1;
    unsigned slice_starts[4];
    bool one_run = (m + 1) * BLOCK_M <= Sq;  // every slice is one run of rows at consecutive positions
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int r = 32 * w + l32, before = 32 * w + max(l32, 1) - 1;
        slice_starts[w] = (unsigned)__ballot(l32 == 0 || q_bits[r] != q_bits[before] || q_pos[r] != q_pos[before] + 1);
        one_run &= slice_starts[w] == 1u;
    }
    // A workgroup takes the groups of eight column tiles blockIdx.x, blockIdx.x + flag_blocks_x, ...
    int it = 0;
    for (int bx = blockIdx.x; bx < flag_groups; bx += flag_blocks_x, ++it) {
        uint8_t (*s_out)[FLAG_COLS_PER_BLOCK] = s_out_buf[it & 1];
        if (it > 0) request_keys(bx);
        const int n = bx * FLAG_COLS_PER_BLOCK + wave * FLAG_TILES_PER_WAVE + half, col = wave * FLAG_TILES_PER_WAVE + half;
        const int64_t kb = kf & M;
        // keys of one bitfield at consecutive positions, all of them there: with such rows the classes follow from the ends
        const int64_t k0 = __shfl(kf, lane & 32);
        const int p0 = __shfl(kp, lane & 32);
        const bool closed = one_run && (__all((kf == k0 && kp == p0 + l32 && (n + 1) * BLOCK_N <= Sk)) != 0);
        if (closed) {
            if (l32 < 4) {
                const int64_t qf = q_bits[32 * l32], qb = qf & M, r0 = q_pos[32 * l32];
                const int64_t first = p0, last = (int64_t)p0 + BLOCK_N - 1;
                uint8_t c;
                if (qf & 1)
                    c = (qb & kb) == 0 || r0 + 31 < first ? 0 : r0 >= last ? 2 : 1;
                else
                    c = qb == kb && qb != 0 ? 2 : 0;
                s_out[l32][col] = c;
            }
        } else {
            int cnt[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                unsigned starts = slice_starts[w];
                int c = 0;
                while (starts != 0u) {  // wave-uniform
                    const int a = __builtin_ctz(starts);
                    starts &= starts - 1u;
                    const int e = starts != 0u ? __builtin_ctz(starts) : 32;  // the run is rows [a, e) of the slice
                    const int64_t qf = q_bits[32 * w + a], qb = qf & M, first = q_pos[32 * w + a];
                    if (qf & 1) {  // text rows: those at or after the key's position
                        const int64_t seen = first + (e - a) - (kp > first ? (int64_t)kp : first);
                        c += (qb & kb) != 0 && seen > 0 ? (int)seen : 0;
                    } else {
                        c += (qb == kb && qb != 0) ? e - a : 0;
                    }
                }
                cnt[w] = c;
            }
#pragma unroll
            for (int off = 16; off > 0; off >>= 1)
#pragma unroll
                for (int w = 0; w < 4; ++w) cnt[w] += __shfl_xor(cnt[w], off);
            if (l32 == 0) {
                const int cols_in_range = max(0, min(BLOCK_N, Sk - n * BLOCK_N));
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int rows = max(0, min(32, Sq - (m * BLOCK_M + 32 * w)));
                    s_out[w][col] = (uint8_t)(cnt[w] == 0 ? 0 : cnt[w] == rows * cols_in_range ? 2 : 1);
                }
            }
        }
        __syncthreads();
        if (tid < 4) {
            static_assert(FLAG_COLS_PER_BLOCK == 8, "one 64-bit word per row");
            *(unsigned long long*)(fine + (int64_t)b * fine_sb + (int64_t)(4 * m + tid) * fine_ss + bx * FLAG_COLS_PER_BLOCK) =
                *(const unsigned long long*)s_out[tid];
        }
    }
}

int launch_indexed_plan(const int64_t* bf, int64_t bf_sb, int L, const int64_t* idx_q, const int64_t* idx_k, int64_t* qbits,
                        int64_t qbits_sb, int64_t* kbits, int64_t kbits_sb, int* qpos, int* kpos, int Sq, int Sk, uint8_t* fine,
                        int64_t fine_sb, int64_t fine_ss, int* order, int64_t order_sb, int* pair_count, int B,
                        hipStream_t stream) {
    const int num_m = (Sq + BLOCK_M - 1) / BLOCK_M, num_n = (Sk + BLOCK_N - 1) / BLOCK_N;
    const int flag_groups = (num_n + FLAG_COLS_PER_BLOCK - 1) / FLAG_COLS_PER_BLOCK;
    const int flag_blocks_x = min(flag_groups, FLAG_MAX_BLOCKS_X);
    dim3 grid(flag_blocks_x + 1, num_m, B);
    if (idx_q != nullptr)
        hipLaunchKernelGGL(indexed_plan_kernel<true>, grid, dim3(FLAG_WAVES * 64), 0, stream, bf, bf_sb, L, idx_q, idx_k, qbits,
                           qbits_sb, kbits, kbits_sb, qpos, (int64_t)0, kpos, Sq, Sk, num_n, fine, fine_sb, fine_ss, order, order_sb,
                           flag_blocks_x, flag_groups, (const int*)nullptr, pair_count);
    else
        hipLaunchKernelGGL(indexed_plan_kernel<false>, grid, dim3(FLAG_WAVES * 64), 0, stream, bf, bf_sb, L, idx_q, idx_k, qbits,
                           qbits_sb, kbits, kbits_sb, qpos, (int64_t)0, kpos, Sq, Sk, num_n, fine, fine_sb, fine_ss, order, order_sb,
                           flag_blocks_x, flag_groups, (const int*)nullptr, pair_count);
    return (int)hipGetLastError();
}

// Flags and plan of a materialized bool mask in one launch: as mask_tile_flags_kernel, with the count kept per
// 32-row slice, so that the four slice classes of every flag tile come out of the same pass over the mask.  The
// slice order is simply "last slice first" (under a causal-like mask the late rows see the most keys); it is
// written by the workgroups of column 0.
// The same pass packs the mask to bits, once per orientation, for the attention kernels (which then never touch the
// mask bytes): thread = key column, so the 32 rows of a slice make one word of col_bits in a register, and a ballot
// over the 32 columns of a tile makes one word of row_bits per row.  Cells outside the mask are 0; the arrays cover
// num_m * 128 rows, ceil(Sk / 128) * 128 keys and an even number of 32-key blocks.
__global__ __launch_bounds__(256) void mask_tile_plan_kernel(const uint8_t* __restrict__ mask, int8_t* __restrict__ flags,
                                                             int64_t flags_stride_b, int64_t flags_stride_m, int Sq,
                                                             int Sk, int num_n, uint8_t* __restrict__ fine,
                                                             int64_t fine_sb, int64_t fine_ss, int* __restrict__ order,
                                                             int64_t order_sb, int* __restrict__ pair_count,
                                                             unsigned* __restrict__ row_bits, int64_t row_bits_sb,
                                                             int64_t row_bits_sn, unsigned* __restrict__ col_bits,
                                                             int64_t col_bits_sb, int64_t col_bits_ss) {
    const int b = blockIdx.z, m = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    if (pair_count != nullptr && blockIdx.x == 0 && m == 0 && b == 0 && tid == 0) *pair_count = 0;
    if (blockIdx.x == 0 && tid < 4) {
        const int ns = (Sq + 31) / 32, slot = 4 * m + tid;
        order[(int64_t)b * order_sb + slot] = slot < ns ? ns - 1 - slot : -1;
    }
    const int col = blockIdx.x * 256 + tid;
    const int r0 = m * BLOCK_M;
    const int n = blockIdx.x * 8 + (tid >> 5);  // this thread's 32-key block
    const int num_n_bits = (num_n + 1) & ~1, sk_pad = ((Sk + 127) >> 7) << 7;
    const bool in = col < Sk;
    const uint8_t* pcol = mask + (int64_t)b * Sq * Sk + (in ? col : 0);
    // lanes 0 and 32 of a wave write the row words of its two 32-key blocks
    unsigned* rb_out = (row_bits != nullptr && (lane & 31) == 0 && n < num_n_bits)
                           ? row_bits + (int64_t)b * row_bits_sb + (int64_t)n * row_bits_sn + r0
                           : nullptr;
    unsigned cw[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        cw[w] = 0;
        const int ra = r0 + 32 * w;
        if (row_bits == nullptr) {
            const int rb = min(ra + 32, Sq);
            for (int r = ra; r < rb; ++r) cw[w] |= (unsigned)(in && pcol[(int64_t)r * Sk] != 0) << (r - ra);
        } else {
            for (int r = ra; r < ra + 32; ++r) {
                const bool a = in && r < Sq && pcol[(int64_t)r * Sk] != 0;
                cw[w] |= (unsigned)a << (r - ra);
                const unsigned long long bal = __ballot(a);
                if (rb_out != nullptr) rb_out[r - r0] = (unsigned)(lane == 0 ? bal : bal >> 32);
            }
        }
    }
    if (col_bits != nullptr && col < sk_pad) {
#pragma unroll
        for (int w = 0; w < 4; ++w) col_bits[(int64_t)b * col_bits_sb + (int64_t)(4 * m + w) * col_bits_ss + col] = cw[w];
    }
    int count[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) count[w] = __popc(cw[w]);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {  // over the 32 columns of a tile
#pragma unroll
        for (int w = 0; w < 4; ++w) count[w] += __shfl_xor(count[w], off);
    }
    if ((tid & 31) == 0 && n < num_n) {
        const int cols = min(BLOCK_N, Sk - n * BLOCK_N);
        int total = 0, cells = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int rows = max(0, min(32, Sq - (r0 + 32 * w)));
            fine[(int64_t)b * fine_sb + (int64_t)(4 * m + w) * fine_ss + n] =
                (uint8_t)(count[w] == 0 ? 0 : count[w] == rows * cols ? 2 : 1);
            total += count[w];
            cells += rows * cols;
        }
        flags[(int64_t)b * flags_stride_b + (int64_t)m * flags_stride_m + n] = total == 0 ? 0 : total == cells ? 2 : 1;
    }
}

// The same for masks whose rows are 4-byte aligned (Sk a multiple of four): a lane takes FOUR key columns and reads
// them as one word per row, a wave takes one 32-row slice, so a workgroup reads 1 KiB per load instruction instead of
// 256 bytes.  The bytes are reduced to one bit each in the word; the four column words of the lane collect them row
// by row, the row word of a 32-key block is the OR of the nibbles of its eight lanes (DPP), staged in LDS and stored
// as runs of 32 rows.
__device__ __forceinline__ unsigned oct_or(unsigned x) {  // OR over groups of eight lanes, result in every lane
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
    x |= (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, false);  // row_half_mirror
    return x;
}
__global__ __launch_bounds__(256) void mask_tile_plan_words_kernel(
    const uint8_t* __restrict__ mask, int8_t* __restrict__ flags, int64_t flags_stride_b, int64_t flags_stride_m, int Sq,
    int Sk, int num_n, uint8_t* __restrict__ fine, int64_t fine_sb, int64_t fine_ss, int* __restrict__ order,
    int64_t order_sb, int* __restrict__ pair_count, unsigned* __restrict__ row_bits, int64_t row_bits_sb,
    int64_t row_bits_sn, unsigned* __restrict__ col_bits, int64_t col_bits_sb, int64_t col_bits_ss) {
    __shared__ unsigned s_rows[4][8][32];  // [slice][32-key block][row]: row words of this workgroup
    __shared__ int s_cnt[4][8];
    const int b = blockIdx.z, m = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (pair_count != nullptr && blockIdx.x == 0 && m == 0 && b == 0 && tid == 0) *pair_count = 0;
    if (blockIdx.x == 0 && tid < 4) {
        const int ns = (Sq + 31) / 32, slot = 4 * m + tid;
        order[(int64_t)b * order_sb + slot] = slot < ns ? ns - 1 - slot : -1;
    }
    const int col0 = blockIdx.x * 256 + 4 * lane;  // first of this lane's four columns (all inside or all outside)
    const int ra = m * BLOCK_M + 32 * w;           // first row of this wave's slice
    const int nb = lane >> 3, n = blockIdx.x * 8 + nb;
    const int num_n_bits = (num_n + 1) & ~1, sk_pad = ((Sk + 127) >> 7) << 7;
    const uint8_t* prow = mask + ((int64_t)b * Sq + ra) * Sk + (col0 < Sk ? col0 : 0);
    unsigned v[32];
#pragma unroll
    for (int r = 0; r < 32; ++r) v[r] = (col0 < Sk && ra + r < Sq) ? *(const unsigned*)(prow + (int64_t)r * Sk) : 0u;
    unsigned cw[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int r = 0; r < 32; ++r) {
        unsigned t = v[r] | (v[r] >> 4);  // any bit of a byte -> its bit 0
        t |= t >> 2;
        t |= t >> 1;
        t &= 0x01010101u;
#pragma unroll
        for (int c = 0; c < 4; ++c) cw[c] |= ((t >> (8 * c)) & 1u) << r;
        const unsigned nib = (t | (t >> 7) | (t >> 14) | (t >> 21)) & 0xFu;  // the four bits side by side
        const unsigned word = oct_or(nib << (4 * (lane & 7)));
        if ((lane & 7) == 0) s_rows[w][nb][r] = word;
    }
    if (col0 < sk_pad) {
        u32x4 out = {cw[0], cw[1], cw[2], cw[3]};
        *(u32x4*)(col_bits + (int64_t)b * col_bits_sb + (int64_t)(4 * m + w) * col_bits_ss + col0) = out;
    }
    // this wave's row words: 8 blocks x 32 rows, each block a run of 32 consecutive words
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int idx = 64 * k + lane, nb2 = idx >> 5, rr = idx & 31, n2 = blockIdx.x * 8 + nb2;
        if (n2 < num_n_bits)
            row_bits[(int64_t)b * row_bits_sb + (int64_t)n2 * row_bits_sn + ra + rr] = s_rows[w][nb2][rr];
    }
    int cnt = __popc(cw[0]) + __popc(cw[1]) + __popc(cw[2]) + __popc(cw[3]);
    cnt += __shfl_xor(cnt, 1);
    cnt += __shfl_xor(cnt, 2);
    cnt += __shfl_xor(cnt, 4);
    if ((lane & 7) == 0) {
        s_cnt[w][nb] = cnt;
        if (n < num_n) {
            const int cols = min(BLOCK_N, Sk - n * BLOCK_N), rows = max(0, min(32, Sq - ra));
            fine[(int64_t)b * fine_sb + (int64_t)(4 * m + w) * fine_ss + n] = (uint8_t)(cnt == 0 ? 0 : cnt == rows * cols ? 2 : 1);
        }
    }
    __syncthreads();
    if (tid < 8 && blockIdx.x * 8 + tid < num_n) {
        const int nn = blockIdx.x * 8 + tid, cols = min(BLOCK_N, Sk - nn * BLOCK_N);
        int total = 0, cells = 0;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            total += s_cnt[x][tid];
            cells += max(0, min(32, Sq - (m * BLOCK_M + 32 * x))) * cols;
        }
        flags[(int64_t)b * flags_stride_b + (int64_t)m * flags_stride_m + nn] = total == 0 ? 0 : total == cells ? 2 : 1;
    }
}

int launch_mask_tile_plan(const uint8_t* mask, int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m,
                          uint8_t* fine, int64_t fine_sb, int64_t fine_ss, int* order, int64_t order_sb, int* pair_count,
                          unsigned* row_bits, int64_t row_bits_sb, int64_t row_bits_sn, unsigned* col_bits,
                          int64_t col_bits_sb, int64_t col_bits_ss, int B, int Sq, int Sk, hipStream_t stream) {
    const int num_m = (Sq + BLOCK_M - 1) / BLOCK_M, num_n = (Sk + BLOCK_N - 1) / BLOCK_N;
    dim3 grid((num_n + 7) / 8, num_m, B);
    if (row_bits != nullptr && col_bits != nullptr && (Sk & 3) == 0 && (reinterpret_cast<uintptr_t>(mask) & 3u) == 0)
        hipLaunchKernelGGL(mask_tile_plan_words_kernel, grid, dim3(256), 0, stream, mask, flags, flags_stride_b,
                           flags_stride_m, Sq, Sk, num_n, fine, fine_sb, fine_ss, order, order_sb, pair_count, row_bits,
                           row_bits_sb, row_bits_sn, col_bits, col_bits_sb, col_bits_ss);
    else
        hipLaunchKernelGGL(mask_tile_plan_kernel, grid, dim3(256), 0, stream, mask, flags, flags_stride_b, flags_stride_m,
                           Sq, Sk, num_n, fine, fine_sb, fine_ss, order, order_sb, pair_count, row_bits, row_bits_sb,
                           row_bits_sn, col_bits, col_bits_sb, col_bits_ss);
    return (int)hipGetLastError();
}

// Numbering of the (32-row slice, 128-key tile) pairs that have work, for the backward that hands dS from the dK/dV
// kernel to the dQ kernel through memory.  The pairs of one key tile -- exactly the slices a dK/dV workgroup lists --
// get consecutive numbers, by ascending slice; the tiles themselves take their blocks of numbers in the order their
// workgroups arrive (one atomic add per tile on *count, which the plan kernels reset):
//   entry[b][s][t]  = number of pair (b, s, t), or -1 where its four classes are all "empty"  (what the dQ kernel looks up)
//   tile_base[b][t] = number of the first pair of key tile (b, t)                             (what dK/dV starts from)
//   *count          = how many pairs there are.
// Which tile gets which block of numbers only decides where a record sits in the workspace, never a result.
// tile_count[b][t] (optional) = number of pairs of key tile (b, t): what tile_order_kernel ranks the tiles by.
// One workgroup per (key tile, batch); thread = slice, 256 slices per sweep.
constexpr int DS_NUM_THREADS = 256;
constexpr int DS_MAX_ORDERED_TILES = MAX_RANKED;  // counts staged in LDS: 32 KiB
__global__ __launch_bounds__(DS_NUM_THREADS) void ds_entries_kernel(const uint8_t* __restrict__ fine, int64_t fine_sb,
                                                                   int64_t fine_ss, int slots, int nkt, int num_n,
                                                                   int* __restrict__ entry, int64_t entry_sb,
                                                                   int* __restrict__ tile_base, int* __restrict__ count,
                                                                   int* __restrict__ tile_count,
                                                                   const int* __restrict__ order, int64_t order_sb,
                                                                   int* __restrict__ group_count, int group_blocks,
                                                                   long long* __restrict__ row_workloads) {
    __shared__ int wave_sum[DS_NUM_THREADS / 64];
    __shared__ int s_base;
    const int b = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if ((int)blockIdx.x >= nkt + group_blocks) {
        // Extra workgroups, one per 128-row block m (those of batch entry 0 do the work): in how many of the block's
        // 128 x 32 tiles, over the whole batch, some pair is allowed -- the sum of (flags > 0) over batch and key
        // columns (reference shardformer/layers/utils.py:161-166).  A 128 x 32 flag is non-zero exactly when one of the
        // classes of its four 32 x 32 tiles is.
        if (b != 0) return;
        const int m = blockIdx.x - nkt - group_blocks, nb = gridDim.y;
        int tiles = 0;
        for (int bb = 0; bb < nb; ++bb) {
            const uint8_t* rows = fine + (int64_t)bb * fine_sb + (int64_t)(4 * m) * fine_ss;
            for (int n = tid; n < num_n; n += DS_NUM_THREADS)
                tiles += (rows[n] | rows[fine_ss + n] | rows[2 * fine_ss + n] | rows[3 * fine_ss + n]) != 0 ? 1 : 0;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) tiles += __shfl_xor(tiles, off);
        if (lane == 0) wave_sum[wave] = tiles;
        __syncthreads();
        if (tid == 0) {
            long long total = 0;
            for (int w = 0; w < DS_NUM_THREADS / 64; ++w) total += wave_sum[w];
            row_workloads[m] = total;
        }
        return;
    }
    if ((int)blockIdx.x >= nkt) {
        // Extra workgroups, one per group of four slices of the slice order: how many 64-key tiles the forward / dQ
        // workgroup of that group visits (the union over its slices), which is what group_order ranks the groups by.
        const int grp = blockIdx.x - nkt, num_m = slots / 4;
        const int* ord = order + (int64_t)b * order_sb + 4 * grp;
        const uint8_t* rows[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) rows[x] = ord[x] >= 0 ? fine + (int64_t)b * fine_sb + (int64_t)order_slice(ord[x]) * fine_ss : nullptr;
        int visits = 0;
        for (int kt = tid; 2 * kt < num_n; kt += DS_NUM_THREADS) {
            unsigned any = 0;
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (rows[x] != nullptr) any |= rows[x][2 * kt] | (2 * kt + 1 < num_n ? rows[x][2 * kt + 1] : 0);
            visits += any != 0 ? 1 : 0;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) visits += __shfl_xor(visits, off);
        if (lane == 0) wave_sum[wave] = visits;
        __syncthreads();
        if (tid == 0) {
            int total = 0;
            for (int w = 0; w < DS_NUM_THREADS / 64; ++w) total += wave_sum[w];
            group_count[b * num_m + grp] = total;
        }
        return;
    }
    const int t = blockIdx.x;
    const uint8_t* col = fine + (int64_t)b * fine_sb + 4 * t;
    unsigned valid = 0;  // which of the tile's four 32-key columns exist
#pragma unroll
    for (int w = 0; w < 4; ++w)
        if (4 * t + w < num_n) valid |= 0xFFu << (8 * w);
    auto has_work = [&](int sl) { return sl < slots && (*(const unsigned*)(col + (int64_t)sl * fine_ss) & valid) != 0; };
    int mine = 0;
    for (int sl = tid; sl < slots; sl += DS_NUM_THREADS) mine += has_work(sl) ? 1 : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off);
    if (lane == 0) wave_sum[wave] = mine;
    __syncthreads();
    if (tid == 0) {
        int total = 0;
        for (int w = 0; w < DS_NUM_THREADS / 64; ++w) total += wave_sum[w];
        const int base = atomicAdd(count, total);
        s_base = base;
        tile_base[(int64_t)b * nkt + t] = base;
        if (tile_count != nullptr) tile_count[b * nkt + t] = total;
    }
    __syncthreads();
    int next = s_base;
    int* out = entry + (int64_t)b * entry_sb + t;
    for (int s0 = 0; s0 < slots; s0 += DS_NUM_THREADS) {
        const int sl = s0 + tid;
        const bool h = has_work(sl);
        const unsigned long long bal = __ballot(h);
        __syncthreads();  // wave_sum is free again
        if (lane == 0) wave_sum[wave] = __popcll(bal);
        __syncthreads();
        int before = 0, all = 0;
        for (int w = 0; w < DS_NUM_THREADS / 64; ++w) {
            if (w < wave) before += wave_sum[w];
            all += wave_sum[w];
        }
        if (sl < slots) out[(int64_t)sl * nkt] = h ? next + before + __popcll(bal & ((1ull << lane) - 1ull)) : -1;
        next += all;
    }
}

// The key tiles (code b * nkt + t) sorted by their number of pairs, most first (ties: lower code first): the order in
// which the dK/dV kernel takes them, so that the long workgroups start first whatever the mask looks like.
// 64 tiles per workgroup, four threads per tile, each comparing against a quarter of all counts (staged in LDS).
// blockIdx.y = 1 ranks a second, independent array the same way (the groups of four slices, for the forward and dQ
// kernels); either array may be absent (n = 0).
// count_host (optional): the number of pairs, under the caller's tag, goes straight to pinned host memory, where the host
// polls for it; a copy on a side stream cost an event on either stream and 60-80 us of host time per plan, and its blit
// kernel took up to 75 us when the forward had filled the chip before it.
__global__ __launch_bounds__(256) void tile_order_kernel(const int* __restrict__ tile_count, int n_tiles,
                                                         int* __restrict__ tile_order,
                                                         const int* __restrict__ group_count, int n_groups,
                                                         int* __restrict__ group_order, const int* __restrict__ count,
                                                         unsigned long long* __restrict__ count_host,
                                                         unsigned long long count_tag, const int* __restrict__ rows_moved, int B) {
    __shared__ __attribute__((aligned(16))) int s_cnt[DS_MAX_ORDERED_TILES];
    __shared__ int s_sum[4];
    const int tid = threadIdx.x;
    if (count_host != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && tid < 64) {
        unsigned moved = 0;  // with sorted rows: whether some sequence's rows have been moved (bit 31), or left (bit 30)
        if (rows_moved != nullptr) {
            int some = 0, left = 0;
            for (int b = tid; b < B; b += 64) {
                some |= rows_moved[b] != 0;
                left |= rows_moved[b] == 0;
            }
            moved = (__any(some) ? 1u << 31 : 0u) | (__any(left) ? 1u << 30 : 0u);
        }
        if (tid == 0)
            __hip_atomic_store(count_host, count_tag | moved | (unsigned)*count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (blockIdx.y == 1) {
        tile_count = group_count;
        n_tiles = n_groups;
        tile_order = group_order;
    }
    if ((int)blockIdx.x * 64 >= n_tiles) return;  // (workgroup-uniform)
    const int padded = (n_tiles + 15) & ~15;
    int mine = 0;
    for (int i = tid; i < padded; i += 256) {
        s_cnt[i] = i < n_tiles ? tile_count[i] : -1;  // padding ranks behind everything
        mine += i < n_tiles ? s_cnt[i] : 0;
    }
    if (blockIdx.y == 1) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off);
        if ((tid & 63) == 0) s_sum[tid >> 6] = mine;
    }
    __syncthreads();
    const int i = blockIdx.x * 64 + (tid >> 2), sub = tid & 3;
    const int c = i < n_tiles ? s_cnt[i] : 0;
    int rank = 0;
    // thread `sub` of a tile takes the groups of four counts number sub, sub + 4, ...
    for (int j4 = sub; 4 * j4 < padded; j4 += 4) {
        const int4 v = *(const int4*)&s_cnt[4 * j4];
        const int j = 4 * j4;
        rank += (v.x > c) | ((v.x == c) & (j < i));
        rank += (v.y > c) | ((v.y == c) & (j + 1 < i));
        rank += (v.z > c) | ((v.z == c) & (j + 2 < i));
        rank += (v.w > c) | ((v.w == c) & (j + 3 < i));
    }
    rank += __shfl_xor(rank, 1);
    rank += __shfl_xor(rank, 2);
    if (sub == 0 && i < n_tiles) {
        tile_order[rank] = i;
        if (blockIdx.y == 1 && rank == 0) tile_order[n_tiles] = level_heads(n_tiles, (long long)s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3], c);
    }
}

// Both launches in one, for plans of up to SMALL_PLAN_WORDS (slice, 128-key tile) pairs (at 16384 the two are as fast): every workgroup computes the
// counts of ALL tiles (or of all groups) for itself -- a few thousand four-byte words out of L2, a dozen per thread --
// and so knows its own base and rank without waiting for anybody.  At 3001 tokens the two launches took 9.4 us and a gap.
// Tiles take their blocks of numbers in the order of their codes.
constexpr int SMALL_PLAN_WORDS = 10240, SMALL_PLAN_ITEMS = 1024, SMALL_PLAN_THREADS = 1024;
__global__ __launch_bounds__(SMALL_PLAN_THREADS) void small_plan_kernel(
    const uint8_t* __restrict__ fine, int64_t fine_sb, int64_t fine_ss, int B, int num_m, int nkt, int num_n,
    int* __restrict__ entry, int64_t entry_sb, int* __restrict__ tile_base, int* __restrict__ count,
    int* __restrict__ tile_order, const int* __restrict__ order, int64_t order_sb, int* __restrict__ group_order,
    long long* __restrict__ row_workloads, unsigned long long* __restrict__ count_host, unsigned long long count_tag) {
    __shared__ __attribute__((aligned(16))) int s_cnt[SMALL_PLAN_ITEMS];
    __shared__ int s_sum[SMALL_PLAN_THREADS / 64], s_rank[SMALL_PLAN_THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int slots = 4 * num_m, n_tiles = B * nkt, n_groups = B * num_m;
    const int role = blockIdx.x;
    // how many counts are larger than count i, or equal and of a lower code, among n counts: the rank of item i
    auto before_me = [&](int j, int i, int mine) { return (s_cnt[j] > mine) | ((s_cnt[j] == mine) & (j < i)); };

    if (role < n_tiles) {  // ---- one key tile
        for (int j = tid; j < n_tiles; j += SMALL_PLAN_THREADS) s_cnt[j] = 0;
        __syncthreads();
        const int words = B * slots * nkt;
        for (int w = tid; w < words; w += SMALL_PLAN_THREADS) {
            const int t = w % nkt, row = w / nkt, b = row / slots, sl = row - b * slots;
            const int cols = min(4, num_n - 4 * t);  // 32-key columns of the tile that exist
            const unsigned valid = cols == 4 ? ~0u : (1u << (8 * cols)) - 1u;
            const unsigned cls = *(const unsigned*)(fine + (int64_t)b * fine_sb + (int64_t)sl * fine_ss + 4 * t);
            if ((cls & valid) != 0) atomicAdd(&s_cnt[b * nkt + t], 1);
        }
        __syncthreads();
        const int mine = s_cnt[role];
        int below = 0, rank = 0;  // pairs of the tiles in front of this one, tiles with more pairs
        for (int j = tid; j < n_tiles; j += SMALL_PLAN_THREADS) {
            below += j < role ? s_cnt[j] : 0;
            rank += before_me(j, role, mine);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            below += __shfl_xor(below, off);
            rank += __shfl_xor(rank, off);
        }
        if (lane == 0) {
            s_sum[wave] = below;
            s_rank[wave] = rank;
        }
        __syncthreads();
        int base = 0, place = 0;
        for (int w = 0; w < SMALL_PLAN_THREADS / 64; ++w) {
            base += s_sum[w];
            place += s_rank[w];
        }
        if (tid == 0) {
            tile_base[role] = base;
            if (tile_order != nullptr) tile_order[place] = role;
            if (role == n_tiles - 1) {
                *count = base + mine;
                if (count_host != nullptr)
                    __hip_atomic_store(count_host, count_tag | (unsigned)(base + mine), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        // number this tile's slices, ascending
        const int b = role / nkt, t = role - b * nkt, cols = min(4, num_n - 4 * t);
        const unsigned valid = cols == 4 ? ~0u : (1u << (8 * cols)) - 1u;
        const uint8_t* col = fine + (int64_t)b * fine_sb + 4 * t;
        int* out = entry + (int64_t)b * entry_sb + t;
        for (int s0 = 0; s0 < slots; s0 += SMALL_PLAN_THREADS) {
            const int sl = s0 + tid;
            const bool h = sl < slots && (*(const unsigned*)(col + (int64_t)sl * fine_ss) & valid) != 0;
            const unsigned long long bal = __ballot(h);
            __syncthreads();  // s_sum is free
            if (lane == 0) s_sum[wave] = __popcll(bal);
            __syncthreads();
            int front = 0, all = 0;
            for (int w = 0; w < SMALL_PLAN_THREADS / 64; ++w) {
                if (w < wave) front += s_sum[w];
                all += s_sum[w];
            }
            if (sl < slots) out[(int64_t)sl * nkt] = h ? base + front + __popcll(bal & ((1ull << lane) - 1ull)) : -1;
            base += all;
        }
        return;
    }
    const int group_blocks = group_order != nullptr ? (n_groups + 63) / 64 : 0, gb = role - n_tiles;
    if (gb < group_blocks) {  // ---- 64 groups of four slices, 16 threads each
        for (int j = tid; j < n_groups; j += SMALL_PLAN_THREADS) s_cnt[j] = 0;
        __syncthreads();
        const int nkt64 = (num_n + 1) / 2;
        for (int w = tid; w < n_groups * nkt64; w += SMALL_PLAN_THREADS) {
            const int g = w / nkt64, kt = w - g * nkt64, b = g / num_m;
            const int* ord = order + (int64_t)b * order_sb + 4 * (g - b * num_m);
            const unsigned valid = 2 * kt + 1 < num_n ? 0xFFFFu : 0xFFu;
            unsigned any = 0;
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (ord[x] >= 0) any |= *(const uint16_t*)(fine + (int64_t)b * fine_sb + (int64_t)order_slice(ord[x]) * fine_ss + 2 * kt);
            if ((any & valid) != 0) atomicAdd(&s_cnt[g], 1);
        }
        __syncthreads();
        const int g = 64 * gb + (tid >> 4), sub = tid & 15;
        int rank = 0;
        if (g < n_groups) {
            const int mine = s_cnt[g];
            for (int j = sub; j < n_groups; j += 16) rank += before_me(j, g, mine);
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) rank += __shfl_xor(rank, off);
        if (g < n_groups && sub == 0) group_order[rank] = g;
        if (gb == 0 && wave == 0) {
            int sum = 0, longest = 0;
            for (int j = lane; j < n_groups; j += 64) {
                sum += s_cnt[j];
                longest = max(longest, s_cnt[j]);
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                sum += __shfl_xor(sum, off);
                longest = max(longest, __shfl_xor(longest, off));
            }
            if (lane == 0) group_order[n_groups] = level_heads(n_groups, sum, longest);
        }
        return;
    }
    // ---- 16 row blocks, one per wave: their non-empty 128 x 32 tiles over the whole batch
    const int m = 16 * (gb - group_blocks) + wave;
    if (m >= num_m) return;
    int tiles = 0;
    for (int b = 0; b < B; ++b) {
        const uint8_t* rows = fine + (int64_t)b * fine_sb + (int64_t)(4 * m) * fine_ss;
        for (int n = lane; n < num_n; n += 64)
            tiles += (rows[n] | rows[fine_ss + n] | rows[2 * fine_ss + n] | rows[3 * fine_ss + n]) != 0 ? 1 : 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) tiles += __shfl_xor(tiles, off);
    if (lane == 0) row_workloads[m] = tiles;
}

int launch_ds_entries(const uint8_t* fine, int64_t fine_sb, int64_t fine_ss, int B, int Sq, int Sk, int* entry,
                      int64_t entry_sb, int* tile_base, int* count, int* tile_count, int* tile_order, const int* order,
                      int64_t order_sb, int* group_count, int* group_order, int64_t* row_workloads, const int* rows_moved,
                      uint64_t* count_host, uint32_t count_tag, hipStream_t stream) {
    const int num_m = (Sq + BLOCK_M - 1) / BLOCK_M;
    const int slots = 4 * num_m, nkt = (Sk + 127) / 128, num_n = (Sk + BLOCK_N - 1) / BLOCK_N;
    const int n_tiles = nkt * B, n_groups = num_m * B;
    if (B <= SMALL_PLAN_ITEMS && (int64_t)n_tiles * slots <= SMALL_PLAN_WORDS && n_tiles <= SMALL_PLAN_ITEMS &&
        n_groups <= SMALL_PLAN_ITEMS && tile_count != nullptr && (group_order == nullptr || order != nullptr)) {
        const int blocks = n_tiles + (group_order != nullptr ? (n_groups + 63) / 64 : 0) + (row_workloads != nullptr ? (num_m + 15) / 16 : 0);
        hipLaunchKernelGGL(small_plan_kernel, dim3(blocks), dim3(SMALL_PLAN_THREADS), 0, stream, fine, fine_sb, fine_ss, B, num_m,
                           nkt, num_n, entry, entry_sb, tile_base, count, tile_order, order, order_sb, group_order,
                           (long long*)row_workloads, (unsigned long long*)count_host, (unsigned long long)count_tag << 32);
        return (int)hipGetLastError();
    }
    if (n_tiles > DS_MAX_ORDERED_TILES || tile_count == nullptr) tile_order = nullptr;
    if (n_groups > DS_MAX_ORDERED_TILES || group_count == nullptr || order == nullptr) group_order = nullptr;
    const int group_blocks = group_order != nullptr ? num_m : 0;
    hipLaunchKernelGGL(ds_entries_kernel, dim3(nkt + group_blocks + (row_workloads != nullptr ? num_m : 0), B),
                       dim3(DS_NUM_THREADS), 0, stream, fine, fine_sb, fine_ss, slots, nkt, num_n, entry, entry_sb,
                       tile_base, count, tile_order != nullptr ? tile_count : nullptr, order, order_sb, group_count,
                       group_blocks, (long long*)row_workloads);
    if (tile_order != nullptr || group_order != nullptr || count_host != nullptr) {
        const int nt = tile_order != nullptr ? n_tiles : 0, ng = group_order != nullptr ? n_groups : 0;
        hipLaunchKernelGGL(tile_order_kernel, dim3(max(1, (max(nt, ng) + 63) / 64), group_order != nullptr ? 2 : 1), dim3(256), 0,
                           stream, tile_count, nt, tile_order, group_count, ng, group_order, count,
                           (unsigned long long*)count_host, (unsigned long long)count_tag << 32, rows_moved, B);
    }
    return (int)hipGetLastError();
}

int launch_tile_flags(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                      int64_t flags_stride_m, int B, int S, hipStream_t stream) {
    const int num_m = (S + BLOCK_M - 1) / BLOCK_M, num_n = (S + BLOCK_N - 1) / BLOCK_N;
    const int flag_groups = (num_n + FLAG_COLS_PER_BLOCK - 1) / FLAG_COLS_PER_BLOCK;
    const int flag_blocks_x = min(flag_groups, FLAG_MAX_BLOCKS_X);
    dim3 grid(flag_blocks_x, num_m, B);
    hipLaunchKernelGGL(tile_flags_kernel<false>, grid, dim3(FLAG_WAVES * 64), 0, stream, bf, bf_stride_b, flags,
                       flags_stride_b, flags_stride_m, S, num_n, (uint8_t*)nullptr, (int64_t)0, (int64_t)0, (int*)nullptr,
                       (int64_t)0, flag_blocks_x, flag_groups, (int*)nullptr, SortedRows{});
    return (int)hipGetLastError();
}

int launch_tile_plan(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                     int64_t flags_stride_m, uint8_t* fine, int64_t fine_sb, int64_t fine_ss, int* order,
                     int64_t order_sb, int* pair_count, int B, int S, hipStream_t stream, int* rows, int64_t* rows_bits,
                     int64_t rows_sb, int* rows_moved) {
    const int num_m = (S + BLOCK_M - 1) / BLOCK_M, num_n = (S + BLOCK_N - 1) / BLOCK_N;
    const int flag_groups = (num_n + FLAG_COLS_PER_BLOCK - 1) / FLAG_COLS_PER_BLOCK;
    const int flag_blocks_x = min(flag_groups, FLAG_MAX_BLOCKS_X);
    // one more column of workgroups: (flag_blocks_x, part, b) ranks 64 slices; 4 num_m slots need
    // ceil(4 num_m / 64) <= num_m parts.  With sorted rows another one sorts, 1024 rows each
    dim3 grid(flag_blocks_x + (rows != nullptr ? 2 : 1), num_m, B);
    hipLaunchKernelGGL(tile_flags_kernel<true>, grid, dim3(FLAG_WAVES * 64), 0, stream, bf, bf_stride_b, flags,
                       flags_stride_b, flags_stride_m, S, num_n, fine, fine_sb, fine_ss, order, order_sb, flag_blocks_x,
                       flag_groups, pair_count, SortedRows{rows, rows_bits, rows_sb, rows_moved});
    return (int)hipGetLastError();
}

// Flags and plan in natural order and the sorted rows in one launch; a second one replaces the plan of the sequences whose rows have
// been moved (the workgroups of the others end at once).  Builder in us, natural order -> here: 17000 tokens, where nothing moves, 28 -> 33
// (a forward over 24637 tokens, 16 heads, D 80: 1.02 times as long with a sort and a whole second plan in front); 65536 tokens,
// moved, 230 -> 420.
int launch_sorted_plan(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m,
                       int* rows, int64_t* rows_bits, int64_t rows_sb, int* rows_moved, uint8_t* fine, int64_t fine_sb,
                       int64_t fine_ss, int* order, int64_t order_sb, int* pair_count, int B, int S, hipStream_t stream) {
    const int rc = launch_tile_plan(bf, bf_stride_b, flags, flags_stride_b, flags_stride_m, fine, fine_sb, fine_ss, order, order_sb,
                                    pair_count, B, S, stream, rows, rows_bits, rows_sb, rows_moved);
    if (rc != 0) return rc;
    const int num_m = (S + BLOCK_M - 1) / BLOCK_M, num_n = (S + BLOCK_N - 1) / BLOCK_N;
    const int flag_groups = (num_n + FLAG_COLS_PER_BLOCK - 1) / FLAG_COLS_PER_BLOCK;
    const int flag_blocks_x = min(flag_groups, FLAG_MAX_BLOCKS_X);
    hipLaunchKernelGGL(indexed_plan_kernel<false>, dim3(flag_blocks_x + 1, num_m, B), dim3(FLAG_WAVES * 64), 0, stream,
                       (const int64_t*)nullptr, (int64_t)0, 0, (const int64_t*)nullptr, (const int64_t*)nullptr, rows_bits, rows_sb,
                       const_cast<int64_t*>(bf), bf_stride_b, rows, rows_sb, (int*)nullptr, S, S, num_n, fine, fine_sb, fine_ss,
                       order, order_sb, flag_blocks_x, flag_groups, rows_moved, (int*)nullptr);
    return (int)hipGetLastError();
}

int launch_materialize_mask(const int64_t* bf, int64_t bf_stride_b, uint8_t* out, int B, int S,
                            hipStream_t stream) {
    dim3 grid(min((S + 255) / 256, 64), S, B);
    hipLaunchKernelGGL(materialize_mask_kernel, grid, dim3(256), 0, stream, bf, bf_stride_b, out, S);
    return (int)hipGetLastError();
}

}  // namespace bam
