// Single-token decode step: one query row per (batch, head) against the whole key / value cache.
// Reference: cornstarch/kernel/interface.py:71-83 hands this case (eval mode, q_len == 1) to flash-attn through
// transformers' flash_attention_forward with attention_mask=None, forwarding `scaling`, `sliding_window` and
// `softcap`.  With one query at the last position, flash-attn's semantics reduce to
//   s_j = scale * q.k_j ;  s_j = softcap * tanh(s_j / softcap)  (if softcap > 0)
//   keys j < Sk - window are dropped                            (if 0 < window < Sk)
//   o = softmax(s) V
// No bitfield is consulted.
//
// The step is bound by reading K and V once; there is one query row per head, so the parallelism has to come from the
// keys.  A unit is one (batch element, kv head, group of up to 32 of its q heads); its 32-key tiles are dealt in turn to
// the waves of the workgroups ("parts") that share the unit:
//   S^T (32 keys x 32 heads) = K Q^T with the K rows of the tile (copied global -> LDS) as the A operand, the q heads of
//   the unit are the 32 "query rows" (the tile is read once for all of them); a lane owns one head (softmax state =
//   per-lane scalars), P^T feeds O^T = V^T P^T from registers, V^T comes from the V tile through the transposing LDS read.
// Dealt in turn and not in runs: a probe that only reads a 256 MiB cache with the same copies reaches 5.9 TB/s when every
// wave walks a run of its own and 6.5 TB/s when neighbouring waves read neighbouring tiles; more bytes in flight per wave
// (two tiles ahead instead of one) changes neither.  Every unit starts at a tile of its own (`turn`), so that the
// units, whose caches often lie a power of two apart, do not walk the memory banks in step (3 % at 64 units).
// A unit with several parts leaves partial results (unnormalized output, maximum, sum) in the workspace; the part that
// arrives last merges them.  They are written and read through to memory (agent-scope accesses): a release fence instead
// writes back the whole L2 of the XCD and cost 15 to 60 us per launch.  Without counters, or with so many parts that one
// workgroup would take too long over them, a second launch merges (decode_combine_kernel).
#include "bam_common.h"
#include "bam_launch.h"
#include "bam_tiles.h"

#include <cfloat>

namespace bam {

constexpr int DEC_KT = 32;        // keys per tile
constexpr int DEC_K_BUFS = 1, DEC_V_BUFS = 2;
template <int D>
constexpr int DEC_WAVE_CHUNKS = (DEC_K_BUFS + DEC_V_BUFS) * DEC_KT * (LDS_COLS<D> / 8);

// softcap * tanh(x / softcap), y = x / softcap.  Below |y| = 1: x + x y^2 P(y^2), so that a score far below the cap keeps its
// own precision (P: tanh(y) / y - 1 over y^2, interpolated at seven Chebyshev nodes of [0, 1]; 8.6e-8 relative).  Above:
// cap (1 - 2 t / (1 + t)) with t = exp(-2 |y|), where the errors of t and of the raw reciprocal carry the small factor
// 2 t / (1 + t).  (1 - t) / (1 + t) for all y cancels: an absolute error of 2e-8 of the cap.  Measured against 64 bits over
// 2^20 scores up to 4 / up to 100, rms error of this / of cap * tanhf(x / cap) / of the quotient form: cap 1 1.7e-8 / 1.7e-8 /
// 4.2e-8, cap 30 5.2e-8 / 9.6e-8 / 3.5e-7, cap 50 5.2e-8 / 1.0e-7 / 5.1e-7, cap 1e3 5.2e-8 / 9.5e-8 / 9.0e-6, cap 1e6 8e-12 /
// 3.8e-8 / 9.3e-3; up to 100: cap 30 7.5e-7 / 7.6e-7 / 1.3e-6, cap 50 1.2e-6 / 1.3e-6 / 2.2e-6.
// `far`: whether the wave holds a score at or beyond the cap; without one the second form is left out.  One sequence, 512 keys,
// 32 / 8 heads, D 128, the whole step: quotient form 7.15 us, both forms for every score 7.41; on another run quotient form
// 7.23, second form where needed 7.23.
__device__ __forceinline__ float cap_score(float x, float cap, float inv_cap, bool far) {
    const float y = x * inv_cap, u = y * y;
    float p = fmaf(-0.000420695491f, u, 0.0025104594f);
    p = fmaf(p, u, -0.00821892172f);
    p = fmaf(p, u, 0.0216601156f);
    p = fmaf(p, u, -0.0539347902f);
    p = fmaf(p, u, 0.133331284f);
    p = fmaf(p, u, -0.333333313f);
    const float small = fmaf(x * u, p, x);
    if (!far) return small;
    const float t = __builtin_amdgcn_exp2f(fabsf(y) * (-2.f * LOG2E));
    const float large = copysignf(cap * fmaf(-2.f * t, __builtin_amdgcn_rcpf(1.f + t), 1.f), x);
    return u < 1.f ? small : large;
}

template <typename T>
__device__ __forceinline__ void store_out4(const DecodeParams& p, int b, int h, int col, const f32x4& x) {
    unsigned short* op = (unsigned short*)p.o + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + col;
    u32x2 w = {T::pack2(x[0], x[1]), T::pack2(x[2], x[3])};
    if (p.o_vec) {
        *(u32x2*)op = w;
    } else {
        op[0] = (unsigned short)w[0];
        op[1] = (unsigned short)(w[0] >> 16);
        op[2] = (unsigned short)w[1];
        op[3] = (unsigned short)(w[1] >> 16);
    }
}

// Running merge of partial results with maxima in the log2 domain.
struct Merge {
    float m = -INFINITY, l = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    __device__ __forceinline__ void add(float ms, float ls, const f32x4& o4) {
        if (ms == -INFINITY) return;  // a part without keys
        const float mnew = fmaxf(m, ms);
        const float a = __builtin_amdgcn_exp2f(m - mnew), w = __builtin_amdgcn_exp2f(ms - mnew);  // a = 0 at first
        m = mnew;
        l = l * a + ls * w;
#pragma unroll
        for (int x = 0; x < 4; ++x) acc[x] = acc[x] * a + o4[x] * w;
    }
};

// Accesses that go through to memory, for results that workgroups on other XCDs read (or write) in the same launch.
__device__ __forceinline__ void store_through(float* p, float x, float y) {
    const u32x2 w = {__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, y)};
    __hip_atomic_store((unsigned long long*)p, __builtin_bit_cast(unsigned long long, w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f32x2 load_through(const float* p) {
    return __builtin_bit_cast(
        f32x2, __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

template <typename T, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES == 1 ? 2 : 1) void decode_kernel(const DecodeParams p) {
    constexpr int NCH = LDS_COLS<D> / 8, KK = D / 16, DB = D / 32, TILE = DEC_KT * NCH, THREADS = 64 * WAVES;
    __shared__ u32x4 sTiles[WAVES][DEC_WAVE_CHUNKS<D>];
    static_assert(DEC_WAVE_CHUNKS<D> * 16 >= 32 * (D + 2) * 4, "a wave's results fit its tile buffers");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
    const int G = p.Hq / p.Hkv, chunks = p.d / 8, first = p.first;
    const int n_tiles = p.n_tiles, parts = p.parts;
    const int unit = (int)((unsigned)blockIdx.x / (unsigned)parts), part = (int)blockIdx.x - unit * parts;
    const unsigned bh = (unsigned)unit / (unsigned)p.row_groups;
    const int rg = unit - (int)bh * p.row_groups, b = (int)(bh / (unsigned)p.Hkv), hk = (int)bh - b * p.Hkv;
    const int h0 = hk * G + 32 * rg;         // first q head of the unit
    const int rows = min(32, G - 32 * rg);   // q heads it holds
    // this wave's tiles: number t0, t0 + step, ... in the unit's order, which starts at tile `turn`
    const int t0 = part * WAVES + wave, step = parts * WAVES;
    const int turn = (int)((unsigned)unit * 7u % (unsigned)n_tiles);
    auto tile_of = [&](int t) { return t + turn < n_tiles ? t + turn : t + turn - n_tiles; };
    u32x4* const sK = sTiles[wave];
    u32x4* const sV = sTiles[wave] + DEC_K_BUFS * TILE;
    const bool q_aligned = ((reinterpret_cast<uintptr_t>(p.q) | (uintptr_t)(2 * p.q_sb) | (uintptr_t)(2 * p.q_sh)) & 15u) == 0;
    const float inv_cap = p.softcap > 0.f ? fminf(1.f / p.softcap, FLT_MAX) : 0.f;  // (finite: a score of 0 stays 0)
    TileStage<D, DEC_KT, 64, true> stK;
    TileStage<D, DEC_KT, 64> stV;
    constexpr int CPT = TileStage<D, DEC_KT, 64>::CPT;
    stK.setup(2 * p.k_ss, chunks, lane, DMA_ZERO);
    stV.setup(2 * p.v_ss, chunks, lane);

    // ---- Q: rows = heads, zero rows past the last head, zero columns past the head dim ----
    u32x4 qreg[KK];
    const u32x4 z = {0u, 0u, 0u, 0u};
    if (q_aligned) {  // wave-uniform: the lane's 16-byte pieces straight from global memory
        const char* qrow = (const char*)p.q + 2 * ((int64_t)b * p.q_sb + (int64_t)(h0 + min(l32, rows - 1)) * p.q_sh);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int c = 2 * kk + hi;
            const u32x4 x = *(const u32x4*)(qrow + (c < chunks ? c : 0) * 16);
            qreg[kk] = l32 < rows && c < chunks ? x : z;
        }
    } else {  // element-wise loads through LDS (a view of q may be only 2-byte aligned)
        unsigned short* sQ = (unsigned short*)sTiles[wave];
        for (int i = lane; i < rows * D; i += 64) {
            const int r = i / D, d = i % D;
            sQ[i] = d < p.d ? ((const unsigned short*)p.q)[(int64_t)b * p.q_sb + (int64_t)(h0 + r) * p.q_sh + d] : 0;
        }
        wait_lds();
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qreg[kk] = l32 < rows ? *(const u32x4*)&sQ[l32 * D + 16 * kk + 8 * hi] : z;
        wait_lds();  // the staging area becomes tile buffers
    }

    const char* kbase = (const char*)p.k + 2 * ((int64_t)b * p.k_sb + (int64_t)hk * p.k_sh);
    const char* vbase = (const char*)p.v + 2 * ((int64_t)b * p.v_sb + (int64_t)hk * p.v_sh);
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    f32x16 zero16;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero16[i] = 0.f;
    float m_i = -INFINITY, l_i = 0.f;  // maximum in the log2 domain; this lane's share of the sum (16 of 32 keys)

    // Tile number t as 1 KiB pieces, global -> LDS.  Past the end of the cache the last tile repeats its last row (its scores
    // are masked).
    auto fetch = [&](int t, int vbuf) {
        const int key0 = first + tile_of(t) * DEC_KT, nvalid = p.Sk - key0;
        const char* kt = kbase + 2 * (int64_t)key0 * p.k_ss;
        const char* vt = vbase + 2 * (int64_t)key0 * p.v_ss;
        const unsigned lk = lds_addr(sK), lv = lds_addr(sV + vbuf * TILE);
        if (nvalid >= DEC_KT) {
            stK.load_full(kt, lk);
            stV.load_full(vt, lv);
        } else {
#pragma unroll
            for (int i = 0; i < CPT; ++i) {
                const int over = max(0, (lane + 64 * i) / NCH - (nvalid - 1));  // rows this lane has to go back
                stK.template copy<3>(kt, stK.goff[i] - (unsigned)(over * (int)(2 * p.k_ss)), lk + 1024u * i);
                stV.template copy<4>(vt, stV.goff[i] - (unsigned)(over * (int)(2 * p.v_ss)), lv + 1024u * i);
            }
        }
    };

    if (t0 < n_tiles) fetch(t0, 0);
    // q has to have arrived here, once: at its first use inside the loop the wait would drain every copy in flight
    // each time round
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) asm volatile("" : "+v"(qreg[kk]));
    int vcur = 0;
    for (int t = t0; t < n_tiles; t += step, vcur ^= 1) {
        wait_async();
        u32x4 ka[KK];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) ka[kk] = lds_read_chunk<D>(sK, l32, 2 * kk + hi);
        wait_lds();  // (also the reads of the previous V tile, whose buffer the next copies take)
        // the next tile is requested as soon as this one's K rows are in registers: its latency runs under this tile's
        // arithmetic and under the other waves of the compute unit
        if (t + step < n_tiles) fetch(t + step, vcur ^ 1);
        f32x16 s = zero16;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) s = T::mfma(ka[kk], qreg[kk], s);

        // scores in the log2 domain: scale, cap, keys past the end
        const int nvalid = p.Sk - (first + tile_of(t) * DEC_KT);
        if (p.softcap > 0.f) {
            float top = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] *= p.scale;
                top = fmaxf(top, fabsf(s[i]));
            }
            if (__all(top < p.softcap)) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = cap_score(s[i], p.softcap, inv_cap, false) * LOG2E;
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = cap_score(s[i], p.softcap, inv_cap, true) * LOG2E;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = s[i] * p.scale * LOG2E;
        }
        if (nvalid < DEC_KT) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 8 * (i >> 2) + 4 * hi + (i & 3) < nvalid ? s[i] : -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
        const float mloc = half_swap_max(mx);        // finite: every tile holds at least one key
        const float mnew = fmaxf(m_i, mloc);
        const float alpha = __builtin_amdgcn_exp2f(m_i - mnew);  // 0 for the first tile
        m_i = mnew;
        float ls = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = __builtin_amdgcn_exp2f(s[i] - mnew);
            ls += s[i];
        }
        l_i = l_i * alpha + ls;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
        u32x4 pb[2];
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) pb[h2] = pack8<T>(s, 8 * h2);
        const u32x4* tV = sV + vcur * TILE;
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const u32x4 va = lds_read_transposed<D>(tV, lane, 16 * h2 + 4 * hi, 32 * db + 16 * half16);
                o[db] = T::mfma(va, pb[h2], o[db]);
            }
    }

    // ---- the waves' results meet in LDS (every wave parks in its own tile buffers, whose reads are done):
    // O^T fragment register i of block db <-> column 32 db + 8 (i/4) + 4 hi + i%4 of head h0 + l32
    const float ltot = half_swap_sum(l_i);
    float* park = (float*)sTiles[wave];  // rows x D outputs, then rows x (maximum, sum)
    wait_lds();
    if (l32 < rows) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                f32x4 w = {o[db][4 * grp], o[db][4 * grp + 1], o[db][4 * grp + 2], o[db][4 * grp + 3]};
                *(f32x4*)(park + l32 * D + 32 * db + 8 * grp + 4 * hi) = w;
            }
        if (hi == 0) {
            park[rows * D + 2 * l32] = m_i;
            park[rows * D + 2 * l32 + 1] = ltot;
        }
    }
    __syncthreads();
    constexpr int COLS = D / 4;  // groups of four columns
    for (int item = tid; item < rows * COLS; item += THREADS) {
        const int r = item / COLS, col = 4 * (item % COLS);
        Merge mg;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float* pw = (const float*)sTiles[w];
            mg.add(pw[rows * D + 2 * r], pw[rows * D + 2 * r + 1], *(const f32x4*)(pw + r * D + col));
        }
        if (parts == 1) {
            const float inv = 1.f / mg.l;
            if (col < p.d) store_out4<T>(p, b, h0 + r, col, mg.acc * inv);
        } else {
            const int64_t rec = ((int64_t)b * p.Hq + h0 + r) * parts + part;
            store_through(p.ws_o + rec * D + col, mg.acc[0], mg.acc[1]);
            store_through(p.ws_o + rec * D + col + 2, mg.acc[2], mg.acc[3]);
            if (col == 0) store_through(p.ws_ml + 2 * rec, mg.m, mg.l);
        }
    }
    if (parts == 1 || p.counters == nullptr) return;

    // ---- every thread's stores have reached memory, then the part is counted; the last one to arrive sees all parts and
    // puts the counter back to zero
    wait_async();
    __syncthreads();
    volatile unsigned* arrived = (volatile unsigned*)sTiles;
    if (tid == 0) *arrived = __hip_atomic_fetch_add(&p.counters[unit], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrived != (unsigned)(parts - 1)) return;
    if (tid == 0) __hip_atomic_store(&p.counters[unit], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr int AHEAD = 8;  // parts requested together: the loop is a chain of memory latencies
    for (int item = tid; item < rows * COLS; item += THREADS) {
        const int r = item / COLS, col = 4 * (item % COLS);
        const int64_t rec = ((int64_t)b * p.Hq + h0 + r) * parts;
        const float* wo = p.ws_o + rec * D + col;
        const float* ml = p.ws_ml + 2 * rec;
        Merge mg;
        for (int s = 0; s < parts; s += AHEAD) {
            f32x4 o4[AHEAD];
            f32x2 ml2[AHEAD];
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                const int sj = min(s + j, parts - 1);
                const f32x2 lo = load_through(wo + (int64_t)sj * D), hi2 = load_through(wo + (int64_t)sj * D + 2);
                o4[j] = f32x4{lo[0], lo[1], hi2[0], hi2[1]};
                ml2[j] = load_through(ml + 2 * sj);
            }
#pragma unroll
            for (int j = 0; j < AHEAD; ++j)
                if (s + j < parts) mg.add(ml2[j][0], ml2[j][1], o4[j]);
        }
        const float inv = 1.f / mg.l;
        if (col < p.d) store_out4<T>(p, b, h0 + r, col, mg.acc * inv);
    }
}

// Merges the parts of one (batch, head): the second launch where the split kernel does not do it.  Thread = four output
// columns x one of several interleaved subsets of the parts; the subsets then meet in LDS.
constexpr int COMBINE_THREADS = 256;
template <typename T>
__global__ __launch_bounds__(COMBINE_THREADS) void decode_combine_kernel(const DecodeParams p) {
    __shared__ float s_m[COMBINE_THREADS], s_l[COMBINE_THREADS];
    __shared__ __attribute__((aligned(16))) float s_acc[COMBINE_THREADS][4];
    const int bh = blockIdx.x, tid = threadIdx.x, b = bh / p.Hq, h = bh % p.Hq, parts = p.parts;
    const int cols = p.D / 4;                 // threads across the columns: 8, 16, 24 or 32
    const int lanes = COMBINE_THREADS / cols; // subsets of the parts
    const int c4 = tid % cols, sl = tid / cols;
    const float* ml = p.ws_ml + 2 * (int64_t)bh * parts;
    const float* wo = p.ws_o + (int64_t)bh * parts * p.D + 4 * c4;
    Merge mg;
    if (sl < lanes) {
        for (int s = sl; s < parts; s += 4 * lanes) {
            f32x4 o4[4];
            float ms[4], ls[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int sj = min(s + j * lanes, parts - 1);
                o4[j] = *(const f32x4*)(wo + (int64_t)sj * p.D);
                ms[j] = ml[2 * sj];
                ls[j] = ml[2 * sj + 1];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (s + j * lanes < parts) mg.add(ms[j], ls[j], o4[j]);
        }
    }
    s_m[tid] = mg.m;
    s_l[tid] = mg.l;
    *(f32x4*)s_acc[tid] = mg.acc;
    __syncthreads();
    if (sl != 0) return;
    for (int j = 1; j < lanes; ++j) {
        const int t = j * cols + c4;
        mg.add(s_m[t], s_l[t], *(const f32x4*)s_acc[t]);
    }
    const float inv = 1.f / mg.l;
    if (4 * c4 < p.d) store_out4<T>(p, b, h, 4 * c4, mg.acc * inv);
}

template <typename T, int D>
static void launch_decode_d(const DecodeParams& p, int units, int waves, hipStream_t stream) {
    if (waves == 1)
        hipLaunchKernelGGL((decode_kernel<T, D, 1>), dim3(units * p.parts), dim3(64), 0, stream, p);
    else
        hipLaunchKernelGGL((decode_kernel<T, D, 4>), dim3(units * p.parts), dim3(256), 0, stream, p);
}
template <typename T>
static int launch_decode_t(const DecodeParams& p, int units, int waves, hipStream_t stream) {
    if (p.D == 128)
        launch_decode_d<T, 128>(p, units, waves, stream);
    else if (p.D == 96)
        launch_decode_d<T, 96>(p, units, waves, stream);
    else if (p.D == 64)
        launch_decode_d<T, 64>(p, units, waves, stream);
    else
        launch_decode_d<T, 32>(p, units, waves, stream);
    if (p.parts > 1 && p.counters == nullptr)
        hipLaunchKernelGGL((decode_combine_kernel<T>), dim3(p.B * p.Hq), dim3(COMBINE_THREADS), 0, stream, p);
    return (int)hipGetLastError();
}

int launch_decode(const DecodeParams& p, const DecodeSplit& s, int dtype, hipStream_t stream) {
    return dtype == 1 ? launch_decode_t<BF16>(p, (int)s.units, s.waves, stream) : launch_decode_t<F16>(p, (int)s.units, s.waves, stream);
}

// How the tiles of one decode step are dealt to workgroups.  Shared by the workspace size and the launch.
DecodeSplit decode_split(int B, int Hq, int Hkv, int Sk, int D, int window) {
    DecodeSplit s;
    s.row_groups = (Hq / Hkv + 31) / 32;
    s.units = (int64_t)B * Hkv * s.row_groups;
    s.first = (window > 0 && window < Sk) ? Sk - window : 0;
    s.n_tiles = (Sk - s.first + DEC_KT - 1) / DEC_KT;
    // Four waves per workgroup, one workgroup per compute unit (their LDS): the waves meet in LDS, so a quarter of the
    // partial results.  Only where that fills the chip in one round, or where there are not even tiles enough to.
    const int64_t slots = D <= 32 ? 512 : 256, most = (s.n_tiles + 3) / 4;
    int64_t parts = slots / s.units;
    if (parts * s.units * 5 >= slots * 4 || most * s.units <= slots) {
        s.waves = 4;
        if (parts > 32 && parts > s.n_tiles / 16) parts = s.n_tiles / 16 > 32 ? s.n_tiles / 16 : 32;  // long merges: 4 tiles a wave
        if (parts > most) parts = most;
    } else {
        // workgroups of one wave: 8 MiB of tiles in flight (512 waves at D = 128; twice as many measured 5 % slower, half
        // as many leave the memory idle), at least two tiles each
        s.waves = 1;
        parts = (65536 / D + s.units - 1) / s.units;
        if (parts > s.n_tiles / 2) parts = s.n_tiles / 2;
    }
    s.parts = parts < 1 ? 1 : (int)parts;
    return s;
}

}  // namespace bam
