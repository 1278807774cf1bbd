// extern "C" boundary of libbam_hip.so: argument validation + kernel launches.
// The declarations (with the reference call sites they replace) are in include/bam_hip.h.
#include "../../include/bam_hip.h"

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>

#include "bam_launch.h"

// Built-in plan workspace of bam_tile_plan_static: device memory that exists once per GPU for as long as the
// process lives.  In host code this name is only a handle for hipGetSymbolAddress; kernels and the other entry
// points are handed the address that call returns for the current device (g_static_plan_ptr).
static __device__ __align__(256) unsigned char g_static_plan_scratch[BAM_STATIC_PLAN_BYTES];

namespace {

constexpr int kMaxDevices = 64;
// per device, resolved on first use (two host threads that get there together both store the same address)
std::atomic<void*> g_static_plan_ptr[kMaxDevices] = {};
// Every bam_tile_plan_static call on a device starts a new generation of that device's array; the plan it returns
// carries the number, and a plan of an older generation (its arrays have been overwritten since) is refused.
std::atomic<int32_t> g_static_plan_generation[kMaxDevices] = {};

thread_local char g_error[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
    return code;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_half_tensor(const char* name, const void* ptr, int64_t sb, int64_t ss, int64_t sh) {
    if (ptr == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: null pointer", name);
    if (!aligned16(ptr)) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: pointer is not 16-byte aligned", name);
    if ((sb % 8) || (ss % 8) || (sh % 8))
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: strides (%lld, %lld, %lld) must be multiples of 8 elements", name,
                    (long long)sb, (long long)ss, (long long)sh);
    // tile copies hold row * stride as 32-bit byte offsets, for up to 128 rows of 2-byte elements
    if (ss < 0 || ss >= (1ll << 23))
        return fail(BAM_ERR_UNSUPPORTED, "%s: sequence stride %lld is outside [0, 2^23) elements", name, (long long)ss);
    return BAM_OK;
}

int check_f32_tensor(const char* name, const void* ptr, int64_t sb, int64_t ss, int64_t sh) {
    if (ptr == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: null pointer", name);
    if (!aligned16(ptr)) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: pointer is not 16-byte aligned", name);
    if ((sb % 4) || (ss % 4) || (sh % 4))
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: strides (%lld, %lld, %lld) must be multiples of 4 elements", name,
                    (long long)sb, (long long)ss, (long long)sh);
    return BAM_OK;
}

// any_dim: the struct form takes every multiple of 8, the older entry points the three head dims they always took
int check_problem(int B, int Sq, int Sk, int Hq, int Hkv, int D, int dtype, bool any_dim = false) {
    if (B <= 0 || Sq <= 0 || Sk <= 0 || Hq <= 0 || Hkv <= 0)
        return fail(BAM_ERR_INVALID_ARGUMENT, "B, S, Hq, Hkv must be positive (got B %d, Sq %d, Sk %d, Hq %d, Hkv %d)", B,
                    Sq, Sk, Hq, Hkv);
    if (Hq % Hkv) return fail(BAM_ERR_INVALID_ARGUMENT, "Hq (%d) must be a multiple of Hkv (%d)", Hq, Hkv);
    if (any_dim ? (D <= 0 || D > 128 || D % 8) : (D != 32 && D != 64 && D != 128))
        return fail(BAM_ERR_UNSUPPORTED, "head dimension %d is not supported (%s)", D,
                    any_dim ? "a multiple of 8 up to 128" : "32, 64 or 128");
    if (dtype != BAM_DTYPE_F16 && dtype != BAM_DTYPE_BF16)
        return fail(BAM_ERR_INVALID_ARGUMENT, "dtype %d is neither BAM_DTYPE_F16 nor BAM_DTYPE_BF16", dtype);
    static_assert(BAM_MAX_SEQLEN == bam::MAX_SEQLEN, "header and kernels disagree on the longest sequence");
    if (Sq > BAM_MAX_SEQLEN || Sk > BAM_MAX_SEQLEN)
        return fail(BAM_ERR_UNSUPPORTED, "S = %d exceeds BAM_MAX_SEQLEN = %d", Sq > Sk ? Sq : Sk, BAM_MAX_SEQLEN);
    if ((int64_t)((Sq + 127) / 128) * B * Hq > 0x7FFFFFFFll || (int64_t)((Sk + 127) / 128) * B * Hkv > 0x7FFFFFFFll)
        return fail(BAM_ERR_UNSUPPORTED, "grid too large");
    return BAM_OK;
}

int launched(int hip_err, const char* what) {
    if (hip_err != 0)
        return fail(BAM_ERR_LAUNCH, "%s: launch failed: %s", what, hipGetErrorString((hipError_t)hip_err));
    return BAM_OK;
}

// Where the kernels find bitfields and positions: one (B, S) tensor for plain attention, gathered
// per-row / per-key arrays plus positions for index-tensor attention.
struct MaskSource {
    int mode;
    const int64_t *bfq, *bfk;
    int64_t bfq_sb, bfk_sb;
    const int *posq, *posk;
    const uint8_t* mask;
    int Sq, Sk;
};

MaskSource plain_source(const int64_t* bf, int64_t bf_stride_b, int S) {
    return MaskSource{bam::MASK_BITFIELD, bf, bf, bf_stride_b, bf_stride_b, nullptr, nullptr, nullptr, S, S};
}

MaskSource dense_source(const uint8_t* mask, int Sq, int Sk) {
    return MaskSource{bam::MASK_DENSE, nullptr, nullptr, 0, 0, nullptr, nullptr, mask, Sq, Sk};
}

// the kernels read the mask four bytes at a time when rows are a multiple of four bytes long
int check_mask(const char* who, const uint8_t* mask) {
    if (reinterpret_cast<uintptr_t>(mask) & 3u) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: mask is not 4-byte aligned", who);
    return BAM_OK;
}

int indexed_source(const bam_index_view* iv, MaskSource& m) {
    if (iv == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "index view: null pointer");
    if (iv->q_bits == nullptr || iv->k_bits == nullptr || iv->q_pos == nullptr || iv->k_pos == nullptr)
        return fail(BAM_ERR_INVALID_ARGUMENT, "index view: q_bits, k_bits, q_pos and k_pos must not be null");
    if ((reinterpret_cast<uintptr_t>(iv->q_bits) & 7u) || (reinterpret_cast<uintptr_t>(iv->k_bits) & 7u) ||
        (reinterpret_cast<uintptr_t>(iv->q_pos) & 3u) || (reinterpret_cast<uintptr_t>(iv->k_pos) & 3u))
        return fail(BAM_ERR_INVALID_ARGUMENT, "index view: misaligned array");
    m = MaskSource{bam::MASK_INDEXED, iv->q_bits, iv->k_bits, iv->q_bits_stride_b, iv->k_bits_stride_b,
                   iv->q_pos,         iv->k_pos,  nullptr,             iv->Sq,              iv->Sk};
    return BAM_OK;
}

// bias may be null.  The kernels read groups of four keys with one access when base and strides allow it.
int fill_bias(bam::AttnParams& p, const char* who, const bam_bias* bias, int Sk) {
    if (bias == nullptr) return BAM_OK;  // p.bias stays null
    if (bias->ptr == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: bias: null pointer", who);
    const int esz = bias->is_f32 ? 4 : 2;
    if (reinterpret_cast<uintptr_t>(bias->ptr) % esz) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: bias: misaligned pointer", who);
    p.bias = bias->ptr;
    p.bias_sb = bias->stride_b;
    p.bias_sh = bias->stride_h;
    p.bias_sm = bias->stride_m;
    p.bias_f32 = bias->is_f32 ? 1 : 0;
    p.bias_vec = (reinterpret_cast<uintptr_t>(bias->ptr) % (4 * esz) == 0) && (bias->stride_b % 4 == 0) &&
                 (bias->stride_h % 4 == 0) && (bias->stride_m % 4 == 0) && (Sk % 4 == 0);
    return BAM_OK;
}

// plan may be null.  It must have been built for this very (B, Sq, Sk).
int fill_plan(bam::AttnParams& p, const char* who, const bam_plan* plan, int B, int Sq, int Sk) {
    if (plan == nullptr) return BAM_OK;  // p.fine stays null
    if (plan->fine == nullptr || plan->order == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: null array", who);
    if (plan->B != B || plan->Sq != Sq || plan->Sk != Sk)
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan was built for B = %d, Sq = %d, Sk = %d, not B = %d, Sq = %d, Sk = %d",
                    who, plan->B, plan->Sq, plan->Sk, B, Sq, Sk);
    if (plan->rows != nullptr) {
        if (p.mask_mode != bam::MASK_BITFIELD)
            return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: sorted rows are for bitfield attention only", who);
        if (plan->rows_bits == nullptr || plan->rows_moved == nullptr || (reinterpret_cast<uintptr_t>(plan->rows_moved) & 3u) || (reinterpret_cast<uintptr_t>(plan->rows) & 3u) || (reinterpret_cast<uintptr_t>(plan->rows_bits) & 7u))
            return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: null or misaligned array of sorted rows", who);
        if (bam::dkdv_far(p)) return BAM_OK;  // such rows are not gathered: from the flags alone
        p.rows = plan->rows;
        p.rows_bits = plan->rows_bits;
        p.rows_sb = plan->rows_stride_b;
        p.rows_moved = plan->rows_moved;
        p.rows_known = plan->rows_known;
    }
    if (plan->generation != 0) {  // laid out in the built-in array of bam_tile_plan_static
        int dev = -1;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices ||
            plan->fine != (const uint8_t*)g_static_plan_ptr[dev].load() ||
            plan->generation != g_static_plan_generation[dev].load())
            return fail(BAM_ERR_INVALID_ARGUMENT,
                        "%s: plan of bam_tile_plan_static is stale (a later call on this GPU has reused the built-in array)",
                        who);
    }
    if (reinterpret_cast<uintptr_t>(plan->order) & 3u) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: misaligned order", who);
    p.fine = plan->fine;
    p.fine_sb = plan->fine_stride_b;
    p.fine_ss = plan->fine_stride_s;
    // (a caller may lay the classes out by itself: rows of ceil(Sk / 32) bytes, at any address)
    p.fine_words = plan->fine_stride_s >= 4 * (((int64_t)Sk + 127) / 128) &&
                   ((reinterpret_cast<uintptr_t>(plan->fine) | (uintptr_t)plan->fine_stride_b | (uintptr_t)plan->fine_stride_s) & 3u) == 0;
    p.order = plan->order;
    p.order_sb = plan->order_stride_b;
    p.tile_order = plan->ds_tile_order;  // may be null
    if (reinterpret_cast<uintptr_t>(plan->group_order) & 3u)
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: misaligned group order", who);
    p.group_order = plan->group_order;   // may be null
    // hand-over of dS from dK/dV to dQ: only with a workspace, for the head dim and lengths its kernels cover
    if (plan->ds_workspace != nullptr && plan->ds_entry != nullptr && plan->ds_tile_base != nullptr && p.D > 64 &&
        Sk <= bam::MAX_LIST * 64 && !bam::dkdv_far(p)) {
        if (reinterpret_cast<uintptr_t>(plan->ds_workspace) & 15u)
            return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: dS workspace is not 16-byte aligned", who);
        if (plan->ds_capacity <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: dS workspace without a capacity", who);
        if ((int64_t)p.Hq * plan->ds_capacity > 0x7FFFFFFFll)  // record numbers are 32-bit in the kernels
            return fail(BAM_ERR_UNSUPPORTED, "%s: plan: dS workspace of %lld pairs x %d heads has too many records", who,
                        (long long)plan->ds_capacity, p.Hq);
        p.ds_entry = plan->ds_entry;
        p.ds_entry_sb = plan->ds_entry_stride_b;
        p.ds_tile_base = plan->ds_tile_base;
        p.ds_ws = plan->ds_workspace;
        p.ds_capacity = plan->ds_capacity;
    }
    if (p.mask_mode == bam::MASK_DENSE && plan->row_bits != nullptr && plan->col_bits != nullptr) {
        if ((reinterpret_cast<uintptr_t>(plan->row_bits) | reinterpret_cast<uintptr_t>(plan->col_bits)) & 3u)
            return fail(BAM_ERR_INVALID_ARGUMENT, "%s: plan: misaligned mask bits", who);
        p.row_bits = plan->row_bits;
        p.row_bits_sb = plan->row_bits_stride_b;
        p.row_bits_sn = plan->row_bits_stride_n;
        p.col_bits = plan->col_bits;
        p.col_bits_sb = plan->col_bits_stride_b;
        p.col_bits_ss = plan->col_bits_stride_s;
    }
    return BAM_OK;
}

void fill_sizes(bam::AttnParams& p, const MaskSource& m, int B, int Hq, int Hkv, int D, float scale) {
    p.bfq = m.bfq;
    p.bfk = m.bfk;
    p.bfq_sb = m.bfq_sb;
    p.bfk_sb = m.bfk_sb;
    p.posq = m.posq;
    p.posk = m.posk;
    p.mask = m.mask;
    p.mask_mode = m.mode;
    p.B = B;
    p.Sq = m.Sq;
    p.Sk = m.Sk;
    p.Hq = Hq;
    p.Hkv = Hkv;
    p.D = D <= 32 ? 32 : D <= 64 ? 64 : D <= 96 ? 96 : 128;
    p.d = D;
    p.num_m = (m.Sq + 127) / 128;
    p.num_n = (m.Sk + 31) / 32;
    p.num_kt = (m.Sk + 127) / 128;
    p.Sq_rounded = p.num_m * 128;
    p.lse_sb = (int64_t)Hq * p.Sq_rounded;
    p.scale = scale;
}

int fwd_impl(const char* who, const void* q, const void* k, const void* v, void* o, float* lse, const MaskSource& m,
             const int8_t* flags, const int64_t* st, int64_t flags_stride_b, int64_t flags_stride_m, int B, int Hq,
             int Hkv, int D, float scale, int dtype, const bam_bias* bias, const bam_plan* plan, void* stream,
             bool any_dim = false);
int bwd_params(bam::AttnParams& p, const char* who, const void* q, const void* k, const void* v, const void* dout,
               const float* lse, const float* delta, void* dq, void* dk, void* dv, const MaskSource& m,
               const int8_t* flags, const int64_t* st, int B, int Hq, int Hkv, int D, float scale, int dtype,
               int accumulate, bool need_dq, bool need_dkdv, const bam_bias* bias, const bam_plan* plan, bool any_dim = false);

}  // namespace

#define BAM_TRY(expr)             \
    do {                          \
        int rc_ = (expr);         \
        if (rc_ != BAM_OK) return rc_; \
    } while (0)

namespace {

int fwd_impl(const char* who, const void* q, const void* k, const void* v, void* o, float* lse, const MaskSource& m,
             const int8_t* flags, const int64_t* st, int64_t flags_stride_b, int64_t flags_stride_m, int B, int Hq,
             int Hkv, int D, float scale, int dtype, const bam_bias* bias, const bam_plan* plan, void* stream,
             bool any_dim) {
    BAM_TRY(check_problem(B, m.Sq, m.Sk, Hq, Hkv, D, dtype, any_dim));
    BAM_TRY(check_half_tensor("q", q, st[0], st[1], st[2]));
    BAM_TRY(check_half_tensor("k", k, st[3], st[4], st[5]));
    BAM_TRY(check_half_tensor("v", v, st[6], st[7], st[8]));
    BAM_TRY(check_half_tensor("o", o, st[9], st[10], st[11]));
    if (lse == nullptr || flags == nullptr || (m.mode != bam::MASK_DENSE && (m.bfq == nullptr || m.bfk == nullptr)))
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: lse, bitfields and flags must not be null", who);
    if (!(scale > 0.f)) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: softmax scale must be > 0 (got %g)", who, scale);
    bam::AttnParams p = {};
    p.q = {q, st[0], st[1], st[2]};
    p.k = {k, st[3], st[4], st[5]};
    p.v = {v, st[6], st[7], st[8]};
    p.o = {o, st[9], st[10], st[11]};
    p.lse = lse;
    p.flags = flags;
    p.flags_sb = flags_stride_b;
    p.flags_sm = flags_stride_m;
    fill_sizes(p, m, B, Hq, Hkv, D, scale);
    BAM_TRY(fill_bias(p, who, bias, m.Sk));
    BAM_TRY(fill_plan(p, who, plan, B, m.Sq, m.Sk));
    return launched(bam::launch_fwd(p, dtype, (hipStream_t)stream), who);
}

// st: strides of q, k, v, do, dq, dk, dv (3 each), then flags_stride_b, flags_stride_m
int bwd_params(bam::AttnParams& p, const char* who, const void* q, const void* k, const void* v, const void* dout,
               const float* lse, const float* delta, void* dq, void* dk, void* dv, const MaskSource& m,
               const int8_t* flags, const int64_t* st, int B, int Hq, int Hkv, int D, float scale, int dtype,
               int accumulate, bool need_dq, bool need_dkdv, const bam_bias* bias, const bam_plan* plan, bool any_dim) {
    BAM_TRY(check_problem(B, m.Sq, m.Sk, Hq, Hkv, D, dtype, any_dim));
    BAM_TRY(check_half_tensor("q", q, st[0], st[1], st[2]));
    BAM_TRY(check_half_tensor("k", k, st[3], st[4], st[5]));
    BAM_TRY(check_half_tensor("v", v, st[6], st[7], st[8]));
    BAM_TRY(check_half_tensor("do", dout, st[9], st[10], st[11]));
    if (accumulate) {
        if (need_dq) BAM_TRY(check_f32_tensor("dq", dq, st[12], st[13], st[14]));
        if (need_dkdv) {
            BAM_TRY(check_f32_tensor("dk", dk, st[15], st[16], st[17]));
            BAM_TRY(check_f32_tensor("dv", dv, st[18], st[19], st[20]));
        }
    } else {
        if (need_dq) BAM_TRY(check_half_tensor("dq", dq, st[12], st[13], st[14]));
        if (need_dkdv) {
            BAM_TRY(check_half_tensor("dk", dk, st[15], st[16], st[17]));
            BAM_TRY(check_half_tensor("dv", dv, st[18], st[19], st[20]));
        }
    }
    p.grad_typed = accumulate ? 0 : 1;
    if (lse == nullptr || delta == nullptr || flags == nullptr ||
        (m.mode != bam::MASK_DENSE && (m.bfq == nullptr || m.bfk == nullptr)))
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: lse, delta, bitfields and flags must not be null", who);
    if (!(scale > 0.f)) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: softmax scale must be > 0 (got %g)", who, scale);
    p.q = {q, st[0], st[1], st[2]};
    p.k = {k, st[3], st[4], st[5]};
    p.v = {v, st[6], st[7], st[8]};
    p.dout = {dout, st[9], st[10], st[11]};
    p.dq = {dq, st[12], st[13], st[14]};
    p.dk = {dk, st[15], st[16], st[17]};
    p.dv = {dv, st[18], st[19], st[20]};
    p.lse = const_cast<float*>(lse);
    p.delta = const_cast<float*>(delta);
    p.flags = flags;
    p.flags_sb = st[21];
    p.flags_sm = st[22];
    fill_sizes(p, m, B, Hq, Hkv, D, scale);
    BAM_TRY(fill_plan(p, who, plan, B, m.Sq, m.Sk));
    return fill_bias(p, who, bias, m.Sk);
}

// with a dS workspace in the plan, dK/dV stores its dS blocks and dQ is computed from them
int launch_dkdv(const bam::AttnParams& p, int dtype, void* stream) {
    return p.ds_ws != nullptr ? bam::launch_bwd_dkdv_save(p, dtype, (hipStream_t)stream)
                              : bam::launch_bwd_dkdv(p, dtype, (hipStream_t)stream);
}
int launch_dq(const bam::AttnParams& p, int dtype, void* stream) {
    return p.ds_ws != nullptr ? bam::launch_bwd_dq_saved(p, dtype, (hipStream_t)stream)
                              : bam::launch_bwd_dq(p, dtype, (hipStream_t)stream);
}

}  // namespace

extern "C" {

const char* bam_last_error(void) { return g_error; }

int bam_abi_version(void) { return 16; }

int bam_tile_flags(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                   int64_t flags_stride_m, int B, int S, void* stream) {
    if (bf == nullptr || flags == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_tile_flags: null pointer");
    if (B <= 0 || S <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_tile_flags: B and S must be positive");
    if (B > 65535 || (S + 127) / 128 > 65535)
        return fail(BAM_ERR_UNSUPPORTED, "bam_tile_flags: grid too large (B = %d, S = %d)", B, S);
    return launched(bam::launch_tile_flags(bf, bf_stride_b, flags, flags_stride_b, flags_stride_m, B, S,
                                           (hipStream_t)stream),
                    "bam_tile_flags");
}

namespace {
// workspace layout: fine | order, each part 256-byte aligned
struct PlanLayout {
    int64_t fine_ss, fine_sb, order_sb, entry_sb, fine_off, order_off, entry_off, base_off, count_off, bytes;
    int64_t row_sn, row_sb, col_ss, col_sb, row_off, col_off, bytes_with_bits, tile_count_off, tile_order_off;
    int64_t group_count_off, group_order_off, row_workloads_off;
    int64_t rows_sb, rows_off, rows_bits_off, rows_moved_off, bytes_with_rows;
};
PlanLayout plan_layout(int B, int Sq, int Sk) {
    const int64_t num_m = (Sq + 127) / 128, num_n = (Sk + 31) / 32, slots = 4 * num_m;
    auto up = [](int64_t x, int64_t a) { return (x + a - 1) / a * a; };
    PlanLayout l;
    l.fine_ss = up(num_n, 16);
    l.fine_sb = slots * l.fine_ss;
    l.order_sb = slots;
    l.fine_off = 0;
    l.order_off = up(B * l.fine_sb, 256);
    l.entry_sb = slots * ((Sk + 127) / 128);
    l.entry_off = l.order_off + up(B * slots * 4, 256);
    l.base_off = l.entry_off + up(B * l.entry_sb * 4, 256);
    l.count_off = l.base_off + up(B * ((Sk + 127) / 128) * 4, 256);
    l.tile_count_off = l.count_off + 256;
    l.tile_order_off = l.tile_count_off + up(B * ((Sk + 127) / 128) * 4, 256);
    l.group_count_off = l.tile_order_off + up(B * ((Sk + 127) / 128) * 4, 256);
    l.group_order_off = l.group_count_off + up(B * num_m * 4, 256);
    l.row_workloads_off = l.group_order_off + up((B * num_m + 1) * 4, 256);
    l.bytes = l.row_workloads_off + up(num_m * 8, 256);
    // the packed mask of bam_mask_tile_plan: rows padded to 128, keys to 128, 32-key blocks to an even number
    l.row_sn = num_m * 128;
    l.row_sb = ((num_n + 1) & ~(int64_t)1) * l.row_sn;
    l.col_ss = ((Sk + 127) / 128) * 128;
    l.col_sb = slots * l.col_ss;
    l.row_off = l.bytes;
    l.col_off = l.row_off + up(B * l.row_sb * 4, 256);
    l.bytes_with_bits = l.col_off + up(B * l.col_sb * 4, 256);
    // the sorted rows of bam_tile_plan_sorted_counted
    l.rows_sb = num_m * 128;
    l.rows_off = l.bytes;
    l.rows_bits_off = l.rows_off + up(B * l.rows_sb * 4, 256);
    l.rows_moved_off = l.rows_bits_off + up(B * l.rows_sb * 8, 256);
    l.bytes_with_rows = l.rows_moved_off + up(B * 4, 256);
    return l;
}
}  // namespace

int64_t bam_plan_workspace_bytes_rect(int B, int Sq, int Sk) {
    if (B <= 0 || Sq <= 0 || Sk <= 0 || (Sq + 31) / 32 > bam::MAX_PLAN_SLICES || Sk > BAM_MAX_SEQLEN) return 0;
    return plan_layout(B, Sq, Sk).bytes;
}

int bam_sorted_plan_workspace_bytes(int B, int S, int64_t* bytes) {
    if (bytes == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_sorted_plan_workspace_bytes: null pointer");
    *bytes = bam_plan_workspace_bytes_rect(B, S, S) == 0 ? 0 : plan_layout(B, S, S).bytes_with_rows;
    return BAM_OK;
}

int64_t bam_plan_workspace_bytes(int B, int S) { return bam_plan_workspace_bytes_rect(B, S, S); }

int64_t bam_mask_plan_workspace_bytes(int B, int Sq, int Sk) {
    if (bam_plan_workspace_bytes_rect(B, Sq, Sk) == 0) return 0;
    return plan_layout(B, Sq, Sk).bytes_with_bits;
}

namespace {
// Checks the workspace and lays the plan's arrays out in it.
int place_plan(const char* who, void* workspace, int64_t workspace_bytes, int B, int Sq, int Sk, bam_plan* plan,
               PlanLayout& l, bool with_bits = false, bool with_rows = false) {
    if (workspace == nullptr || plan == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
    int64_t need = with_bits ? bam_mask_plan_workspace_bytes(B, Sq, Sk) : bam_plan_workspace_bytes_rect(B, Sq, Sk);
    if (with_rows) BAM_TRY(bam_sorted_plan_workspace_bytes(B, Sq, &need));
    if (need == 0) return fail(BAM_ERR_UNSUPPORTED, "%s: no plan is built for Sq = %d, Sk = %d", who, Sq, Sk);
    if (workspace_bytes < need)
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: workspace of %lld bytes, %lld needed", who, (long long)workspace_bytes,
                    (long long)need);
    if (reinterpret_cast<uintptr_t>(workspace) & 255u)
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: workspace is not 256-byte aligned", who);
    l = plan_layout(B, Sq, Sk);
    char* w = (char*)workspace;
    plan->fine = (const uint8_t*)(w + l.fine_off);
    plan->fine_stride_b = l.fine_sb;
    plan->fine_stride_s = l.fine_ss;
    plan->order = (const int32_t*)(w + l.order_off);
    plan->order_stride_b = l.order_sb;
    plan->ds_entry = (const int32_t*)(w + l.entry_off);
    plan->ds_entry_stride_b = l.entry_sb;
    plan->ds_tile_base = (const int32_t*)(w + l.base_off);
    plan->ds_count = (const int32_t*)(w + l.count_off);
    plan->ds_tile_order = (int64_t)B * ((Sk + 127) / 128) <= bam::MAX_RANKED ? (const int32_t*)(w + l.tile_order_off) : nullptr;
    plan->group_order = (int64_t)B * ((Sq + 127) / 128) <= bam::MAX_RANKED ? (const int32_t*)(w + l.group_order_off) : nullptr;
    plan->row_workloads = with_rows ? nullptr : (const int64_t*)(w + l.row_workloads_off);
    plan->rows = with_rows ? (const int32_t*)(w + l.rows_off) : nullptr;
    plan->rows_bits = with_rows ? (const int64_t*)(w + l.rows_bits_off) : nullptr;
    plan->rows_stride_b = with_rows ? l.rows_sb : 0;
    plan->rows_moved = with_rows ? (const int32_t*)(w + l.rows_moved_off) : nullptr;
    plan->rows_known = BAM_ROWS_UNKNOWN;
    plan->reserved = 0;
    plan->ds_workspace = nullptr;
    plan->ds_capacity = 0;
    plan->row_bits = with_bits ? (const uint32_t*)(w + l.row_off) : nullptr;
    plan->row_bits_stride_b = with_bits ? l.row_sb : 0;
    plan->row_bits_stride_n = with_bits ? l.row_sn : 0;
    plan->col_bits = with_bits ? (const uint32_t*)(w + l.col_off) : nullptr;
    plan->col_bits_stride_b = with_bits ? l.col_sb : 0;
    plan->col_bits_stride_s = with_bits ? l.col_ss : 0;
    plan->B = B;
    plan->Sq = Sq;
    plan->Sk = Sk;
    plan->generation = 0;
    return BAM_OK;
}

// second launch of every plan builder: numbers the (slice, 128-key tile) pairs that have work
int number_pairs(const char* who, const bam_plan* plan, const PlanLayout& l, void* workspace, uint64_t* count_host,
                 uint32_t count_tag, void* stream) {
    return launched(bam::launch_ds_entries(plan->fine, plan->fine_stride_b, plan->fine_stride_s, plan->B, plan->Sq, plan->Sk,
                                           const_cast<int*>(plan->ds_entry), plan->ds_entry_stride_b,
                                           const_cast<int*>(plan->ds_tile_base),
                                           const_cast<int*>(plan->ds_count),
                                           (int*)((char*)workspace + l.tile_count_off),
                                           const_cast<int*>(plan->ds_tile_order), plan->order, plan->order_stride_b,
                                           (int*)((char*)workspace + l.group_count_off),
                                           const_cast<int*>(plan->group_order),
                                           const_cast<int64_t*>(plan->row_workloads), plan->rows_moved, count_host, count_tag,
                                           (hipStream_t)stream),
                    who);
}
}  // namespace

int bam_tile_plan(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                  int64_t flags_stride_m, void* workspace, int64_t workspace_bytes, int B, int S, bam_plan* plan,
                  void* stream) {
    return bam_tile_plan_counted(bf, bf_stride_b, flags, flags_stride_b, flags_stride_m, workspace, workspace_bytes, B, S, plan,
                                 nullptr, 0, stream);
}

int bam_tile_plan_counted(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                          int64_t flags_stride_m, void* workspace, int64_t workspace_bytes, int B, int S, bam_plan* plan,
                          uint64_t* count_host, uint32_t count_tag, void* stream) {
    if (bf == nullptr || flags == nullptr || workspace == nullptr || plan == nullptr)
        return fail(BAM_ERR_INVALID_ARGUMENT, "bam_tile_plan: null pointer");
    if (B <= 0 || S <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_tile_plan: B and S must be positive");
    if (B > 65535 || (S + 127) / 128 > 65535)
        return fail(BAM_ERR_UNSUPPORTED, "bam_tile_plan: grid too large (B = %d, S = %d)", B, S);
    PlanLayout l;
    BAM_TRY(place_plan("bam_tile_plan", workspace, workspace_bytes, B, S, S, plan, l));
    char* w = (char*)workspace;
    BAM_TRY(launched(bam::launch_tile_plan(bf, bf_stride_b, flags, flags_stride_b, flags_stride_m, (uint8_t*)(w + l.fine_off),
                                           l.fine_sb, l.fine_ss, (int*)(w + l.order_off), l.order_sb,
                                           (int*)(w + l.count_off), B, S, (hipStream_t)stream),
                     "bam_tile_plan"));
    return number_pairs("bam_tile_plan", plan, l, workspace, count_host, count_tag, stream);
}

int bam_tile_plan_sorted_counted(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                                 int64_t flags_stride_m, void* workspace, int64_t workspace_bytes, int B, int S, bam_plan* plan,
                                 uint64_t* count_host, uint32_t count_tag, void* stream) {
    const char* who = "bam_tile_plan_sorted_counted";
    if (bf == nullptr || flags == nullptr || workspace == nullptr || plan == nullptr)
        return fail(BAM_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
    if (B <= 0 || S <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: B and S must be positive", who);
    if (B > 65535) return fail(BAM_ERR_UNSUPPORTED, "%s: grid too large (B = %d, S = %d)", who, B, S);
    if ((int64_t)B * ((S + 31) / 32) * ((S + 127) / 128) >= 1ll << 30)
        return fail(BAM_ERR_UNSUPPORTED, "%s: too many pairs of slices and key tiles (B = %d, S = %d)", who, B, S);
    PlanLayout l;
    BAM_TRY(place_plan(who, workspace, workspace_bytes, B, S, S, plan, l, false, true));
    char* w = (char*)workspace;
    BAM_TRY(launched(bam::launch_sorted_plan(bf, bf_stride_b, flags, flags_stride_b, flags_stride_m, (int*)(w + l.rows_off), (int64_t*)(w + l.rows_bits_off), l.rows_sb,
                                             (int*)(w + l.rows_moved_off), (uint8_t*)(w + l.fine_off), l.fine_sb, l.fine_ss, (int*)(w + l.order_off), l.order_sb,
                                             (int*)(w + l.count_off), B, S, (hipStream_t)stream),
                     who));
    return number_pairs(who, plan, l, workspace, count_host, count_tag, stream);
}

int bam_tile_plan_static(const int64_t* bf, int64_t bf_stride_b, int8_t* flags, int64_t flags_stride_b,
                         int64_t flags_stride_m, int B, int S, bam_plan* plan, void* stream) {
    if (B <= 0 || S <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_tile_plan_static: B and S must be positive");
    const int64_t need = bam_plan_workspace_bytes(B, S);
    if (need == 0 || need > BAM_STATIC_PLAN_BYTES)
        return fail(BAM_ERR_UNSUPPORTED,
                    "bam_tile_plan_static: B = %d, S = %d needs a plan workspace of %lld bytes, the built-in one holds %lld "
                    "(use bam_tile_plan with a workspace of your own)",
                    B, S, (long long)need, (long long)BAM_STATIC_PLAN_BYTES);
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(BAM_ERR_LAUNCH, "bam_tile_plan_static: no current device (or more than %d devices)", kMaxDevices);
    void* ptr = g_static_plan_ptr[dev].load(std::memory_order_acquire);
    if (ptr == nullptr) {
        // once per device, with that device current: the array's own address on this GPU
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_static_plan_scratch));
        if (e != hipSuccess || ptr == nullptr)
            return fail(BAM_ERR_LAUNCH, "bam_tile_plan_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
        g_static_plan_ptr[dev].store(ptr, std::memory_order_release);
    }
    BAM_TRY(bam_tile_plan(bf, bf_stride_b, flags, flags_stride_b, flags_stride_m, ptr, BAM_STATIC_PLAN_BYTES, B, S, plan,
                          stream));
    int32_t gen = g_static_plan_generation[dev].fetch_add(1) + 1;
    if (gen <= 0) g_static_plan_generation[dev].store(gen = 1);
    plan->generation = gen;
    return BAM_OK;
}

int bam_plan_indexed(const bam_index_view* iv, void* workspace, int64_t workspace_bytes, int B, bam_plan* plan,
                     void* stream) {
    return bam_plan_indexed_counted(iv, workspace, workspace_bytes, B, plan, nullptr, 0, stream);
}

static int plan_indexed(const char* who, const bam_index_view* iv, const int64_t* bf, int64_t bf_stride_b, int L,
                        const int64_t* idx_q, const int64_t* idx_k, void* workspace, int64_t workspace_bytes, int B,
                        bam_plan* plan, uint64_t* count_host, uint32_t count_tag, void* stream) {
    MaskSource m;
    BAM_TRY(indexed_source(iv, m));
    if (B <= 0 || m.Sq <= 0 || m.Sk <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "%s: B, Sq and Sk must be positive", who);
    if (B > 65535) return fail(BAM_ERR_UNSUPPORTED, "%s: B is limited to 65535 (got %d)", who, B);
    PlanLayout l;
    BAM_TRY(place_plan(who, workspace, workspace_bytes, B, m.Sq, m.Sk, plan, l));
    char* w = (char*)workspace;
    BAM_TRY(launched(bam::launch_indexed_plan(bf, bf_stride_b, L, idx_q, idx_k, const_cast<int64_t*>(m.bfq), m.bfq_sb,
                                              const_cast<int64_t*>(m.bfk), m.bfk_sb, const_cast<int*>(m.posq),
                                              const_cast<int*>(m.posk), m.Sq, m.Sk, (uint8_t*)(w + l.fine_off), l.fine_sb,
                                              l.fine_ss, (int*)(w + l.order_off), l.order_sb, (int*)(w + l.count_off), B,
                                              (hipStream_t)stream),
                     who));
    return number_pairs(who, plan, l, workspace, count_host, count_tag, stream);
}

int bam_plan_indexed_counted(const bam_index_view* iv, void* workspace, int64_t workspace_bytes, int B, bam_plan* plan,
                             uint64_t* count_host, uint32_t count_tag, void* stream) {
    return plan_indexed("bam_plan_indexed", iv, nullptr, 0, 0, nullptr, nullptr, workspace, workspace_bytes, B, plan, count_host,
                        count_tag, stream);
}

int bam_gather_plan_indexed(const int64_t* bf, int64_t bf_stride_b, int L, const int64_t* idx_q, const int64_t* idx_k,
                            const bam_index_view* iv, void* workspace, int64_t workspace_bytes, int B, bam_plan* plan,
                            uint64_t* count_host, uint32_t count_tag, void* stream) {
    if (bf == nullptr || idx_q == nullptr || idx_k == nullptr || L <= 0)
        return fail(BAM_ERR_INVALID_ARGUMENT, "bam_gather_plan_indexed: null pointer or empty sequence");
    return plan_indexed("bam_gather_plan_indexed", iv, bf, bf_stride_b, L, idx_q, idx_k, workspace, workspace_bytes, B, plan,
                        count_host, count_tag, stream);
}

int bam_mask_tile_plan(const uint8_t* mask, int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m, void* workspace,
                       int64_t workspace_bytes, int B, int Sq, int Sk, bam_plan* plan, void* stream) {
    return bam_mask_tile_plan_counted(mask, flags, flags_stride_b, flags_stride_m, workspace, workspace_bytes, B, Sq, Sk, plan,
                                      nullptr, 0, stream);
}

int bam_mask_tile_plan_counted(const uint8_t* mask, int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m,
                               void* workspace, int64_t workspace_bytes, int B, int Sq, int Sk, bam_plan* plan,
                               uint64_t* count_host, uint32_t count_tag, void* stream) {
    if (mask == nullptr || flags == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_mask_tile_plan: null pointer");
    if (B <= 0 || Sq <= 0 || Sk <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_mask_tile_plan: B, Sq and Sk must be positive");
    if (B > 65535 || (Sq + 127) / 128 > 65535)
        return fail(BAM_ERR_UNSUPPORTED, "bam_mask_tile_plan: grid too large (B = %d, Sq = %d)", B, Sq);
    PlanLayout l;
    BAM_TRY(place_plan("bam_mask_tile_plan", workspace, workspace_bytes, B, Sq, Sk, plan, l, true));
    char* w = (char*)workspace;
    BAM_TRY(launched(bam::launch_mask_tile_plan(mask, flags, flags_stride_b, flags_stride_m, (uint8_t*)(w + l.fine_off),
                                                l.fine_sb, l.fine_ss, (int*)(w + l.order_off), l.order_sb,
                                                (int*)(w + l.count_off), (unsigned*)(w + l.row_off), l.row_sb, l.row_sn,
                                                (unsigned*)(w + l.col_off), l.col_sb, l.col_ss, B, Sq, Sk,
                                                (hipStream_t)stream),
                     "bam_mask_tile_plan"));
    return number_pairs("bam_mask_tile_plan", plan, l, workspace, count_host, count_tag, stream);
}

int64_t bam_ds_workspace_bytes(int Hq, int64_t pairs) {
    if (Hq <= 0 || pairs <= 0) return 0;
    return (int64_t)Hq * pairs * 8192;
}

int bam_materialize_mask(const int64_t* bf, int64_t bf_stride_b, uint8_t* out, int B, int S, void* stream) {
    if (bf == nullptr || out == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_materialize_mask: null pointer");
    if (B <= 0 || S <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_materialize_mask: B and S must be positive");
    if (B > 65535 || S > 65535)
        return fail(BAM_ERR_UNSUPPORTED, "bam_materialize_mask: B and S are limited to 65535 (got %d, %d)", B, S);
    return launched(bam::launch_materialize_mask(bf, bf_stride_b, out, B, S, (hipStream_t)stream),
                    "bam_materialize_mask");
}

int bam_flag_row_workloads(const int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m, int B, int num_m,
                           int num_n, int32_t* out, void* stream) {
    if (flags == nullptr || out == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_flag_row_workloads: null pointer");
    if (B <= 0 || num_m <= 0 || num_n <= 0)
        return fail(BAM_ERR_INVALID_ARGUMENT, "bam_flag_row_workloads: B, num_m and num_n must be positive");
    return launched(bam::launch_flag_row_workloads(flags, flags_stride_b, flags_stride_m, B, num_m, num_n, out,
                                                   (hipStream_t)stream),
                    "bam_flag_row_workloads");
}

int bam_gather_bitfields(const int64_t* bf, int64_t bf_stride_b, int L, const int64_t* idx, int n, int64_t* out_bits,
                         int64_t out_stride_b, int32_t* out_pos, int B, void* stream) {
    if (bf == nullptr || idx == nullptr || out_bits == nullptr || out_pos == nullptr)
        return fail(BAM_ERR_INVALID_ARGUMENT, "bam_gather_bitfields: null pointer");
    if (B <= 0 || L <= 0 || n <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_gather_bitfields: B, L and n must be positive");
    if (B > 65535) return fail(BAM_ERR_UNSUPPORTED, "bam_gather_bitfields: B is limited to 65535 (got %d)", B);
    return launched(bam::launch_gather_bitfields(bf, bf_stride_b, L, idx, n, out_bits, out_stride_b, out_pos, B,
                                                 (hipStream_t)stream),
                    "bam_gather_bitfields");
}

#define BAM_FWD_STRIDES                                                                                     \
    {q_stride_b, q_stride_s, q_stride_h, k_stride_b, k_stride_s, k_stride_h, v_stride_b, v_stride_s, v_stride_h, \
     o_stride_b, o_stride_s, o_stride_h}

int bam_fwd(const void* q, const void* k, const void* v, void* o, float* lse, const int64_t* bf,
            const int8_t* flags, int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
            int64_t k_stride_b, int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b,
            int64_t v_stride_s, int64_t v_stride_h, int64_t o_stride_b, int64_t o_stride_s,
            int64_t o_stride_h, int64_t bf_stride_b, int64_t flags_stride_b, int64_t flags_stride_m, int B,
            int S, int Hq, int Hkv, int D, float scale, int dtype, const bam_bias* bias, const bam_plan* plan,
            void* stream) {
    const int64_t st[12] = BAM_FWD_STRIDES;
    return fwd_impl("bam_fwd", q, k, v, o, lse, plain_source(bf, bf_stride_b, S), flags, st, flags_stride_b,
                    flags_stride_m, B, Hq, Hkv, D, scale, dtype, bias, plan, stream);
}

int bam_fwd_indexed(const void* q, const void* k, const void* v, void* o, float* lse, const bam_index_view* iv,
                    const int8_t* flags, int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                    int64_t k_stride_b, int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b,
                    int64_t v_stride_s, int64_t v_stride_h, int64_t o_stride_b, int64_t o_stride_s,
                    int64_t o_stride_h, int64_t flags_stride_b, int64_t flags_stride_m, int B, int Hq, int Hkv,
                    int D, float scale, int dtype, const bam_bias* bias, const bam_plan* plan,
        void* stream) {
    MaskSource m;
    BAM_TRY(indexed_source(iv, m));
    const int64_t st[12] = BAM_FWD_STRIDES;
    return fwd_impl("bam_fwd_indexed", q, k, v, o, lse, m, flags, st, flags_stride_b, flags_stride_m, B, Hq, Hkv, D,
                    scale, dtype, bias, plan, stream);
}

int bam_bwd_preprocess(const void* o, const void* dout, float* delta, int64_t o_stride_b, int64_t o_stride_s,
                       int64_t o_stride_h, int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h,
                       int B, int S, int Hq, int D, int dtype, void* stream) {
    BAM_TRY(check_problem(B, S, S, Hq, Hq, D, dtype));
    BAM_TRY(check_half_tensor("o", o, o_stride_b, o_stride_s, o_stride_h));
    BAM_TRY(check_half_tensor("do", dout, do_stride_b, do_stride_s, do_stride_h));
    if (delta == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_bwd_preprocess: delta must not be null");
    bam::AttnParams p = {};
    p.o = {o, o_stride_b, o_stride_s, o_stride_h};
    p.dout = {dout, do_stride_b, do_stride_s, do_stride_h};
    p.delta = delta;
    fill_sizes(p, plain_source(nullptr, 0, S), B, Hq, Hq, D, 1.f);  // the preprocess kernel never looks at the mask
    return launched(bam::launch_bwd_preprocess(p, dtype, (hipStream_t)stream), "bam_bwd_preprocess");
}

#define BAM_BWD_STRIDES                                                                                      \
    {q_stride_b,  q_stride_s,  q_stride_h,  k_stride_b,  k_stride_s,  k_stride_h,  v_stride_b,  v_stride_s,  \
     v_stride_h,  do_stride_b, do_stride_s, do_stride_h, dq_stride_b, dq_stride_s, dq_stride_h, dk_stride_b, \
     dk_stride_s, dk_stride_h, dv_stride_b, dv_stride_s, dv_stride_h, flags_stride_b, flags_stride_m}

int bam_bwd(const void* q, const void* k, const void* v, const void* dout, const float* lse,
            const float* delta, void* dq, void* dk, void* dv, const int64_t* bf, const int8_t* flags,
            int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b,
            int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
            int64_t v_stride_h, int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h,
            int64_t dq_stride_b, int64_t dq_stride_s, int64_t dq_stride_h, int64_t dk_stride_b,
            int64_t dk_stride_s, int64_t dk_stride_h, int64_t dv_stride_b, int64_t dv_stride_s,
            int64_t dv_stride_h, int64_t bf_stride_b, int64_t flags_stride_b, int64_t flags_stride_m, int B,
            int S, int Hq, int Hkv, int D, float scale, int dtype, int accumulate, const bam_bias* bias,
            const bam_plan* plan, void* stream) {
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd", q, k, v, dout, lse, delta, dq, dk, dv, plain_source(bf, bf_stride_b, S), flags, st, B,
                       Hq, Hkv, D, scale, dtype, accumulate, true, true, bias, plan));
    BAM_TRY(launched(launch_dkdv(p, dtype, stream), "bam_bwd (dk/dv)"));
    return launched(launch_dq(p, dtype, stream), "bam_bwd (dq)");
}

int bam_bwd_dkdv(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                 const float* delta, void* dk, void* dv, const int64_t* bf, const int8_t* flags,
                 int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b,
                 int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
                 int64_t v_stride_h, int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h,
                 int64_t dk_stride_b, int64_t dk_stride_s, int64_t dk_stride_h, int64_t dv_stride_b,
                 int64_t dv_stride_s, int64_t dv_stride_h, int64_t bf_stride_b, int64_t flags_stride_b,
                 int64_t flags_stride_m, int B, int S, int Hq, int Hkv, int D, float scale, int dtype,
                 int accumulate, const bam_bias* bias, const bam_plan* plan, void* stream) {
    void* dq = nullptr;
    const int64_t dq_stride_b = 0, dq_stride_s = 0, dq_stride_h = 0;
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd_dkdv", q, k, v, dout, lse, delta, dq, dk, dv, plain_source(bf, bf_stride_b, S), flags,
                       st, B, Hq, Hkv, D, scale, dtype, accumulate, false, true, bias, plan));
    return launched(launch_dkdv(p, dtype, stream), "bam_bwd_dkdv");
}

int bam_bwd_dq(const void* q, const void* k, const void* v, const void* dout, const float* lse,
               const float* delta, void* dq, const int64_t* bf, const int8_t* flags, int64_t q_stride_b,
               int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b, int64_t k_stride_s,
               int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s, int64_t v_stride_h,
               int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h, int64_t dq_stride_b,
               int64_t dq_stride_s, int64_t dq_stride_h, int64_t bf_stride_b, int64_t flags_stride_b,
               int64_t flags_stride_m, int B, int S, int Hq, int Hkv, int D, float scale, int dtype,
               int accumulate, const bam_bias* bias, const bam_plan* plan, void* stream) {
    void *dk = nullptr, *dv = nullptr;
    const int64_t dk_stride_b = 0, dk_stride_s = 0, dk_stride_h = 0, dv_stride_b = 0, dv_stride_s = 0, dv_stride_h = 0;
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd_dq", q, k, v, dout, lse, delta, dq, dk, dv, plain_source(bf, bf_stride_b, S), flags, st,
                       B, Hq, Hkv, D, scale, dtype, accumulate, true, false, bias, plan));
    return launched(launch_dq(p, dtype, stream), "bam_bwd_dq");
}

int bam_bwd_dkdv_indexed(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                         const float* delta, void* dk, void* dv, const bam_index_view* iv, const int8_t* flags,
                         int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b,
                         int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
                         int64_t v_stride_h, int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h,
                         int64_t dk_stride_b, int64_t dk_stride_s, int64_t dk_stride_h, int64_t dv_stride_b,
                         int64_t dv_stride_s, int64_t dv_stride_h, int64_t flags_stride_b, int64_t flags_stride_m,
                         int B, int Hq, int Hkv, int D, float scale, int dtype, int accumulate, const bam_bias* bias, const bam_plan* plan,
        void* stream) {
    MaskSource m;
    BAM_TRY(indexed_source(iv, m));
    void* dq = nullptr;
    const int64_t dq_stride_b = 0, dq_stride_s = 0, dq_stride_h = 0;
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd_dkdv_indexed", q, k, v, dout, lse, delta, dq, dk, dv, m, flags, st, B, Hq, Hkv, D, scale,
                       dtype, accumulate, false, true, bias, plan));
    return launched(launch_dkdv(p, dtype, stream), "bam_bwd_dkdv_indexed");
}

int bam_bwd_dq_indexed(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                       const float* delta, void* dq, const bam_index_view* iv, const int8_t* flags,
                       int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b,
                       int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
                       int64_t v_stride_h, int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h,
                       int64_t dq_stride_b, int64_t dq_stride_s, int64_t dq_stride_h, int64_t flags_stride_b,
                       int64_t flags_stride_m, int B, int Hq, int Hkv, int D, float scale, int dtype,
                       int accumulate, const bam_bias* bias, const bam_plan* plan,
        void* stream) {
    MaskSource m;
    BAM_TRY(indexed_source(iv, m));
    void *dk = nullptr, *dv = nullptr;
    const int64_t dk_stride_b = 0, dk_stride_s = 0, dk_stride_h = 0, dv_stride_b = 0, dv_stride_s = 0, dv_stride_h = 0;
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd_dq_indexed", q, k, v, dout, lse, delta, dq, dk, dv, m, flags, st, B, Hq, Hkv, D, scale,
                       dtype, accumulate, true, false, bias, plan));
    return launched(launch_dq(p, dtype, stream), "bam_bwd_dq_indexed");
}

// ---- the struct form of the attention calls
static int attn_source(const bam_attn* a, MaskSource& m) {
    if (a->mode == BAM_MASK_INDEXED) return indexed_source(a->index, m);
    if (a->mode == BAM_MASK_DENSE) {
        BAM_TRY(check_mask("bam_attn", a->mask));
        m = dense_source(a->mask, a->Sq, a->Sk);
        return BAM_OK;
    }
    if (a->mode != BAM_MASK_BITFIELD) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn: unknown mode %d", a->mode);
    if (a->Sq != a->Sk) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn: Sq and Sk must match in bitfield mode");
    m = plain_source(a->bf, a->bf_stride_b, a->Sq);
    return BAM_OK;
}

int bam_attn_fwd(const bam_attn* a, void* stream) {
    if (a == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_fwd: null pointer");
    MaskSource m;
    BAM_TRY(attn_source(a, m));
    const int64_t st[12] = {a->q.stride_b, a->q.stride_s, a->q.stride_h, a->k.stride_b, a->k.stride_s, a->k.stride_h,
                            a->v.stride_b, a->v.stride_s, a->v.stride_h, a->o.stride_b, a->o.stride_s, a->o.stride_h};
    return fwd_impl("bam_attn_fwd", a->q.ptr, a->k.ptr, a->v.ptr, a->o.ptr, a->lse, m, a->flags, st, a->flags_stride_b,
                    a->flags_stride_m, a->B, a->Hq, a->Hkv, a->D, a->scale, a->dtype, a->bias, a->plan, stream, true);
}

// How many workgroups share the q heads of a kv head in dK/dV.  One workgroup per (key tile, kv head) walks all of them one after
// the other and the launch lasts as long as the first key tile's; dealt to parts, the tiles level out over the 256 compute units.
// The price is fp32 sums through memory and a launch that adds them.  The estimate, in us: a step over a pair of slices takes
// `step`, a workgroup kStart steps besides, tiles fall off linearly in length (as a causal mask's do, or less where the plan's pairs
// are known to be more, or there is no mask); the launch takes the longest workgroup, or the work per compute unit and kTail of the
// longest, or (level lists: what the causal fit has in kTail) what a compute unit takes that gets k + 1 of the 256 k + 1 longest.
// Fitted to 42 training steps with segments (D 32, 64, 128; 6 to 32 q heads, 1 to 8 kv heads, 300 to 9000 tokens), of which it takes
// the fastest number of parts, or one within 5 %; gains of a few per cent are not there (1 x 16384 tokens, 2 parts: dK/dV 4115 ->
// 4069 and 56 for the sum).  One part -> parts, kernels of a step, us, 32 / 8 heads, D 128: 2 x 700 147 -> 120 (4), 2500 380 -> 305
// (2), 3001 453 -> 355 (2), 5000 861 -> 790 (2), but 4 x 1537 (416 workgroups) 412 -> 445; 16 / 4 heads, 9000 tokens 1404 -> 1255;
// D 64: 3001 tokens 322 -> 256, 5000 560 -> 513.  At least 32 steps have to go: below, the host is what a training step waits for
// (4 x 400 tokens, 6 / 1 heads, D 40, 35 steps: 94 -> 58 to 98 us with the speed of the host; 2 x 283, 6 / 2 heads, 10 steps: 86 ->
// 91; 300 tokens, 32 / 8 heads, 15 steps: kernels 87 -> 68, not taken).
// Nothing hidden, backward, us, 32 / 8 heads, D 128, parts of the causal estimate -> of the known lists: 2500 tokens 434 (2) -> 405
// (1), 3001 526 (2) -> 496 (1), 2 x 1537 311 (2) -> 287 (1), 5000 1336 (2) -> 1282 (4); no mask: 2500 479 (2) -> 424 (1).
// Up to D 64 the host does not wait for the pairs, so a mask that hides nothing gets the causal estimate's parts: D 64, 3001 tokens
// one part 314, two 330, 4096 501 / 506, but 5000 983 / 821.
static int dkdv_parts(const bam_attn* a) {
    if (a->head_runs > 1 || a->B <= 0 || a->Sk <= 0 || a->Hkv <= 0 || a->Hq <= a->Hkv || a->Hq % a->Hkv || a->Sq > bam::MAX_SLICE_LIST * 32)
        return 1;
    if (bam::far_rows(a->q.stride_s, a->Sq, a->D) || bam::far_rows(a->dout.stride_s, a->Sq, a->D) ||
        bam::far_rows(a->k.stride_s, a->Sk, a->D) || bam::far_rows(a->v.stride_s, a->Sk, a->D))
        return 1;  // (the instantiation for such rows has no parts)
    const int G = a->Hq / a->Hkv;
    const double tiles = (a->Sk + 127) / 128, pairs = (a->Sq + 63) / 64, step = a->D > 96 ? 1.25 : a->D > 64 ? 1.1 : a->D > 32 ? 0.79 : 0.63;
    constexpr double kStart = 7.8, kTail = 0.28, kBytesPerUs = 8.7e6, kLaunch = 6;  // (the parts stay in the last-level cache)
    const double units = a->B * (double)a->Hkv * tiles, rows = (double)a->B * a->Sk * a->Hkv;
    double mean = a->mode == BAM_MASK_DENSE && a->mask == nullptr ? pairs : (pairs + 1) / 2;
    if (a->pairs > 0) mean = std::min(pairs, std::max(mean, a->pairs / (2.0 * a->B * tiles)));
    auto estimate = [&](int parts) {
        const double longest = pairs * G / parts, share = units * (mean * G + kStart * parts) / 256 + kTail * longest;
        double time = longest + kStart > share ? longest + kStart : share;
        for (int k = 1; mean > (pairs + 1) / 2 && k <= 8 && 256 * k < units * parts; ++k)
            time = std::max(time, (k + 1) * (longest - 2 * (longest - mean * G / parts) * 256 * k / (units * parts) + kStart));
        return step * time + (parts > 1 ? kLaunch + 2 * 2 * 4 * rows * a->D * parts / kBytesPerUs : 0);
    };
    const double one = estimate(1);
    int best = 1;
    double least = one - (one > 130 ? 0.06 * one : 8);  // the host's launch and allocation have to come out, and the estimate's error
    for (int parts = 2; parts <= G; ++parts) {
        if (G % parts || 2 * 4 * rows * a->D * parts > 1e9 || units * parts > 1e6) continue;
        if ((G - G / parts) * pairs < 32) continue;
        const double t = estimate(parts);
        if (t < least) {
            least = t;
            best = parts;
        }
    }
    return best;
}
static int64_t dkdv_part_floats(const bam_attn* a, int parts) { return (int64_t)a->B * a->Sk * a->Hkv * parts * a->D; }

int bam_attn_bwd_parts(const bam_attn* a, int64_t* bytes) {
    if (a == nullptr || bytes == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_bwd_parts: null pointer");
    const int parts = dkdv_parts(a);
    *bytes = parts > 1 ? 2 * 4 * dkdv_part_floats(a, parts) : 0;
    return BAM_OK;
}

// The parameters of a backward, all heads at once, with the plan and the workspace of `a` (plan: where they are put together).
static int attn_bwd_params(const bam_attn* a, bam_plan& plan, bam::AttnParams& all) {
    MaskSource m;
    BAM_TRY(attn_source(a, m));
    BAM_TRY(check_problem(a->B, m.Sq, m.Sk, a->Hq, a->Hkv, a->D, a->dtype, true));
    BAM_TRY(check_half_tensor("o", a->o.ptr, a->o.stride_b, a->o.stride_s, a->o.stride_h));
    BAM_TRY(check_half_tensor("do", a->dout.ptr, a->dout.stride_b, a->dout.stride_s, a->dout.stride_h));
    const int runs = a->head_runs > 1 ? a->head_runs : 1;
    if (a->Hkv % runs) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_bwd: %d runs do not divide %d kv heads", runs, a->Hkv);
    if (runs > 1 && a->bias != nullptr)  // a bias is indexed by absolute head
        return fail(BAM_ERR_UNSUPPORTED, "bam_attn_bwd: heads are not taken in runs with a bias");
    if (a->plan != nullptr) {
        plan = *a->plan;
        plan.ds_workspace = a->ds_workspace;
        plan.ds_capacity = a->ds_capacity;
    }
    const int64_t st[23] = {a->q.stride_b,    a->q.stride_s,    a->q.stride_h,    a->k.stride_b,  a->k.stride_s,  a->k.stride_h,
                            a->v.stride_b,    a->v.stride_s,    a->v.stride_h,    a->dout.stride_b, a->dout.stride_s,
                            a->dout.stride_h, a->dq.stride_b,   a->dq.stride_s,   a->dq.stride_h, a->dk.stride_b, a->dk.stride_s,
                            a->dk.stride_h,   a->dv.stride_b,   a->dv.stride_s,   a->dv.stride_h, a->flags_stride_b,
                            a->flags_stride_m};
    BAM_TRY(bwd_params(all, "bam_attn_bwd", a->q.ptr, a->k.ptr, a->v.ptr, a->dout.ptr, a->lse, a->delta, a->dq.ptr, a->dk.ptr,
                       a->dv.ptr, m, a->flags, st, a->B, a->Hq, a->Hkv, a->D, a->scale, a->dtype, a->accumulate, true, true,
                       a->bias, nullptr, true));
    all.o = {a->o.ptr, a->o.stride_b, a->o.stride_s, a->o.stride_h};
    if (reinterpret_cast<uintptr_t>(a->lse_scaled) & 3u)
        return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_bwd: lse_scaled is not 4-byte aligned");
    all.lse_scaled = a->bias == nullptr && all.D <= 64 ? a->lse_scaled : nullptr;
    // (a run's workspace is checked with the run's heads)
    if (a->plan != nullptr && runs == 1) BAM_TRY(fill_plan(all, "bam_attn_bwd", &plan, a->B, m.Sq, m.Sk));
    return BAM_OK;
}
static bool attn_bwd_one_launch(const bam_attn* a, const bam::AttnParams& all, int parts) {
    return a->head_runs <= 1 && bam::both_in_one_launch(all, (int64_t)all.num_kt * all.B * all.Hkv * parts, a->pairs);
}

int bam_attn_bwd_takes_ds(const bam_attn* a, int* takes) {
    if (a == nullptr || takes == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_bwd_takes_ds: null pointer");
    *takes = a->plan != nullptr && a->D > 64 && a->Sk <= 131072 ? 1 : 0;
    if (*takes == 0 || !bam::one_launch_sizes(a->Sq, a->Sk, a->B, a->Hq)) return BAM_OK;
    bam_plan plan;
    bam::AttnParams all = {};
    BAM_TRY(attn_bwd_params(a, plan, all));
    all.ds_ws = nullptr;
    if (attn_bwd_one_launch(a, all, dkdv_parts(a))) *takes = 0;
    return BAM_OK;
}

int bam_attn_bwd(const bam_attn* a, void* stream) {
    if (a == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_bwd: null pointer");
    bam_plan plan;
    bam::AttnParams all = {};
    BAM_TRY(attn_bwd_params(a, plan, all));
    const int runs = a->head_runs > 1 ? a->head_runs : 1, hq = a->Hq / runs, hk = a->Hkv / runs, gsz = a->accumulate ? 4 : 2;
    // head dims up to 64: the dQ kernel runs first and computes delta on the way; above, dK/dV needs it first
    const bool dq_first = all.D <= 64;
    if (!dq_first) BAM_TRY(launched(bam::launch_bwd_preprocess(all, a->dtype, (hipStream_t)stream), "bam_attn_bwd (delta)"));
    const int parts = a->parts_workspace != nullptr ? dkdv_parts(a) : 1;
    const bool one_launch = attn_bwd_one_launch(a, all, parts);
    // launch_kv: what launches dK/dV, given its parameters; the parts are added up behind it
    auto with_parts = [&](const bam::AttnParams& p, auto launch_kv) -> int {
        if (parts == 1) return launched(launch_kv(p), "bam_attn_bwd (dk/dv)");
        const int64_t floats = dkdv_part_floats(a, parts);
        if (a->parts_bytes < 2 * 4 * floats || (reinterpret_cast<uintptr_t>(a->parts_workspace) & 15u))
            return fail(BAM_ERR_INVALID_ARGUMENT, "bam_attn_bwd: parts workspace of %lld bytes, %lld needed, 16-byte aligned",
                        (long long)a->parts_bytes, (long long)(2 * 4 * floats));
        bam::AttnParams part = p;
        const int64_t sh = a->D, ss = sh * p.Hkv * parts, sb = ss * p.Sk;
        float* ws = (float*)a->parts_workspace;
        part.dk = {ws, sb, ss, sh};
        part.dv = {ws + floats, sb, ss, sh};
        part.grad_typed = 2;
        part.kv_parts = parts;
        part.Hkv = p.Hkv * parts;
        BAM_TRY(launched(launch_kv(part), "bam_attn_bwd (dk/dv)"));
        return launched(bam::launch_sum_parts(p, ws, ws + floats, parts, a->dtype, (hipStream_t)stream), "bam_attn_bwd (sum)");
    };
    auto dkdv = [&](const bam::AttnParams& p) -> int {
        return with_parts(p, [&](const bam::AttnParams& kv) { return launch_dkdv(kv, a->dtype, stream); });
    };
    // The heads in runs of whole kv heads, every run through the same dS workspace: the launches of a stream run in
    // order, so a run's dQ kernel has read the workspace before the next run's dK/dV kernel writes it.
    for (int r = 0; r < runs; ++r) {
        bam::AttnParams p = all;
        auto skip = [&](bam::Tensor4& t, int heads, int bytes) { t.ptr = (const char*)t.ptr + (int64_t)r * heads * t.sh * bytes; };
        skip(p.q, hq, 2);
        skip(p.k, hk, 2);
        skip(p.v, hk, 2);
        skip(p.o, hq, 2);  // (up to head dim 64 the dQ kernel computes delta from it)
        skip(p.dout, hq, 2);
        skip(p.dq, hq, gsz);
        skip(p.dk, hk, gsz);
        skip(p.dv, hk, gsz);
        p.lse += (int64_t)r * hq * p.Sq_rounded;
        p.delta += (int64_t)r * hq * p.Sq_rounded;
        if (p.lse_scaled != nullptr) p.lse_scaled += (int64_t)r * hq * p.Sq_rounded;
        p.Hq = hq;
        p.Hkv = hk;
        if (a->plan != nullptr && runs > 1) BAM_TRY(fill_plan(p, "bam_attn_bwd", &plan, a->B, p.Sq, p.Sk));
        if (one_launch) {
            if (dq_first) BAM_TRY(launched(bam::launch_bwd_preprocess(p, a->dtype, (hipStream_t)stream), "bam_attn_bwd (delta)"));
            bam::AttnParams q = p;
            q.o.ptr = nullptr;  // (delta is there)
            BAM_TRY(with_parts(p, [&](const bam::AttnParams& kv) { return bam::launch_bwd_both(kv, q, a->dtype, (hipStream_t)stream); }));
            continue;
        }
        if (dq_first) {
            BAM_TRY(launched(launch_dq(p, a->dtype, stream), "bam_attn_bwd (dq)"));
            BAM_TRY(dkdv(p));
            continue;
        }
        BAM_TRY(dkdv(p));
        BAM_TRY(launched(launch_dq(p, a->dtype, stream), "bam_attn_bwd (dq)"));
    }
    return BAM_OK;
}

// ---- pinned host words the plan builders publish their pair counts to
int bam_host_words_alloc(uint64_t** words, int n) {
    if (words == nullptr || n <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_host_words_alloc: null pointer or no words");
    void* p = nullptr;
    const hipError_t e = hipHostMalloc(&p, (size_t)n * 8, hipHostMallocPortable | hipHostMallocCoherent);
    if (e != hipSuccess) return fail(BAM_ERR_LAUNCH, "bam_host_words_alloc: %s", hipGetErrorString(e));
    for (int i = 0; i < n; ++i) ((uint64_t*)p)[i] = 0;
    *words = (uint64_t*)p;
    return BAM_OK;
}
int bam_host_words_free(uint64_t* words) {
    const hipError_t e = words != nullptr ? hipHostFree(words) : hipSuccess;
    return e == hipSuccess ? BAM_OK : fail(BAM_ERR_LAUNCH, "bam_host_words_free: %s", hipGetErrorString(e));
}

// the D the kernels are compiled for
static int compiled_dim(int d) { return d <= 32 ? 32 : d <= 64 ? 64 : d <= 96 ? 96 : 128; }

int64_t bam_decode_workspace_bytes(int B, int Sk, int Hq, int Hkv, int D, int window) {
    if (B <= 0 || Sk <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || D <= 0 || D > 128 || window < 0) return 0;
    const bam::DecodeSplit s = bam::decode_split(B, Hq, Hkv, Sk, compiled_dim(D), window);
    return s.parts > 1 ? (int64_t)B * Hq * s.parts * (compiled_dim(D) + 2) * 4 : 0;
}

static int decode_impl(const void* q, const void* k, const void* v, void* o, int64_t q_stride_b, int64_t q_stride_h,
                       int64_t k_stride_b, int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
                       int64_t v_stride_h, int64_t o_stride_b, int64_t o_stride_h, int B, int Sk, int Hq, int Hkv, int D, float scale,
                       int dtype, int window, float softcap, void* workspace, int64_t workspace_bytes, uint32_t* counters,
                       int64_t n_counters, bool any_dim, void* stream) {
    BAM_TRY(check_problem(B, 1, Sk, Hq, Hkv, D, dtype, any_dim));
    BAM_TRY(check_half_tensor("k", k, k_stride_b, k_stride_s, k_stride_h));
    BAM_TRY(check_half_tensor("v", v, v_stride_b, v_stride_s, v_stride_h));
    if (q == nullptr || o == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: null pointer");
    if ((reinterpret_cast<uintptr_t>(q) & 1u) || (reinterpret_cast<uintptr_t>(o) & 1u))
        return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: q / o are not 2-byte aligned");
    if (!(scale > 0.f)) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: softmax scale must be > 0 (got %g)", scale);
    if (window < 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: window must be >= 0 (0 = none), got %d", window);
    if (!(softcap >= 0.f)) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: softcap must be >= 0 (0 = none), got %g", softcap);
    bam::DecodeParams p = {};
    p.D = compiled_dim(D);
    p.d = D;
    const bam::DecodeSplit s = bam::decode_split(B, Hq, Hkv, Sk, p.D, window);
    if ((int64_t)B * Hq > 0x7FFFFFFFll || s.units * s.parts > 0x7FFFFFFFll) return fail(BAM_ERR_UNSUPPORTED, "bam_decode: grid too large");
    if (s.parts > 1) {
        const int64_t need = bam_decode_workspace_bytes(B, Sk, Hq, Hkv, D, window);
        if (workspace == nullptr || workspace_bytes < need)
            return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: workspace of %lld bytes, %lld needed",
                        (long long)(workspace == nullptr ? 0 : workspace_bytes), (long long)need);
        if (reinterpret_cast<uintptr_t>(workspace) & 15u)
            return fail(BAM_ERR_INVALID_ARGUMENT, "bam_decode: workspace is not 16-byte aligned");
        p.ws_o = (float*)workspace;
        p.ws_ml = p.ws_o + (int64_t)B * Hq * s.parts * p.D;
        // The last part merges where that is a short step.  Not in a captured graph: its replays may overlap the caller's
        // eager calls, and the counters serve one call at a time.
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (counters != nullptr && s.units <= n_counters && s.parts <= 32 &&
            hipStreamIsCapturing((hipStream_t)stream, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone)
            p.counters = counters;
    }
    p.row_groups = s.row_groups;
    p.parts = s.parts;
    p.first = s.first;
    p.n_tiles = s.n_tiles;
    p.o_vec = ((reinterpret_cast<uintptr_t>(o) & 7u) == 0 && o_stride_b % 4 == 0 && o_stride_h % 4 == 0) ? 1 : 0;
    p.q = q;
    p.k = k;
    p.v = v;
    p.o = o;
    p.q_sb = q_stride_b;
    p.q_sh = q_stride_h;
    p.k_sb = k_stride_b;
    p.k_ss = k_stride_s;
    p.k_sh = k_stride_h;
    p.v_sb = v_stride_b;
    p.v_ss = v_stride_s;
    p.v_sh = v_stride_h;
    p.o_sb = o_stride_b;
    p.o_sh = o_stride_h;
    p.B = B;
    p.Sk = Sk;
    p.Hq = Hq;
    p.Hkv = Hkv;
    p.scale = scale;
    p.softcap = softcap;
    return launched(bam::launch_decode(p, s, dtype, (hipStream_t)stream), "bam_decode");
}

int bam_decode(const void* q, const void* k, const void* v, void* o, int64_t q_stride_b, int64_t q_stride_h,
               int64_t k_stride_b, int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
               int64_t v_stride_h, int64_t o_stride_b, int64_t o_stride_h, int B, int Sk, int Hq, int Hkv, int D, float scale,
               int dtype, int window, float softcap, void* workspace, int64_t workspace_bytes, void* stream) {
    return decode_impl(q, k, v, o, q_stride_b, q_stride_h, k_stride_b, k_stride_s, k_stride_h, v_stride_b, v_stride_s, v_stride_h,
                       o_stride_b, o_stride_h, B, Sk, Hq, Hkv, D, scale, dtype, window, softcap, workspace, workspace_bytes,
                       nullptr, 0, false, stream);
}

int bam_decode_counted(const void* q, const void* k, const void* v, void* o, int64_t q_stride_b, int64_t q_stride_h,
                       int64_t k_stride_b, int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
                       int64_t v_stride_h, int64_t o_stride_b, int64_t o_stride_h, int B, int Sk, int Hq, int Hkv, int D,
                       float scale, int dtype, int window, float softcap, void* workspace, int64_t workspace_bytes,
                       uint32_t* counters, int64_t n_counters, void* stream) {
    return decode_impl(q, k, v, o, q_stride_b, q_stride_h, k_stride_b, k_stride_s, k_stride_h, v_stride_b, v_stride_s, v_stride_h,
                       o_stride_b, o_stride_h, B, Sk, Hq, Hkv, D, scale, dtype, window, softcap, workspace, workspace_bytes,
                       counters, n_counters, true, stream);
}

int bam_mask_tile_flags(const uint8_t* mask, int8_t* flags, int64_t flags_stride_b, int64_t flags_stride_m, int B,
                        int Sq, int Sk, void* stream) {
    if (mask == nullptr || flags == nullptr) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_mask_tile_flags: null pointer");
    if (B <= 0 || Sq <= 0 || Sk <= 0) return fail(BAM_ERR_INVALID_ARGUMENT, "bam_mask_tile_flags: B, Sq and Sk must be positive");
    if (B > 65535 || (Sq + 127) / 128 > 65535)
        return fail(BAM_ERR_UNSUPPORTED, "bam_mask_tile_flags: grid too large (B = %d, Sq = %d)", B, Sq);
    return launched(bam::launch_mask_tile_flags(mask, flags, flags_stride_b, flags_stride_m, B, Sq, Sk, (hipStream_t)stream),
                    "bam_mask_tile_flags");
}

int bam_fwd_masked(const void* q, const void* k, const void* v, void* o, float* lse, const uint8_t* mask,
                   const int8_t* flags, int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h,
                   int64_t k_stride_b, int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b,
                   int64_t v_stride_s, int64_t v_stride_h, int64_t o_stride_b, int64_t o_stride_s,
                   int64_t o_stride_h, int64_t flags_stride_b, int64_t flags_stride_m, int B, int Sq, int Sk, int Hq,
                   int Hkv, int D, float scale, int dtype, const bam_bias* bias, const bam_plan* plan,
        void* stream) {
    BAM_TRY(check_mask("bam_fwd_masked", mask));
    const int64_t st[12] = BAM_FWD_STRIDES;
    return fwd_impl("bam_fwd_masked", q, k, v, o, lse, dense_source(mask, Sq, Sk), flags, st, flags_stride_b,
                    flags_stride_m, B, Hq, Hkv, D, scale, dtype, bias, plan, stream);
}

int bam_bwd_dkdv_masked(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                        const float* delta, void* dk, void* dv, const uint8_t* mask, const int8_t* flags,
                        int64_t q_stride_b, int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b,
                        int64_t k_stride_s, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s,
                        int64_t v_stride_h, int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h,
                        int64_t dk_stride_b, int64_t dk_stride_s, int64_t dk_stride_h, int64_t dv_stride_b,
                        int64_t dv_stride_s, int64_t dv_stride_h, int64_t flags_stride_b, int64_t flags_stride_m,
                        int B, int Sq, int Sk, int Hq, int Hkv, int D, float scale, int dtype, int accumulate,
                        const bam_bias* bias, const bam_plan* plan,
        void* stream) {
    BAM_TRY(check_mask("bam_bwd_dkdv_masked", mask));
    void* dq = nullptr;
    const int64_t dq_stride_b = 0, dq_stride_s = 0, dq_stride_h = 0;
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd_dkdv_masked", q, k, v, dout, lse, delta, dq, dk, dv, dense_source(mask, Sq, Sk), flags,
                       st, B, Hq, Hkv, D, scale, dtype, accumulate, false, true, bias, plan));
    return launched(launch_dkdv(p, dtype, stream), "bam_bwd_dkdv_masked");
}

int bam_bwd_dq_masked(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                      const float* delta, void* dq, const uint8_t* mask, const int8_t* flags, int64_t q_stride_b,
                      int64_t q_stride_s, int64_t q_stride_h, int64_t k_stride_b, int64_t k_stride_s,
                      int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_s, int64_t v_stride_h,
                      int64_t do_stride_b, int64_t do_stride_s, int64_t do_stride_h, int64_t dq_stride_b,
                      int64_t dq_stride_s, int64_t dq_stride_h, int64_t flags_stride_b, int64_t flags_stride_m, int B,
                      int Sq, int Sk, int Hq, int Hkv, int D, float scale, int dtype, int accumulate, const bam_bias* bias, const bam_plan* plan,
        void* stream) {
    BAM_TRY(check_mask("bam_bwd_dq_masked", mask));
    void *dk = nullptr, *dv = nullptr;
    const int64_t dk_stride_b = 0, dk_stride_s = 0, dk_stride_h = 0, dv_stride_b = 0, dv_stride_s = 0, dv_stride_h = 0;
    const int64_t st[23] = BAM_BWD_STRIDES;
    bam::AttnParams p = {};
    BAM_TRY(bwd_params(p, "bam_bwd_dq_masked", q, k, v, dout, lse, delta, dq, dk, dv, dense_source(mask, Sq, Sk), flags, st,
                       B, Hq, Hkv, D, scale, dtype, accumulate, true, false, bias, plan));
    return launched(launch_dq(p, dtype, stream), "bam_bwd_dq_masked");
}

}  // extern "C"
