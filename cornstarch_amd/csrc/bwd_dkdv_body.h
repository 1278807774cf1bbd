// The work of dK/dV workgroup `block`, for the parameters p and with the LDS arrays that the function around this text declares:
// bwd_dkdv_kernel, dkdv_work and (NARROW: four waves) bwd_dkdv_narrow_kernel (bwd_kernels.h).  As one function that they call it costs a
// launch of nothing but dK/dV 0.8 to 1 % above head dim 64 (8192 tokens, 32 / 8 heads, D 128: step 1727 -> 1741 us): the compiler
// spreads its registers another way.
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave & 3, st = wave >> 2;
    const int hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
    const int Sq = p.Sq, Sk = p.Sk;
    const int G = p.Hq / p.Hkv;

    const int unit = block;
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
    if constexpr (!NARROW) {
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
        for (int i = 0; i < (NARROW ? 0 : (128 * NCH) / DKDV_THREADS); ++i) {
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
    if constexpr (NARROW) {  // from memory, zeros past the head dim
        static_assert(KV_REGS && !DENSE && !SORTED && !SAVE && !LONG, "the forms it is compiled for");
        const char* kp = (const char*)p.k.ptr + 2 * ((int64_t)b * p.k.sb + (int64_t)key * p.k.ss + (int64_t)kv_head * p.k.sh);
        const char* vp = (const char*)p.v.ptr + 2 * ((int64_t)b * p.v.sb + (int64_t)key * p.v.ss + (int64_t)kv_head * p.v.sh);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const int c = 16 * kk + 8 * hi;
            u32x4 x = {0u, 0u, 0u, 0u}, y = {0u, 0u, 0u, 0u};
            if (kvalid && c < p.d) {
                x = *(const u32x4*)(kp + 2 * c);
                y = *(const u32x4*)(vp + 2 * c);
            }
            kfrag[kk] = x;
            vfrag[kk] = y;
        }
    }
    auto load_kv_operands = [&]() {  // after the V tile has been negated and a barrier has published it
        if (KV_REGS && !NARROW && !kv_loaded) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                kfrag[kk] = lds_read_chunk<D>(sK, 32 * kg + l32, 2 * kk + hi);
                vfrag[kk] = lds_read_chunk<D>(sV, 32 * kg + l32, 2 * kk + hi);
            }
            kv_loaded = true;
        }
    };

    typedef SliceStage<D, NARROW ? DKDV_NARROW_THREADS : DKDV_THREADS> Stage;
    constexpr int CPT = Stage::CPT;
    // copy instructions per wave and tile: Q, dO, one of the small rows and (IDX) the row positions
    constexpr int NLOADS = 2 * CPT + 1 + (IDX ? 1 : 0);
    static_assert(NLOADS <= 2 * KK * (NARROW ? 2 : 1), "one copy per MFMA of the S / dP phase");
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

    // Where this lane reads in tile 0, as byte addresses.  What a k-slice, a block of columns, a half of the tile and the other array add
    // are constants, XORed (the swizzle of chunk_slot takes bits 0 to 3 of the row; the tiles start at multiples of 256) or in the
    // instruction.  From chunk_slot access by access, a block of 32 x 32 took 133 vector instructions beside its MFMAs at head dim
    // 128, 99 now, and 256 registers, 234 now.  Step, us, D 128: 8192 tokens, 32 / 8 heads 1720 -> 1696, 65536 47.5 -> 46.7 ms, 4 x 1537
    // 364.5 -> 359, a bool mask, 2 x 4096, 16 heads 502 -> 494; 2 x 2003, 16 heads, D 96 169.2 -> 167.2.
    constexpr unsigned ROW_BYTES = NCH * 16, DO_AT = NB * TILE_BYTES, DELTA_AT = NB * DKDV_QT * 4;
    const int lane16 = lane & 15;
    const unsigned chunk_lane = ldsQ + 16u * (unsigned)chunk_slot<D>(l32, hi);
    const unsigned transposed_lane =
        ldsQ + 16u * (unsigned)chunk_slot<D>(4 * hi + (lane16 >> 2), 2 * half16 + ((lane16 & 3) >> 1)) + 8u * (lane16 & 1);
    const unsigned kv_lane = NARROW ? 0u : lds_addr(sK) + 16u * (unsigned)chunk_slot<D>(32 * kg + l32, hi);

    // One 64-row tile held in buffer cur against this wave's 32 keys; the wave's 32 rows sit at sequence
    // rows myrow0.. and its class for them is cls.  The copies of the next tile into the other buffer
    // are issued one per MFMA of the S / dP phase, or back to back when this wave has nothing to compute.
    // The wave's flag class is extracted with a per-lane copy of the key group number on purpose: a branch
    // condition the compiler can prove wave-uniform makes it restructure the loop around that branch, and the
    // result needs far more registers than a wave has.
    const int kg_lane = (tid >> 6) & 3;
    // SAVE: where this lane's two chunks sit inside a 2 KiB block (key l32, rows 4 hi + {0..3, 8..11}, then those 16 further on, 1 KiB behind and
    // four keys across): either store of the wave fills 1 KiB in one piece.  With a key's 64 bytes side by side each store filled every
    // other 16 bytes: dK/dV alone, us, a causal mask, 8192 tokens, 32 / 8 heads, D 128 1149 -> 1137 (without any store 1012: what is left is the
    // power that the writes take).  The keys change places in fours so that dQ's transposing reads spread over the LDS banks.
    const unsigned ds_first = (unsigned)(kg * 2048 + hi * 512 + (l32 ^ (8 * hi)) * 16), ds_second = (ds_first ^ 64u) + 1024u;
    // SAVE: the pairs (slice, this key tile) that have work are numbered consecutively from ds_base, by ascending slice,
    // i.e. in the order of the slice list: pair number = ds_base + position in the list
    int ds_base = 0;
    if (SAVE) ds_base = __builtin_amdgcn_readfirstlane(p.ds_tile_base[(int64_t)b * p.num_kt + nt]);
    // BIAS, per-key form (row stride 0): this lane's bias value for the head in work
    float bias_key = 0.f;
    int bias_head = -1;
    auto fetch_bias_key = [&](int h) {
        if (BIAS && (KEY_BIAS || p.bias_sm == 0) && h != bias_head) {
            bias_head = h;
            bias_key = kvalid ? load_bias1<T>(p.bias, (int64_t)b * p.bias_sb + (int64_t)h * p.bias_sh + key, p.bias_f32 != 0) : 0.f;
            asm volatile("" : "+v"(bias_key));  // arrives here, not at its first use between the tile copies
        }
    };
    // BESIDE: the chain of S ends before that of dP begins, so that the exponentials are taken beside the MFMAs of dP, and the gradients of 16 rows
    // beside the dV and dK products of the 16 before (a wave overlaps its own vector work with its own MFMAs).  It gives where a unit's eight
    // waves do not fill each other's gaps all the time: step, us, D 128, both chains side by side -> one after the other: 4 x 1537 tokens, 32 / 8
    // heads 312.3 -> 309.4, 2048, 8 heads 101.3 -> 100.5, 8192, 32 / 8 1580 -> 1576, 65536 41.99 -> 41.89 ms, D 96 2 x 2003 166.6 -> 166.1 (the products alone
    // half of it, the chains alone -1.5 %).  Head dim 64 2 x 4096, 16 heads, a bias 375.8 -> 377.1, with four waves 1016 -> 1063 (168 registers are too few);
    // a bool mask 461.5 -> 461.6, with spills.
    constexpr bool KEY_ROW = BIAS && KEY_BIAS, BESIDE = D > 64 && !DENSE && (!BIAS || KEY_BIAS);

    // ds_pos: position of the wave's slice in the slice list.
    // returns true when the wave has issued its two dS stores (they may stay in flight over the end of the iteration)
    // pos_cur, pos_nxt: the buffers of the tile's positions and of those that are copied now
    // qr: this wave's rows inside the 64-row tile.  NARROW: the caller issues the copies; what derives from the lane is derived anew for
    // every block (`own`), it would take the registers of the K and V operands otherwise
    auto tile_step = [&](const int qr, int cur, int cls, int h_cur, int myrow0, int ds_pos, const TileSource& next, int nxt, int pos_cur,
                         int pos_nxt) __attribute__((always_inline)) -> bool {
        if (cls == 0) {
#pragma unroll
            for (int j = 0; j < (NARROW ? 0 : NLOADS); ++j) issue_copy(j, next, nxt, pos_nxt);
            return false;
        }
        const int ds_e = ds_base + ds_pos;
        int own = lane;
        if (NARROW) asm volatile("" : "+v"(own));
        const int lane = own, hi = lane >> 5, l32 = lane & 31, half16 = (lane >> 4) & 1;
        // ---- S = Q K^T and dP = dO V^T : 32 queries x 32 keys, two accumulator chains; both operands of
        // every MFMA come from LDS and are requested AHEAD MFMAs in front of their use
        // The V tile in LDS is NEGATED (see negate_v_tile), and the dP accumulator starts from delta instead of
        // zero: the chain then delivers delta - dO V^T = -(dP - delta) with no subtraction left for the VALU.
        // The sign is carried through dS into dK and taken back by the epilogue.
        f32x16 s, dp;
        const unsigned tile_at = (unsigned)(cur * TILE_BYTES + qr * ROW_BYTES);
        const unsigned row_at = 16u * hi + (lds_addr(sLse) + (unsigned)(cur * (DKDV_QT * 4) + qr * 4));
        {
            constexpr int NOP = 2 * KK, AHEAD = D > 64 ? 2 : 3;
            constexpr int FIRST = SORTED ? (NOP - NLOADS < 4 ? NOP - NLOADS : 4) : 0;  // the copies start behind MFMA FIRST - 1
            constexpr unsigned V_AT = 128 * ROW_BYTES;
            const unsigned at = chunk_lane + tile_at;
            u32x4 a[NOP], bb[NOP];
            auto is_dp = [](int j) { return BESIDE ? j >= KK : (j & 1) != 0; };
            auto slice = [](int j) { return BESIDE ? j % KK : j >> 1; };
            auto operand = [&](int j) { return lds_read16<u32x4>((at ^ (unsigned)(32 * slice(j))) + (is_dp(j) ? DO_AT : 0u)); };
            auto kv = [&](int j) {
                if constexpr (KV_REGS)
                    return is_dp(j) ? vfrag[slice(j)] : kfrag[slice(j)];
                else
                    return lds_read16<u32x4>((kv_lane ^ (unsigned)(32 * slice(j))) + (is_dp(j) ? V_AT : 0u));
            };
            auto read_delta = [&]() {
#pragma unroll
                for (int grp = 0; grp < 4; ++grp) {
                    const f32x4 d4 = lds_read16<f32x4>(row_at + DELTA_AT + 32u * grp);
#pragma unroll
                    for (int x = 0; x < 4; ++x) dp[4 * grp + x] = d4[x];
                }
            };
            static_assert(!BESIDE || (KK >= 4 && !SCALED), "the rows' lse is asked for by the first four MFMAs of dP");
            f32x4 l4[4];
            auto probability = [&](int i) {
                s[i] = __builtin_amdgcn_exp2f(fmaf(KEY_ROW ? fmaf(s[i], p.scale, bias_key) : s[i], c2, l4[i >> 2][i & 3] * -LOG2E));
            };
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                a[j] = operand(j);
                bb[j] = kv(j);
                if (!BESIDE && j == 0) read_delta();
            }
            // beside MFMA m of dP, from the second one on (S is there by then), and behind the last
            auto probabilities = [&](int m) {
#pragma unroll
                for (int i = 16 * (m - 1) / KK; i < 16 * m / KK; ++i) probability(i);
            };
#pragma unroll
            for (int j = 0; j < NOP; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                if (j + AHEAD < NOP) {
                    a[j + AHEAD] = operand(j + AHEAD);
                    bb[j + AHEAD] = kv(j + AHEAD);
                }
                if (BESIDE && j == KK - 2) read_delta();
                if (is_dp(j))
                    dp = T::mfma(a[j], bb[j], dp);
                else
                    s = T::mfma(a[j], bb[j], slice(j) == 0 ? zero16 : s);
                if (BESIDE && j >= KK) {
                    if (j - KK < 4) l4[(j - KK) & 3] = lds_read16<f32x4>(row_at + 32u * (j - KK));
                    if (j > KK) probabilities(j - KK);
                }
                if (!NARROW && j >= FIRST && j - FIRST < NLOADS) issue_copy(j - FIRST, next, nxt, pos_nxt);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (BESIDE) probabilities(KK);
        }
        // ---- P = exp(scale s - lse) on allowed pairs, -dS/scale = P (delta - dP)   (the factor `-scale` of dS
        // is applied once to dK in the epilogue).  C fragment: register i <-> query row
        // 8*(i/4) + 4*hi + i%4 of this wave's 32 rows.
        if (BESIDE) {
            // (taken above)
        } else if (BIAS && (KEY_BIAS || p.bias_sm == 0)) {
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
        if (!BESIDE) {
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                const f32x4 l4 = lds_read16<f32x4>(row_at + 32u * grp);
#pragma unroll
                for (int x = 0; x < 4; ++x) s[4 * grp + x] = __builtin_amdgcn_exp2f(fmaf(s[4 * grp + x], c2, SCALED ? -l4[x] : l4[x] * -LOG2E));
            }
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
                if constexpr (NARROW) {  // (row by row: 20 registers less)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        __builtin_amdgcn_sched_barrier(0);
                        const int r = 8 * (i >> 2) + 4 * hi + (i & 3);
                        QueryBits qb;
                        qb.a_lo = sWq[wave][0][r];
                        qb.a_hi = sWq[wave][1][r];
                        qb.x_lo = sWq[wave][2][r];
                        qb.x_hi = sWq[wave][3][r];
                        qb.lim = (int)sWq[wave][4][r];
                        qb.text = (unsigned)qb.lim < 0x7FFFFFFFu;
                        s[i] = allow_pair(qb, klo, khi, kpos) ? s[i] : 0.f;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                } else
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
        u32x4 pb[2], dsb[2];
        // ---- dV^T += dO^T P ; dK^T += Q^T dS -------------------------------------------------
        if constexpr (BESIDE) {
            const unsigned at = transposed_lane + tile_at;
            // MFMA j: 16 rows (j / 2 DB), dV then dK, block of columns j % DB
            constexpr int N2 = 4 * DB, AHEAD2 = 2;
            u32x4 tr[N2];
            auto operand = [&](int j) {
                const int t = j / (2 * DB), db = j % DB;
                const unsigned x = (at ^ (64u * db)) + 16u * t * ROW_BYTES, y = (at ^ (64u * db + 16u)) + (16u * t + 8u) * ROW_BYTES;
                const unsigned from = (j / DB) & 1 ? 0u : DO_AT;
                return lds_read_transposed_at(x + from, y + from);
            };
#pragma unroll
            for (int j = 0; j < AHEAD2; ++j) tr[j] = operand(j);
            pb[0] = pack8<T>(s, 0);
            // beside the MFMAs: step i = 0..3 of the gradients of 16 rows
            auto grad = [&](int t, int w) {
                const int i = 8 * t + 2 * w;
                dp[i] *= s[i];  // -dS / scale
                dp[i + 1] *= s[i + 1];
                dsb[t][w] = T::pack2(dp[i], dp[i + 1]);
                if (t == 0) pb[1][w] = T::pack2(s[8 + 2 * w], s[9 + 2 * w]);
            };
#pragma unroll
            for (int j = 0; j < N2; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                if (j + AHEAD2 < N2) tr[j + AHEAD2] = operand(j + AHEAD2);
                const int t = j / (2 * DB), db = j % DB;
                if ((j / DB) & 1)
                    dk[db] = T::mfma(tr[j], dsb[t], dk[db]);
                else
                    dv[db] = T::mfma(tr[j], pb[t], dv[db]);
                if (j < 2 * DB)
#pragma unroll
                    for (int w = 4 * (j % DB) / DB; w < 4 * (j % DB + 1) / DB; ++w) grad(j / DB, w);
            }
            __builtin_amdgcn_sched_barrier(0);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) dp[i] = s[i] * dp[i];  // -dS / scale
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                pb[t] = pack8<T>(s, 8 * t);
                dsb[t] = pack8<T>(dp, 8 * t);
            }
            const unsigned at = transposed_lane + tile_at;
            u32x4 tg[2][DB], tq[2][DB];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    const unsigned x = (at ^ (64u * db)) + 16u * t * ROW_BYTES, y = (at ^ (64u * db + 16u)) + (16u * t + 8u) * ROW_BYTES;
                    tg[t][db] = lds_read_transposed_at(x + DO_AT, y + DO_AT);
                    tq[t][db] = lds_read_transposed_at(x, y);
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
            // (also where the last-level cache could hold them: without the hint there, D 96, 2 x 2003 tokens, 16 heads, inputs that change from
            // step to step 158.7 -> 166.4 us)
            const unsigned rec_no = (unsigned)__builtin_amdgcn_readfirstlane(h_cur * (int)p.ds_capacity + ds_e);
            const char* rec = (const char*)p.ds_ws + ((uint64_t)rec_no << 13);
            asm volatile("global_store_dwordx4 %0, %2, %4 nt\n\tglobal_store_dwordx4 %1, %3, %4 nt"
                         :
                         : "v"(ds_first), "v"(ds_second), "v"(dsb[0]), "v"(dsb[1]), "s"(rec)
                         : "memory");
        }
        return SAVE;
    };

    // Sequences of more than MAX_SLICE_LIST slices are walked in several passes, from the end, each with a list
    // of its own; dK and dV live in registers and simply carry over.
    for (int s_end = ns_total;;) {
        lds_barrier();
        const int n = NARROW ? __builtin_amdgcn_readfirstlane(sCount) : sCount;
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
            if constexpr (NARROW) {
                if (!v_negated) {
                    arrived(kfrag);
                    arrived(vfrag);
#pragma unroll
                    for (int kk = 0; kk < (KV_REGS ? KK : 1); ++kk)
#pragma unroll
                        for (int e = 0; e < 4; ++e) vfrag[kk][e] ^= 0x80008000u;
                    v_negated = true;
                }
            } else if (!v_negated) {  // K, V and the first tile have landed
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
                int x_lo = entry_lo(r_req), x_hi = entry_hi(r_req);
                TileSource next;
                const int p1 = SORTED ? (pos_cur == 2 ? 0 : pos_cur + 1) : nxt, p2 = SORTED ? (pos_cur == 0 ? 2 : pos_cur - 1) : nxt;
                if constexpr (SORTED) {
                    next = gathered_source(hv_nxt, sQpos[p1], (n_lo >> 8) * 32, (n_hi >> 8) * 32, (a_lo >> 8) * 32, (a_hi >> 8) * 32);
                } else {
                    next = tile_source(hv_nxt, (n_lo >> 8) * 32, (n_hi >> 8) * 32);
                }
                const int mine = st ? e_hi : e_lo;
                fetch_bias_key(hk * G + g_cur);
                if constexpr (NARROW) {  // both slices, one after the other
#pragma unroll
                    for (int j = 0; j < NLOADS; ++j) issue_copy(j, next, nxt, nxt);
                    x_lo = __builtin_amdgcn_readfirstlane(x_lo);
                    x_hi = __builtin_amdgcn_readfirstlane(x_hi);
#pragma unroll (D > 32 ? 1 : 2)
                    for (int half = 0; half < 2; ++half) {
                        const int e = half ? e_hi : e_lo;
                        tile_step(32 * half, cur, (e >> (2 * kg_lane)) & 3, hk * G + g_cur, (e >> 8) * 32, 0, next, nxt, cur, nxt);
                    }
                }
                const bool stored = !NARROW && tile_step(32 * st, cur, (mine >> (2 * kg_lane)) & 3, hk * G + g_cur, (mine >> 8) * 32, n - 2 - 2 * r_cur + st,
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
                if constexpr (NARROW) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[4 * grp + i] *= factor;
                    continue;
                }
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
    if constexpr (NARROW) {
        if (!kvalid) return;
        finish(dk, 0, -p.scale, p.dk);
        finish(dv, 1, 1.f, p.dv);
        return;
    }
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
