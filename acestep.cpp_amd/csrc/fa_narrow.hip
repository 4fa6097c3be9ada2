// fa_narrow.hip -- MFMA flash attention with 16 queries per wave (gfx950).
//
// Serves the prefill calls that do not fill the chip with 128-query
// workgroups (fa_mfma.hip): the encoders (src/qwen3-enc.h:195-199), the DiT
// on short songs (src/dit-graph.h:227-231, :348-352), the next piece of a
// prompt (src/qwen3-lm.h:465-469).  One workgroup = 4 waves = 64 consecutive
// queries of one (batch, q head); each wave owns 16.  Keys come in the same
// 64-key K/V tiles (DMA into LDS, XOR-swizzled rows, class-0 tiles skipped).
//
//   S^T[16 keys x 16 q] = K . Q^T     v_mfma_f32_16x16x32
//   O^T[16 dims x 16 q] += V^T . P^T  same MFMA, 32 keys per step
//
// What bounds such a call is the chain of one workgroup's tiles, not the
// chip: with one workgroup per CU a tile of fa_mfma.hip takes ~2300 cycles
// (1024 of them matrix work) and one of this kernel ~1700 for half the
// queries, on twice as many CUs.  The copies of a tile (32 KB through the
// CU's 64 B/clk load path: at least 512 cycles) run NST - 1 tiles ahead in a
// ring of NST stages: four (132 KB, one workgroup per CU) where the grid has
// at most one workgroup per CU, two (66 KB, two per CU) otherwise.  Kernel
// times against the 128- and 192-query kernels: 437 tokens x 16 heads under a
// window 12.4 against 16.3 us, without a mask 11.6 against 19.7 us.  (Few jobs
// over many key tiles take fa_mfma.hip's key split: 333 tokens x 32 heads over
// 2133 keys 30.8 us there, 38.3 here, 41.0 with neither.)
//
// Measured and dropped: two waves per query group, each with 32 queries and
// half of a tile's keys, (m, l, O) merged at the end: half the LDS reads per
// product, but 113 against 99 us on eight encoder layers, since the softmax
// of one block then hides under too few products.
//
// Lane l = 16 g + n holds query n and keys 4g..4g+3 of each 16-key block
// (the layout of fa_wide.hip), so a query's scores are spread over lanes n,
// n+16, n+32, n+48; the reference max is equal across them, and the row
// maximum over the four lanes is taken only when some lane's own maximum
// exceeds the reference by more than 8 (exp2 domain).

#include "fa_prefill.h"
#include "once_per_device.h"

namespace mxfa {

enum : int { kNarrowNone = 0, kNarrowDense = 1, kNarrowUnal = 2, kNarrowSm = 3 };   // mask modes (Unal: odd rows)

constexpr int kNarrowStage = kStageBytes + 1024;   // K, V, then 256 B per wave: its rows' liveness words (128 B used)
template <int NST> constexpr int narrow_lds() { return NST * kNarrowStage; }

// T: K/V type; CAP: logit softcap.
template <int T, int MODE, bool CAP, int NST>
__device__ __forceinline__ void fa_narrow_body(const FaArgs &a) {
    constexpr bool SM = MODE == kNarrowSm, DENSE = MODE == kNarrowDense || MODE == kNarrowUnal;
    constexpr bool kLo = T == T_BF16 || MODE == kNarrowUnal;   // P as a hi/lo pair (fa_mfma.hip)
    constexpr float kUp = kLo ? pair_up<T>() : 0.0f;
    constexpr int kPer = 8 + (DENSE ? 1 : 0);   // copies per stage
    using MF = Mfma16<T>;
    using V8 = typename MF::v8;
    static_assert(kD == 128, "kernel is written for D = 128");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    warm_args();
    const int tid = (int)__builtin_amdgcn_workitem_id_x();
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, g = lane >> 4;
    int qt, head, kvh, b;
    bool second = false;   // (no staggered start: measured level)
    pf_job(a, a.n_qt_n, qt, head, kvh, b, second);
    const int bk = div_fast(b, a.fd_rk3);
    const int q0w = qt * kPfNarrowBM + wave * 16;
    const int qrow = min(q0w + n16, a.Sq - 1);   // rows past Sq: the last row (not stored)

    const int plane = a.mask ? mod_fast(b, a.fd_m3, a.m_ne3) * a.m_ne2 + mod_fast(head, a.fd_m2, a.m_ne2) : 0;
    TileClasses tc{0u, 0u, DENSE};
    if constexpr (DENSE) {
        const uint32_t *row = (const uint32_t *)(a.tile_class64 + ((int64_t)plane * 2 * a.n_qt + qt) * a.n_kt_pad);
        if (4 * lane < a.n_kt) tc.w0 = row[lane];
        if (256 + 4 * lane < a.n_kt) tc.w1 = row[64 + lane];
    }
    // structured mask: as fa_mfma.hip, over the job's 64 rows
    int sm_kt_first = 0, sm_kt_end = 0, sm_in_lo = 0, sm_in_hi = 0, row_lo = 0, row_hi = 0;
    int sm_lo = 0, sm_hi = 0, sm_kt_lo = -1, sm_kt_hi = -1;   // the keys the rows see together, their ragged end tiles
    if constexpr (SM) {
        const int q_first = qt * kPfNarrowBM, q_last = min(q_first + kPfNarrowBM, a.Sq) - 1;
        int lo_f, hi_f, lo_l, hi_l;
        sm_row_range(a, b, q_first, lo_f, hi_f);
        sm_row_range(a, b, q_last, lo_l, hi_l);
        sm_kt_first = __builtin_amdgcn_readfirstlane(max(lo_f, 0) / kPfBN);
        sm_kt_end = __builtin_amdgcn_readfirstlane(lo_f < hi_l ? (hi_l + kPfBN - 1) / kPfBN : 0);
        sm_lo = __builtin_amdgcn_readfirstlane(lo_f);
        sm_hi = __builtin_amdgcn_readfirstlane(hi_l);
        if (sm_lo % kPfBN) sm_kt_lo = sm_kt_first;
        if (sm_hi % kPfBN) sm_kt_hi = sm_kt_end - 1;
        sm_in_lo = __builtin_amdgcn_readfirstlane(lo_l);
        sm_in_hi = __builtin_amdgcn_readfirstlane(hi_f);
        sm_row_range(a, b, qrow, row_lo, row_hi);
    }
    const int n_kt = a.n_kt;
    auto next_live = [&](int kt) __attribute__((always_inline)) -> int {
        if constexpr (SM) {
            const int k = max(kt, sm_kt_first);
            return k < sm_kt_end ? k : n_kt;
        } else {
            return tc.next_live(min(kt, n_kt), n_kt);
        }
    };
    auto class_of = [&](int kt) __attribute__((always_inline)) -> int {
        if constexpr (SM)
            return (kt * kPfBN >= sm_in_lo && kt * kPfBN + kPfBN <= sm_in_hi) ? 1
                   : kt == sm_kt_lo || kt == sm_kt_hi ? 2 | kTileDeadKeys : 2;
        else return tc.at(kt);
    };
    const char *mplane = DENSE ? a.mask + (int64_t)(mod_fast(head, a.fd_m2, a.m_ne2)) * a.m_nb2 + (int64_t)mod_fast(b, a.fd_m3, a.m_ne3) * a.m_nb3 : a.q;
    const __amdgpu_buffer_rsrc_t mrs =
        __builtin_amdgcn_make_buffer_rsrc((void *)mplane, (short)0, DENSE ? (int)a.m_plane_bytes : 0, 0x00020000);
    const uint32_t mrow_off = (uint32_t)qrow * (uint32_t)a.m_nb1 + 8u * (uint32_t)g;
    const float slope_l2 = DENSE ? alibi_slope(a, head) * kLog2e : 0.0f;
    const float sl2 = a.scale * kLog2e;
    const float sc_in = a.softcap_in;
    const bool lean_ok = !CAP && sl2 > 0.0f;   // the lean path takes max over raw scores

    // K and V rows of this (batch, kv head): copies as in fa_wide.hip
    const char *kbase = a.k + (int64_t)kvh * a.k_nb2 + (int64_t)bk * a.k_nb3;
    const char *vbase = a.v + (int64_t)kvh * a.v_nb2 + (int64_t)bk * a.v_nb3;
    const uint64_t k_avail = (uint64_t)(a.Skv - 1) * (uint64_t)a.k_nb1 + 2 * kD;
    const uint64_t v_avail = (uint64_t)(a.Skv - 1) * (uint64_t)a.v_nb1 + 2 * kD;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void *)smem);
    const uint32_t k_row = (uint32_t)a.k_nb1, v_row = (uint32_t)a.v_nb1;
    const int dkey = lane >> 4, dslot = lane & 15;
    uint32_t vk[4], vv[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        vk[c] = (uint32_t)(4 * c + dkey) * k_row + 16u * (uint32_t)(dslot ^ swz_k(4 * c + dkey));
        vv[c] = (uint32_t)(4 * c + dkey) * v_row + 16u * (uint32_t)(dslot ^ swz_v(4 * c + dkey));
    }
    // this wave's liveness words of a tile: 16 rows x 8 bytes, 4 bytes per
    // lane of the first 32 lanes (the others read past the resource: zeros)
    const char *bbase = nullptr;
    if constexpr (DENSE)
        if (a.tile_bits)
            bbase = (const char *)(a.tile_bits + ((int64_t)plane * a.n_qt + qt / 2) * a.n_kt * kPfBM +
                                   (qt & 1) * kPfNarrowBM + wave * 16);
    const i32x4 rk = buf_rsrc(kbase, (uint32_t)min(k_avail, (uint64_t)0xFFFFFFFFu));
    const i32x4 rv = buf_rsrc(vbase, (uint32_t)min(v_avail, (uint64_t)0xFFFFFFFFu));
    const i32x4 rb = buf_rsrc(bbase ? bbase : a.q, bbase ? (uint32_t)(a.n_kt - 1) * kPfBM * 8 + 128u : 0u);
    const uint32_t vb = lane < 32 ? 4u * (uint32_t)lane : 0x80000000u;   // (past the resource: zeros)
    // copy i of tile kt's eight into stage st (K rows for even i, V rows for
    // odd); `words`: the tile's liveness words of this wave
    auto copy = [&](int kt, int st, int i) __attribute__((always_inline)) {
        const uint32_t l0 = lds0 + (uint32_t)st * kNarrowStage + (uint32_t)(16 * wave) * 256u;
        const uint32_t row = (uint32_t)(kt * kPfBN + 16 * wave);
        if (i & 1) dma16_buf(rv, vv[i >> 1] + row * v_row, l0 + kTileBytes + 4 * (i >> 1) * 256);
        else dma16_buf(rk, vk[i >> 1] + row * k_row, l0 + 4 * (i >> 1) * 256);
    };
    auto words = [&](int kt, int st) __attribute__((always_inline)) {
        if constexpr (DENSE)
            dma4_buf(rb, vb + (uint32_t)kt * (kPfBM * 8),
                     lds0 + (uint32_t)st * kNarrowStage + kStageBytes + (uint32_t)wave * 256u);
    };

    // Ring of live tiles: kq[0] is computed next, kq[0 .. NST-2] are in
    // flight or landed (n_kt: none).
    int kq[NST];
    kq[0] = next_live(0);
#pragma unroll
    for (int i = 0; i < NST - 1; i++) {
        if (kq[i] < n_kt) {
            words(kq[i], i);
#pragma unroll
            for (int j = 0; j < 8; j++) copy(kq[i], i, j);
        }
        kq[i + 1] = next_live(kq[i] + 1);
    }

    // Q^T operands: qv[t] = Q[query n][32t + 8g .. +7], F32 rounded to T, or
    // already in T (a.q16)
    V8 qv[4];
    {
        const char *qh = a.q + (int64_t)head * a.q_nb2 + (int64_t)b * a.q_nb3 + (int64_t)qrow * a.q_nb1;
        if (a.q16) {
#pragma unroll
            for (int t = 0; t < 4; t++) qv[t] = __builtin_bit_cast(V8, *(const u16x8 *)(qh + 2 * (32 * t + 8 * g)));
        } else {
            f32x4 x[4][2];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                x[t][0] = *(const f32x4 *)(qh + 4 * (32 * t + 8 * g));
                x[t][1] = *(const f32x4 *)(qh + 4 * (32 * t + 8 * g) + 16);
            }
#pragma unroll
            for (int t = 0; t < 4; t++) qv[t] = __builtin_bit_cast(V8, cvt8<T>(x[t][0], x[t][1]));
        }
    }

    WaveKeys wk;   // (lands with Q)
    if constexpr (DENSE) wk.init(a, plane, qt, 1, wave, lane);

    // (Q is waited for here: the wait the compiler would otherwise put at the
    // operands' first use, inside the tile loop, drains the copies in flight)
#pragma unroll
    for (int t = 0; t < 4; t++) asm volatile("" : "+v"(qv[t]));

    // LDS operand addresses (fa_wide.hip): K operand (key block kb, dim step
    // t) at kb0 ^ 64t of block kb, V^T operand (half p, dim block db) at
    // vb0 ^ 32db of half p
    const int vrow = 4 * g + (n16 >> 2);
    const uint32_t kb0 = n16 * 256 + 16 * (g ^ n16);
    const uint32_t vb0 = vrow * 256 + 8 * (n16 & 1) + 16 * ((n16 & 3) >> 1) + 16 * swz_v(vrow);

    f32x4 o[8];
#pragma unroll
    for (int db = 0; db < 8; db++) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m2 = -INFINITY, lsum = 0.0f;

    // General tiles (mask, tail, softcap, non-positive scale): a half's
    // scores become x = scale*s (+softcap) + slope*mask in the exp2 domain,
    // -inf for masked keys and keys past Skv (lane: key 16kb + 4g + i).
    auto general_x = [&](f32x4 (&s)[2], int key0, int cl, uint32_t bits) __attribute__((always_inline)) {
        auto val = [&](float sc, float mv) __attribute__((always_inline)) -> float {
            if constexpr (CAP) return (a.softcap * fast_tanh(sc * sc_in)) * kLog2e + mv;
            else return fmaf(sc, sl2, mv);
        };
        if constexpr (SM) {
            const int lo_rel = row_lo - key0 - 4 * g, hi_rel = row_hi - key0 - 4 * g;
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int off = 16 * kb + i;
                    const float x = val(s[kb][i], 0.0f);
                    s[kb][i] = (off >= lo_rel && off < hi_rel) ? x : -INFINITY;
                }
            return;
        }
        const int kmax = a.Skv - key0 - 4 * g;
        if (DENSE && cl == 3) {   // 0 / -inf: the row's liveness word (0 past Skv)
            const uint32_t w = bits >> (4 * g);
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x = val(s[kb][i], 0.0f);
                    s[kb][i] = ((w >> (16 * kb + i)) & 1u) ? x : -INFINITY;
                }
            return;
        }
        u16x4 mw[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        if (DENSE && cl == 2) {
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
                const uint32_t off = mrow_off + 2u * (uint32_t)(key0 + 16 * kb);
                if constexpr (MODE == kNarrowUnal) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        mw[kb][i] = __builtin_amdgcn_raw_buffer_load_b16(mrs, off + 2u * i, 0, 0);
                } else {
                    mw[kb] = __builtin_bit_cast(u16x4, __builtin_amdgcn_raw_buffer_load_b64(mrs, off, 0, 0));
                }
            }
        }
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float mv = h2f_bits(mw[kb][i]) * slope_l2;
                const float x = val(s[kb][i], mv);
                s[kb][i] = (mv == -INFINITY || 16 * kb + i >= kmax) ? -INFINITY : x;
            }
    };
    // probabilities of key block kb of a half into the P^T operand
    auto probs = [&](const f32x4 (&s)[2], int kb, float gs, float mneg, u16x8 &pw, u16x8 &pl)
                     __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            const float p0 = fast_exp2(fmaf(s[kb][i], gs, mneg));
            const float p1 = fast_exp2(fmaf(s[kb][i + 1], gs, mneg));
            u16x2 h, l;
            if constexpr (kLo) {
                p_pair<T>(p0, p1, h, l);
                pl[4 * kb + i] = l[0];
                pl[4 * kb + i + 1] = l[1];
            } else {
                h = u16x2{MF::from_f32(p0), MF::from_f32(p1)};
            }
            pw[4 * kb + i] = h[0];
            pw[4 * kb + i + 1] = h[1];
        }
    };
    auto psum = [&](const u16x8 &pw, const u16x8 &pl) __attribute__((always_inline)) -> float {
        float l = sum8<T>(pw, 0.0f);
        if constexpr (kLo) l = sum8<T>(pl, l);
        return l;
    };
    auto max8 = [&](const f32x4 (&s)[2]) __attribute__((always_inline)) {
        return fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    };

    // One 64-key tile as two 32-key halves (the phases of fa_wide.hip); the
    // copies of tile kn (kn < n_kt) into stage sn go out one per two steps
    // of R1 and R2.
    constexpr int kLook = 6, kRing = 8;
    auto tile = [&](int kt, int cls, int st, int kn, int sn) __attribute__((always_inline)) {
        const bool do_issue = kn < n_kt;   // uniform
        if (do_issue) words(kn, sn);
        const int cl = cls & 3;
        const int key0 = kt * kPfBN;
        const bool general =
            __builtin_amdgcn_readfirstlane((int)(cl >= 2 || key0 + kPfBN > a.Skv || !lean_ok)) != 0;
        const float gs = general ? 1.0f : sl2;   // wave-uniform
        const uint8_t *sp = smem + st * kNarrowStage;
        uint64_t bits = 0;
        if (DENSE && cl == 3) bits = *(const uint64_t *)(sp + kStageBytes + wave * 256 + n16 * 8);
        u16x8 op[kRing];
        auto kread = [&](int kb, int t) __attribute__((always_inline)) -> u16x8 {
            return *(const u16x8 *)(sp + kb * 16 * 256 + (kb0 ^ (64u * (uint32_t)t)));
        };
        auto vread = [&](int p, int db) __attribute__((always_inline)) -> u16x8 {
            const uint8_t *q = sp + kTileBytes + p * 32 * 256 + (vb0 ^ (32u * (uint32_t)db));
            const u16x4 p0 = lds_read_tr16(q);
            const u16x4 p1 = lds_read_tr16(q + 16 * 256);
            return u16x8{p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
        };
        auto fetch = [&](int n) __attribute__((always_inline)) {
            if (n < 8) op[n % kRing] = kread(n & 1, n >> 1);
            else if (n < 16) op[n % kRing] = kread(2 + (n & 1), (n - 8) >> 1);
            else if (n < 24) op[n % kRing] = vread(0, n - 16);
            else if (n < 32) op[n % kRing] = vread(1, n - 24);
        };
        auto qk = [&](f32x4 (&s)[2], int n) __attribute__((always_inline)) {
            const int t = (n & 7) >> 1, kb = n & 1;
            s[kb] = MF::run(__builtin_bit_cast(V8, op[n % kRing]), qv[t], t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[kb]);
        };
        auto pv = [&](const u16x8 &pw, const u16x8 &pl, int n) __attribute__((always_inline)) {
            f32x4 &od = o[n & 7];
            od = MF::run(__builtin_bit_cast(V8, op[n % kRing]), __builtin_bit_cast(V8, pw), od);
            if constexpr (kLo) od = MF::run(__builtin_bit_cast(V8, op[n % kRing]), __builtin_bit_cast(V8, pl), od);
        };
        f32x4 sa[2], sb[2];
        u16x8 pa = {}, pb = {}, pal = {}, pbl = {};

        // ---- R1: QK a ----
#pragma unroll
        for (int n = 0; n < kLook; n++) fetch(n);
#pragma unroll
        for (int n = 0; n < 8; n++) {
            fetch(n + kLook);
            qk(sa, n);
            if (do_issue && (n & 1)) copy(kn, sn, n >> 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (general) general_x(sa, key0, cl, (uint32_t)bits);
        __builtin_amdgcn_sched_barrier(0);

        // ---- R2: QK b | softmax a (speculative) ----
        const float mneg0 = (m2 == -INFINITY) ? 0.0f : -m2;
        float mxa = 0.0f;
#pragma unroll
        for (int n = 0; n < 8; n++) {
            fetch(8 + n + kLook);
            qk(sb, 8 + n);
            if (n == 0) mxa = max8(sa);
            if (n == 2) probs(sa, 0, gs, mneg0, pa, pal);
            if (n == 5) probs(sa, 1, gs, mneg0, pa, pal);
            if (do_issue && (n & 1)) copy(kn, sn, 4 + (n >> 1));
            __builtin_amdgcn_sched_barrier(0);
        }
        float la = psum(pa, pal);
        // keep the speculative softmax here (it would sink past R3)
        asm volatile("" ::"v"(pa), "v"(la), "v"(mxa));
        if constexpr (kLo) asm volatile("" ::"v"(pal));
        if (general) general_x(sb, key0 + 32, cl, (uint32_t)(bits >> 32));
        __builtin_amdgcn_sched_barrier(0);

        // ---- R3: tile max, reference update (rare) ----
        const float bmax = fmaxf(mxa, max8(sb)) * gs;
        if (__builtin_amdgcn_ballot_w64(bmax > m2 + (8.0f + kUp)) != 0) {   // wave-uniform
            const float rmax = max_pair16(max_half32(bmax));         // over the query's four lanes
            const float mnew = fmaxf(m2, rmax - kUp);
            const float alpha = (m2 == -INFINITY) ? 1.0f : fast_exp2(m2 - mnew);
            m2 = mnew;
            lsum *= alpha;
#pragma unroll
            for (int db = 0; db < 8; db++) o[db] *= alpha;
            const float mn = (m2 == -INFINITY) ? 0.0f : -m2;
            probs(sa, 0, gs, mn, pa, pal);
            probs(sa, 1, gs, mn, pa, pal);
            la = psum(pa, pal);
        }
        const float mneg = (m2 == -INFINITY) ? 0.0f : -m2;
        __builtin_amdgcn_sched_barrier(0);

        // ---- R4: PV a | softmax b ----
#pragma unroll
        for (int n = 0; n < 8; n++) {
            fetch(16 + n + kLook);
            pv(pa, pal, 16 + n);
            if (n == 0) probs(sb, 0, gs, mneg, pb, pbl);
            if (n == 3) probs(sb, 1, gs, mneg, pb, pbl);
            __builtin_amdgcn_sched_barrier(0);
        }
        const float lb = psum(pb, pbl);
        __builtin_amdgcn_sched_barrier(0);

        // ---- R5: PV b ----
#pragma unroll
        for (int n = 0; n < 8; n++) {
            fetch(24 + n + kLook);
            pv(pb, pbl, 24 + n);
            __builtin_amdgcn_sched_barrier(0);
        }
        lsum += la + lb;
    };

    // Per tile: wait for this wave's copies of it (those of the later tiles
    // stay in flight), one barrier (every wave's copies have landed, and
    // every wave is done with the stage the next copies go to), compute.
    int st = 0;
    while (kq[0] < n_kt) {
        const int cls = __builtin_amdgcn_readfirstlane(class_of(kq[0]));
        if constexpr (NST == 4) {
            if (kq[2] < n_kt) MXFA_WAIT_VMCNT(2 * kPer);
            else if (kq[1] < n_kt) MXFA_WAIT_VMCNT(kPer);
            else MXFA_WAIT_VMCNT(0);
        } else {
            static_assert(NST == 2, "stages");
            MXFA_WAIT_VMCNT(0);
        }
        if constexpr (MODE != kNarrowNone)   // V of keys that no row of the job sees (fa_prefill.h)
            if (__builtin_expect(cls & kTileDeadKeys, 0)) {
                const uint32_t dead =
                    SM ? dead_outside(sm_lo, sm_hi, kq[0] * kPfBN + 16 * wave) : wk.dead(kq[0], wave, lane);
                zero_dead_v(dead, lds0 + (uint32_t)(st * kNarrowStage + kTileBytes + 16 * wave * 256));
            }
        __builtin_amdgcn_s_barrier();
        tile(kq[0], cls, st, kq[NST - 1], st == 0 ? NST - 1 : st - 1);
#pragma unroll
        for (int i = 0; i < NST - 1; i++) kq[i] = kq[i + 1];
        kq[NST - 1] = next_live(kq[NST - 2] + 1);
        st = st + 1 == NST ? 0 : st + 1;
    }

    // O leaves as whole rows through the stage after the last tile's, which
    // every wave was done with at the last tile's barrier (fa_wide.hip).
    const float l = sum_pair16(sum_pair32(lsum));
    const float inv = (l == 0.0f) ? 0.0f : 1.0f / l;
    uint8_t *ost = smem + st * kNarrowStage + wave * 8192;
    float *drow = a.dst + ((int64_t)b * a.Sq * a.Nh + head) * kD;   // + q * Nh * kD per row
#pragma unroll
    for (int db = 0; db < 8; db++)
        *(f32x4 *)(ost + n16 * 512 + 16 * ((4 * db + g) ^ n16)) = o[db] * inv;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int rl = 2 * i + (lane >> 5), c = lane & 31;
        const f32x4 v = *(const f32x4 *)(ost + rl * 512 + 16 * (c ^ rl));
        if (q0w + rl < a.Sq) *(f32x4 *)(drow + (int64_t)(q0w + rl) * a.Nh * kD + 4 * c) = v;
    }
}

template <int T, int MODE, bool CAP, int NST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
fa_narrow_kernel(const FaArgs a) {
    fa_narrow_body<T, MODE, CAP, NST>(a);
}

template <int T, int MODE, bool CAP, int NST>
static hipError_t launch_nst(const FaArgs &a, hipStream_t stream) {
    constexpr int bytes = narrow_lds<NST>();
    // (the dynamic LDS limit is per function and device, set once on each)
    static OncePerDevice attr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    e = attr.run(dev, [] {
        return hipFuncSetAttribute((const void *)fa_narrow_kernel<T, MODE, CAP, NST>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    });
    if (e != hipSuccess) return e;
    const dim3 grid((uint32_t)a.n_qt_n * (uint32_t)a.Nh * (uint32_t)a.B);
    hipLaunchKernelGGL((fa_narrow_kernel<T, MODE, CAP, NST>), grid, dim3(256), bytes, stream, a);
    return hipGetLastError();
}

template <int T, bool CAP>
static hipError_t launch_mode(const FaArgs &a, hipStream_t stream) {
    const int64_t jobs = (int64_t)a.n_qt_n * a.Nh * a.B;
    if (a.sm_flags) return launch_nst<T, kNarrowSm, CAP, 4>(a, stream);
    if (a.mask) return a.mask_unal ? launch_nst<T, kNarrowUnal, CAP, 4>(a, stream)
                                   : launch_nst<T, kNarrowDense, CAP, 4>(a, stream);
    return jobs <= kPfCus ? launch_nst<T, kNarrowNone, CAP, 4>(a, stream) : launch_nst<T, kNarrowNone, CAP, 2>(a, stream);
}

// Masked calls of at most one workgroup per CU, unmasked ones of at most
// two.  Measured per call against the kernels with more queries per
// workgroup (F16 unless said, 16 heads):
//   workgroups  no mask        bf16           window 128     2.. x 500 keys
//   64          13.1 (14.5)    12.9 (12.3)    16.6 (19.0)    19.5 (21.1) us
//   128         12.2 (20.8)    13.4 (18.2)    17.1 (20.3)    19.4 (21.3)
//   256         13.0 (21.4)    14.2 (19.3)    17.8 (21.8)    21.0 (22.6)
//   352         20.2 (26.5)    23.1 (24.2)    21.0 (22.7)    23.9 (23.4)
//   480         44.2 (54.8)    51.8 (51.7)    23.9 (25.4)    25.0 (24.5)
//   544         41.0 (36.3)    47.0 (48.5)    27.2 (29.0)    34.8 (29.7)
// A causal mask as metadata over 2000 earlier keys, 384 workgroups of 32
// heads: 68.8 (68.0).  A mask and its structured form keep to one rule, so
// that both take the same kernel.
bool fa_narrow_serves(const FaArgs &a) {
    const int64_t jobs = (int64_t)((a.Sq + kPfNarrowBM - 1) / kPfNarrowBM) * a.Nh * a.B;
    return jobs <= (a.mask || a.sm_flags ? kPfCus : 2 * kPfCus);
}

hipError_t launch_fa_narrow(const FaArgs &a, int ktype, hipStream_t stream) {
    const bool cap = a.softcap != 0.0f;
    switch (ktype) {
        case T_F16: return cap ? launch_mode<T_F16, true>(a, stream) : launch_mode<T_F16, false>(a, stream);
        case T_BF16: return cap ? launch_mode<T_BF16, true>(a, stream) : launch_mode<T_BF16, false>(a, stream);
        default: return hipErrorInvalidValue;   // (Q8_0 calls stay on fa_mfma.hip: level at best)
    }
}

}  // namespace mxfa
