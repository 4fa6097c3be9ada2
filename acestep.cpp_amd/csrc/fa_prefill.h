// fa_prefill.h -- pieces shared by the three MFMA prefill kernels
// (fa_mfma.hip: 32 queries per wave; fa_wide.hip: 48; fa_narrow.hip: 16):
// LDS tile geometry, the XCD-aware job order, tile classes held in
// registers, and cross-lane pair reductions.
#pragma once

#include "mxfa_common.h"
#include "mxfa_internal.h"

namespace mxfa {

constexpr int kTileBytes = 16384;            // K or V rows of one 64-key tile
constexpr int kStageBytes = 2 * kTileBytes;  // K + V
constexpr int kPfLds = 2 * kStageBytes;      // double buffered: 64 KB
constexpr uint32_t kXcds = 8;                // MI355X: workgroups go round-robin to 8 XCDs
constexpr uint32_t kCusPerXcd = 32;          // 256 CUs
constexpr int64_t kPfCus = 256;

// Job of this workgroup among n_qt * Nh * B (query tile, q head, batch)
// jobs.  Workgroup ids go round-robin to the XCDs; each XCD gets a
// contiguous block of the job list, which is ordered by (batch, kv head),
// then by query tile from the last (longest under a causal mask) down, then
// by q head within the GQA group: the q tiles that share K/V rows run on one
// XCD and share its L2.  Within an XCD the order snakes over rounds of
// kCusPerXcd: the XCD's dispatcher gives each CU one workgroup per round, so
// odd rounds run reversed and a CU pairs a long causal tile with a short
// one.  `second`: the workgroup is the CU's second of the first pair (every
// CU of the XCD holds a pair).
__device__ __forceinline__ void pf_place(const FaArgs &a, int n_qt, int J, int &qt, int &head, int &kvh, int &b) {
    // job J: (batch, kv head) major, then the query tile from the last one
    // down, then the q head within the group
    const int u = div_fast(J, a.fd_unit), r = J - u * a.G * n_qt, t = div_fast(r, a.fd_G);
    qt = __builtin_amdgcn_readfirstlane(n_qt - 1 - t);
    b = __builtin_amdgcn_readfirstlane(div_fast(u, a.fd_nkv));
    kvh = __builtin_amdgcn_readfirstlane(u - b * a.Nkv);
    head = __builtin_amdgcn_readfirstlane(kvh * a.G + r - t * a.G);
}
__device__ __forceinline__ void pf_job(const FaArgs &a, int n_qt, int &qt, int &head, int &kvh, int &b, bool &second) {
    const uint32_t L = __builtin_amdgcn_workgroup_id_x();
    const uint32_t N = (uint32_t)(n_qt * a.Nh * a.B);
    const uint32_t nq = N / kXcds, nr = N % kXcds, x = L % kXcds, s0 = L / kXcds;
    const uint32_t n_x = x < nr ? nq + 1 : nq;
    const uint32_t rnd = s0 / kCusPerXcd, w = s0 % kCusPerXcd;
    const uint32_t cnt = min(kCusPerXcd, n_x - rnd * kCusPerXcd);
    const uint32_t s = (rnd & 1) ? rnd * kCusPerXcd + (cnt - 1 - w) : s0;
    const uint32_t J = x < nr ? x * (nq + 1) + s : nr * (nq + 1) + (x - nr) * nq + s;
    pf_place(a, n_qt, (int)J, qt, head, kvh, b);
    second = rnd == 1 && n_x >= 2 * kCusPerXcd;
}

// The same for a key-split grid of n_qt * Nh * B * a.pf_parts workgroups: the
// parts of a job are neighbours on one XCD, jobs in pf_job's order.
__device__ __forceinline__ void pf_unit(const FaArgs &a, int n_qt, int &job, int &part, int &qt, int &head, int &kvh,
                                        int &b) {
    const uint32_t L = __builtin_amdgcn_workgroup_id_x();
    const uint32_t N = (uint32_t)(n_qt * a.Nh * a.B) * (uint32_t)a.pf_parts;
    const uint32_t nq = N / kXcds, nr = N % kXcds, x = L % kXcds;
    const int U = (int)(x * nq + min(x, nr) + L / kXcds);
    job = __builtin_amdgcn_readfirstlane(div_fast(U, a.fd_parts));
    part = __builtin_amdgcn_readfirstlane(U - job * a.pf_parts);
    pf_place(a, n_qt, job, qt, head, kvh, b);
}

// Tile classes of one (plane, query tile) row live in registers: lane l
// holds the class bytes of key tiles 4l..4l+3 (w0: tiles < 256, w1: tiles
// 256..511), read with v_readlane (uniform, no memory wait in the loop).
struct TileClasses {
    uint32_t w0, w1;
    bool present;
    __device__ __forceinline__ int at(int kt) const {
        if (!present) return 1;
        const uint32_t w = kt < 256 ? __builtin_amdgcn_readlane(w0, (kt >> 2) & 63)
                                    : __builtin_amdgcn_readlane(w1, ((kt - 256) >> 2) & 63);
        return (int)((w >> (8 * (kt & 3))) & 0xFFu);
    }
    // live tiles among the first n (every lane active)
    __device__ __forceinline__ int count(int n, int lane) const {
        if (!present) return n;
        int c = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(4 * lane + i < n && ((w0 >> (8 * i)) & 0xFFu)));
            c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(256 + 4 * lane + i < n && ((w1 >> (8 * i)) & 0xFFu)));
        }
        return c;
    }
    // (readfirstlane: the result is wave-uniform, and the compiler must
    // know it to keep the tile loop on scalar branches)
    __device__ __forceinline__ int next_live(int kt, int n) const {
        if (!present) return kt;
        while (kt < n && at(kt) == 0) kt++;
        return __builtin_amdgcn_readfirstlane(kt);
    }
};

// Class bytes (0 all -inf, 1 all zero, 2 mixed) of the union of two row
// ranges' tiles, four at a time: equal classes stand, different ones make
// the tile mixed, with dead keys to look for.
__device__ __forceinline__ uint32_t class_union4(uint32_t x, uint32_t y) {
    const uint32_t d = x ^ y;
    const uint32_t nz = (((d & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | d) & 0x80808080u;   // bit 7: byte differs
    const uint32_t m = (nz >> 7) * 0xFFu;
    return (x & ~m) | (0x01010101u * (2 | kTileDeadKeys) & m);
}

// Max of a lane's value and the same register of lane l ^ 32 (one
// v_permlane32_swap).
__device__ __forceinline__ float max_pair32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                    false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}

// Keys that no query of a workgroup may see have P = 0, but 0 times a NaN or
// an infinity in a masked V slot would be NaN in every row of the tile (ggml
// skips such keys: ggml-cpu/ops.cpp, flash_attn_ext_f16_one_chunk).  Each wave
// zeroes the V rows of such keys among the 16 it has copied, before the
// tile's barrier, in the tiles that have any (kTileDeadKeys).  The other tiles
// pay a test: 2 x 1085 tokens under a window of 128 34.1 -> 34.4 us, over 238
// encoder keys with 31 of padding 25.7 -> 26.2, eight encoder layers 96.6 ->
// 97.9.  (Measured and dropped: masking the V operands of mixed tiles, 5 to 8
// % on the DiT's masked calls; leaving the rows out of the copies, 3 %; a look
// at O and a second pass where it is not finite, 2 %, and 10 % where that pass
// made the compiler spill.)
//
// WaveKeys: the keys that some row of the job may see among the 16 of each
// tile that this wave copies; lane l holds those of tile base + l.
struct WaveKeys {
    const uint32_t *p = nullptr;   // this wave's half word of tile 0, first row (NULL: not known)
    int rows = 0, n_kt = 0, base = 0;
    uint32_t u = 0;
    __device__ __forceinline__ void load(int base_, int lane) {
        base = base_;
        u = 0;
        if (base + lane < n_kt)
            for (int r = 0; r < rows; r++) u |= p[2 * ((int64_t)r * n_kt + base + lane)];
    }
    // row0: the job's first 64-query row of the plane (of 2 * a.n_qt)
    __device__ __forceinline__ void init(const FaArgs &a, int plane, int row0, int rows_, int wave, int lane) {
        if (!a.tile_keys) return;
        rows = min(rows_, 2 * a.n_qt - row0);
        n_kt = a.n_kt;
        p = (const uint32_t *)(a.tile_keys + ((int64_t)plane * 2 * a.n_qt + row0) * n_kt) + (wave >> 1);
        load(0, lane);
    }
    // bit j: no query sees key 16 wave + j of tile kt (uniform; every lane active)
    __device__ __forceinline__ uint32_t dead(int kt, int wave, int lane) {
        if (!p) return 0;
        if (kt - base >= 64 || kt < base) load(kt & ~63, lane);
        return ~((uint32_t)__builtin_amdgcn_readlane(u, kt & 63) >> (16 * (wave & 1))) & 0xFFFFu;
    }
};
// The same where the rows together see the keys [lo, hi); key0: the wave's first.
__device__ __forceinline__ uint32_t dead_outside(int lo, int hi, int key0) {
    const int l = min(max(lo - key0, 0), 16), h = min(max(hi - key0, 0), 16);
    return ~((0xFFFFu << l) & ((1u << h) - 1u)) & 0xFFFFu;
}
// v: LDS address of the wave's first V row (copy c: key 4c + lane / 16, 16
// bytes a lane).  Three registers: the lane id is counted anew and the zeros
// go out as dwords, or fa_wide.hip, which has none to spare, spills.
__device__ __forceinline__ void zero_dead_v(uint32_t dead, uint32_t v) {
    const uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const uint32_t addr = v + 16 * lane;
    for (uint32_t c = 0; c < 4; c++)
        if ((dead >> (4 * c + (lane >> 4))) & 1u)
            asm volatile("ds_write_b32 %0, %1\n\tds_write_b32 %0, %1 offset:4\n\t"
                         "ds_write_b32 %0, %1 offset:8\n\tds_write_b32 %0, %1 offset:12"
                         :
                         : "v"(addr + 1024 * c), "v"(0u)
                         : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}
}  // namespace mxfa
