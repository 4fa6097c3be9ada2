// mxfa_common.h -- shared device types and helpers for the gfx950 kernels.
//
// Layout conventions used by every kernel (ggml order, ne[0] innermost):
//   q   F32  [D, Sq, Nh, B]   strided view (q_nb1..3)
//   k,v F16/BF16 [D, Skv, Nkv, Bk] (k_nb1..3 / v_nb1..3), or Q8_0 blocks
//   mask F16 [>=Skv, >=Sq, Nm2, Nm3] (m_nb1..3), broadcast by modulo
//   dst F32 [D, Nh, Sq, B] contiguous
// A "row" of the attention problem is one (query iq1, q head) pair; the
// rows that share one KV head (GQA) are packed together into MFMA tiles.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace mxfa {

constexpr int kD = 128;                 // head size handled by the kernels
constexpr float kLog2e = 1.4426950408889634f;

enum : int { T_F32 = 0, T_F16 = 1, T_Q8_0 = 8, T_BF16 = 30 };

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

// Structured masks (mxfa_flash_attn_ext_masked): the mask as metadata.  Key
// j is live for query row i of batch b iff
//   j < len[b % n_len]            (kSmLengths: padding, qwen3-lm.h:879,
//                                  dit-sampler.h:303)
//   j <= pos0 + i                 (kSmCausal: qwen3-lm.h:605, qwen3-enc.h:433)
//   |pos0 + i - j| <= window      (kSmWindow: dit-sampler.h:282,
//                                  cond-enc.h:317, :341)
// -- the same as a dense F16 mask holding 0 there and -inf elsewhere.
// kSmDevice: lengths (and pos0 when sm_pos0_dev is set) live in device
// memory and are read by the kernels when they run, so a captured launch
// follows values the host rewrites between graph replays.
constexpr int kSmCausal = 1, kSmWindow = 2, kSmLengths = 4, kSmDevice = 8;
constexpr int kSmMaxLen = 64;   // per-batch lengths carried in the arguments

// n / d for 0 <= n < 2^31 by a multiplication: with s = ceil(log2 d) and
// mul = floor(2^32 (2^s - d) / d) + 1, n / d = (mulhi(n, mul) + n) >> s
// (Granlund and Montgomery, "Division by invariant integers using
// multiplication", 1994).  A division by an argument takes the kernels ~150
// cycles of dependent instructions; their prologues had a dozen ahead of the
// first load.
struct FastDiv {
    uint32_t mul, sh;
};
inline FastDiv fast_div(uint32_t d) {
    const uint32_t s = d > 1 ? 32 - (uint32_t)__builtin_clz(d - 1) : 0;
    return FastDiv{(uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << s) - d)) / d + 1), s};
}
__device__ __forceinline__ int div_fast(int n, FastDiv f) { return (int)((__umulhi((uint32_t)n, f.mul) + (uint32_t)n) >> f.sh); }
__device__ __forceinline__ int mod_fast(int n, FastDiv f, int d) { return n - div_fast(n, f) * d; }

// Arguments shared by the attention kernels (passed by value).
struct FaArgs {
    const char *q, *k, *v, *mask;
    float *dst;
    int64_t q_nb1, q_nb2, q_nb3;
    int64_t k_nb1, k_nb2, k_nb3;
    int64_t v_nb1, v_nb2, v_nb3;
    int64_t m_nb1, m_nb2, m_nb3;
    int32_t m_ne2, m_ne3;
    int32_t Sq, Nh, B, Skv, Nkv, G, rk3;  // G = Nh/Nkv, rk3 = B/Bk
    FastDiv fd_G, fd_rk3, fd_m2, fd_m3;   // dividers of G, rk3, m_ne2, m_ne3
    FastDiv fd_nkv;                       // Nkv
    FastDiv fd_rt, fd_gy, fd_hs, fd_chunk;   // decode: row_tiles, Nkv * row_tiles, n_splits / 2, chunk
    FastDiv fd_unit, fd_kt, fd_qt;        // prefill: G * query tiles of the kernel that runs, n_kt, n_qt
    int32_t M;                            // rows per (b, kv head) = Sq*G
    int32_t row_tiles;                    // decode kernel: ceil(M/16)
    float scale, softcap;                 // softcap == 0: off
    float max_bias, l2m0, l2m1;           // ALiBi (max_bias == 0: off): log2 of ggml's m0, m1
    float softcap_in;                     // scale / softcap (softcap != 0)
    uint32_t n_head_log2;
    // mask row alignment (8 / 16 bytes for every row start); mask_vec4:
    // 8-byte aligned rows holding at least round_up(Skv, 4) entries;
    // mask_vec16: the same with at least 16 entries (16-key DMA blocks)
    int32_t mask_al8, mask_al16, mask_vec4, mask_vec16;
    int32_t mask_unal;                    // prefill: rows not 8-byte aligned, or not of a multiple of 4 entries
    uint32_t m_plane_bytes;               // prefill: bytes of one mask plane, (ne1 - 1) * nb1 + 2 * ne0
    // split-KV
    int32_t n_splits, chunk;
    int32_t dec_live;                     // > 0: decode grid is the list of live splits (structured masks)
    int32_t dec_pair;                     // > 0: paired splits, the even split of a pair streams dec_pair keys
    float *part_o, *part_ml;
    int *tickets;                         // one per (b, kv head, row tile), zero between calls
    // prefill: per (mask plane, q tile, k tile) class (see fa_mfma.hip), and
    // for the mixed tiles whose values are all 0 or -inf (class 3) one 64-bit
    // liveness word per query row (NULL: no words, no class 3)
    const uint8_t *tile_class;
    uint64_t *tile_bits;
    uint64_t *tile_keys;                  // keys that some row of a 64-query half of a tile may see
    int32_t n_qt, n_kt;                   // tiles along Sq and Skv
    const uint8_t *tile_class64;          // the same classes per 64-query half of a tile (fa_narrow.hip)
    int32_t pf_parts, pf_tiles;           // fa_mfma.hip: key split, workgroups per job (0: none), live tiles per part
    FastDiv fd_parts, fd_tiles;
    int32_t n_qt_n;                       // fa_narrow.hip: 64-query tiles along Sq
    int32_t n_qt_w;                       // fa_wide.hip: 192-query tiles along Sq (0: not used)
    int32_t n_kt_pad;                     // class row stride (n_kt rounded up to 4)
    // structured mask (sm_flags == 0: none; then `mask` may hold a dense one)
    int32_t q16;                          // Q stored in K's 16-bit type (no conversion on load)
    int32_t sm_flags, sm_window, sm_pos0, sm_nlen;
    const int32_t *sm_len_dev;            // kSmDevice: lengths in device memory (else sm_len)
    const int32_t *sm_pos0_dev;           // kSmDevice: pos0 in device memory, or NULL (sm_pos0)
    int32_t sm_len[kSmMaxLen];            // (sm_nlen is 1 or B)
};

// Brings the kernel arguments (all but the structured mask's lengths) into
// the scalar cache with one dword per 64-byte line, all in flight together.
// The compiler loads arguments in groups where it needs them, each group a
// cold miss of its own: three in a row ahead of a decode workgroup's first
// load.
__device__ __forceinline__ void warm_args() {
    typedef const __attribute__((address_space(4))) int32_t karg;
    karg *p = (karg *)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int kLines = (int)((offsetof(FaArgs, sm_len) + 63) / 64);
    static_assert(kLines <= 10, "lines listed below");
    int x[10];
#pragma unroll
    for (int i = 0; i < 10; i++) x[i] = p[16 * (i < kLines ? i : kLines - 1)];
    asm volatile("" ::"s"(x[0]), "s"(x[1]), "s"(x[2]), "s"(x[3]), "s"(x[4]), "s"(x[5]), "s"(x[6]), "s"(x[7]),
                 "s"(x[8]), "s"(x[9]));
}

// Cross-lane steps at VALU latency (DPP, v_permlane*_swap) instead of LDS
// crossbar permutes (ds_bpermute, ~100 cycles each).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
}
// AND over the 16 lanes of each row: quad_perm [1,0,3,2] and [2,3,0,1]
// combine each quad, row_half_mirror (i <- 7-i) the two quads of each 8,
// row_mirror (i <- 15-i) the two 8s.  Needs every lane active.
__device__ __forceinline__ uint32_t and_rows16(uint32_t v) {
    v &= dpp_u32<0xB1>(v);
    v &= dpp_u32<0x4E>(v);
    v &= dpp_u32<0x141>(v);
    v &= dpp_u32<0x140>(v);
    return v;
}
// OR over the 16 lanes of each row (the same DPP steps as and_rows16).
__device__ __forceinline__ uint32_t or_rows16(uint32_t v) {
    v |= dpp_u32<0xB1>(v);
    v |= dpp_u32<0x4E>(v);
    v |= dpp_u32<0x141>(v);
    v |= dpp_u32<0x140>(v);
    return v;
}
// max of x over lanes l and l ^ 16 (v_permlane16_swap pairs rows r, r ^ 1)
// and over lanes l and l ^ 32 (v_permlane32_swap pairs the two halves)
__device__ __forceinline__ float max_pair16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                    false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __forceinline__ float max_half32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                    false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}

// sum of x over lanes l and l ^ 32, l ^ 16
__device__ __forceinline__ float sum_pair32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                    false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float sum_pair16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                    false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
// max / sum of x over the wave's 64 lanes (the DPP steps of and_rows16, then
// the row pairs); every lane active, every lane gets the result
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, dpp_u32<CTRL>(__builtin_bit_cast(uint32_t, v)));
}
__device__ __forceinline__ float wave_max(float x) {
    x = fmaxf(x, dpp_f<0xB1>(x));
    x = fmaxf(x, dpp_f<0x4E>(x));
    x = fmaxf(x, dpp_f<0x141>(x));
    x = fmaxf(x, dpp_f<0x140>(x));
    return max_half32(max_pair16(x));
}
__device__ __forceinline__ float wave_sum(float x) {
    x += dpp_f<0xB1>(x);
    x += dpp_f<0x4E>(x);
    x += dpp_f<0x141>(x);
    x += dpp_f<0x140>(x);
    return sum_pair32(sum_pair16(x));
}
__device__ __forceinline__ int wave_max_i(int x) {
    x = max(x, (int)dpp_u32<0xB1>((uint32_t)x));
    x = max(x, (int)dpp_u32<0x4E>((uint32_t)x));
    x = max(x, (int)dpp_u32<0x141>((uint32_t)x));
    x = max(x, (int)dpp_u32<0x140>((uint32_t)x));
    const auto r = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
    x = max((int)(uint32_t)r[0], (int)(uint32_t)r[1]);
    const auto q = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
    return max((int)(uint32_t)q[0], (int)(uint32_t)q[1]);
}

// Live keys [lo, hi) of query row iq1 of batch b under the structured mask
// (both ends are non-decreasing in iq1, so the rows of a tile cover
// [lo(first row), hi(last row)) and all of them see [lo(last), hi(first))).
// With kSmDevice the values come from device memory (the host never calls
// this for such a spec); they are clamped here, as the host checks the
// others: pos0 to [0, 2^30), a negative length to 0.
// The device values are read with relaxed agent-scope atomic loads: a plain
// load would let the compiler fold "device pointer or kernel-argument array"
// into one flat load through a selected pointer, which read wrong lengths.
__device__ __forceinline__ int sm_dev_load(const int32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__host__ __device__ __forceinline__ void sm_row_range(const FaArgs &a, int b, int iq1, int &lo, int &hi) {
    int p0 = a.sm_pos0;
#if defined(__HIP_DEVICE_COMPILE__)
    if (a.sm_pos0_dev) {
        const int d = sm_dev_load(a.sm_pos0_dev);
        p0 = d < 0 ? 0 : (d > (1 << 30) - 1 ? (1 << 30) - 1 : d);
    }
#endif
    const int p = p0 + iq1;
    lo = 0;
    hi = a.Skv;
    if (a.sm_flags & kSmLengths) {
        int len = a.sm_len[a.sm_nlen == 1 ? 0 : b];
#if defined(__HIP_DEVICE_COMPILE__)
        if (a.sm_len_dev) len = sm_dev_load(a.sm_len_dev + (a.sm_nlen == 1 ? 0 : b));
#endif
        len = len < 0 ? 0 : len;
        hi = hi < len ? hi : len;
    }
    if (a.sm_flags & kSmCausal) hi = hi < p + 1 ? hi : p + 1;
    if (a.sm_flags & kSmWindow) {
        lo = lo > p - a.sm_window ? lo : p - a.sm_window;
        hi = hi < p + a.sm_window + 1 ? hi : p + a.sm_window + 1;
    }
}

// MFMA 16x16x32 for the two 16-bit float formats (8 k-values per lane).
template <int T> struct Mfma16;
template <> struct Mfma16<T_F16> {
    typedef f16x8 v8;
    static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint16_t from_f32(float x) {
        return __builtin_bit_cast(uint16_t, (_Float16)x);
    }
};
template <> struct Mfma16<T_BF16> {
    typedef bf16x8 v8;
    static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint16_t from_f32(float x) {
        return __builtin_bit_cast(uint16_t, (__bf16)x);
    }
};

// MFMA 32x32x16 for the two 16-bit float formats (8 k-values per lane).
template <int T> struct Mfma32;
template <> struct Mfma32<T_F16> {
    typedef f16x8 v8;
    static __device__ __forceinline__ f32x16 run(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma32<T_BF16> {
    typedef bf16x8 v8;
    static __device__ __forceinline__ f32x16 run(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

__device__ __forceinline__ float h2f_bits(uint16_t h) {
    return (float)__builtin_bit_cast(_Float16, h);
}

// Convert 8 floats to 8 16-bit values of format T (round to nearest even),
// returned as the raw bits.
template <int T>
__device__ __forceinline__ u16x8 cvt8(f32x4 lo, f32x4 hi) {
    u16x8 r;
    r[0] = Mfma16<T>::from_f32(lo[0]);
    r[1] = Mfma16<T>::from_f32(lo[1]);
    r[2] = Mfma16<T>::from_f32(lo[2]);
    r[3] = Mfma16<T>::from_f32(lo[3]);
    r[4] = Mfma16<T>::from_f32(hi[0]);
    r[5] = Mfma16<T>::from_f32(hi[1]);
    r[6] = Mfma16<T>::from_f32(hi[2]);
    r[7] = Mfma16<T>::from_f32(hi[3]);
    return r;
}

// bf16 keeps 8 significant bits: a probability rounded once to bf16 for the
// PV product is off by up to 2^-9 relative, which on short or peaked rows
// moves the output by ~1e-3.  The bf16 kernels therefore feed the PV MFMA
// twice, with hi = RNE_bf16(p) and lo = RNE_bf16(p - hi): hi + lo carries
// p to ~2^-17 relative.  bf16_lo returns the raw bits of lo for the hi
// part `h` (raw bits) of p; p - hi is exact in fp32.
__device__ __forceinline__ uint16_t bf16_lo(float p, uint16_t h) {
    return __builtin_bit_cast(uint16_t, (__bf16)(p - __builtin_bit_cast(float, (uint32_t)h << 16)));
}
// P of two keys as the PV product's operand pairs (raw bits): bf16 as above.
// In f16, which carries P to ~2^-22 so (the decode kernels, whose error then
// does not depend on how the keys are split, and the prefill kernels under odd
// mask rows), hi is cut below p, not rounded: lo = RNE_f16(p - hi) >= p 2^-14
// is then positive, and an infinity of V stays one in both products (inf * 0
// or inf * -x would make it NaN).  So that lo is not rounded to 0 for small
// weights, these kernels hold their maxima kPairUp low (pair_up): P is at most
// 2^(8 + 7), and lo positive down to weights of 2^-18.  (hi rounded: one token
// over 4096 keys 2.4e-7 of 64 bits; cut at p (1 - 2^-11) 3.0e-7, at 1 - 2^-14
// 2.7e-7.)
constexpr float kPairUp = 7.0f;
template <int T> constexpr float pair_up() { return T == T_F16 ? kPairUp : 0.0f; }
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int T>
__device__ __forceinline__ void p_pair(float p0, float p1, u16x2 &hi, u16x2 &lo) {
    if constexpr (T == T_BF16) {
        hi = u16x2{Mfma16<T>::from_f32(p0), Mfma16<T>::from_f32(p1)};
        lo = u16x2{bf16_lo(p0, hi[0]), bf16_lo(p1, hi[1])};
    } else {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        constexpr float kBelow = 1.0f - 0x1p-14f;
        hi = __builtin_bit_cast(u16x2, __builtin_amdgcn_cvt_pkrtz(p0 * kBelow, p1 * kBelow));
        const f32x2 r = {p0 - h2f_bits(hi[0]), p1 - h2f_bits(hi[1])};
        lo = __builtin_bit_cast(u16x2, __builtin_convertvector(r, h2));
    }
}
template <int T>
__device__ __forceinline__ void p_pair8(f32x4 a, f32x4 b, u16x8 &hi, u16x8 &lo) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        u16x2 h, l;
        p_pair<T>(i < 2 ? a[2 * i] : b[2 * i - 4], i < 2 ? a[2 * i + 1] : b[2 * i - 3], h, l);
        hi[2 * i] = h[0];
        hi[2 * i + 1] = h[1];
        lo[2 * i] = l[0];
        lo[2 * i + 1] = l[1];
    }
}

// Sum of 8 16-bit values of format T (the rounded probabilities that feed
// the PV product) with v_dot2 against (1, 1): the softmax denominator then
// sums exactly the weights the numerator uses.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
template <int T>
__device__ __forceinline__ float sum8(u16x8 p, float acc) {
    const u32x4 w = __builtin_bit_cast(u32x4, p);
    if constexpr (T == T_F16) {
        const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t wi = w[i];   // bit_cast of a vector element lvalue reads element 0
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, wi), one, acc, false);
        }
    } else {
        const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t wi = w[i];
            acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, wi), one, acc, false);
        }
    }
    return acc;
}

// ALiBi slope of head h (ggml's formula m0^(h+1), or m1^(2(h - n_head_log2)
// + 1); 1 when max_bias == 0), as exp2(e * log2 m) with the host's log2 of
// m0 and m1 (inline: a libm pow call would cost a register save per call
// site).
__device__ __forceinline__ float alibi_slope(const FaArgs &a, int h) {
    if (a.max_bias <= 0.0f) return 1.0f;
    const uint32_t hu = (uint32_t)h;
    return hu < a.n_head_log2 ? __builtin_amdgcn_exp2f(a.l2m0 * (float)(hu + 1))
                              : __builtin_amdgcn_exp2f(a.l2m1 * (float)(2 * (hu - a.n_head_log2) + 1));
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// tanh(x) = 1 - 2 / (e^(2x) + 1) with the hardware exp2 and reciprocal
// (absolute error ~1e-7; saturates to +-1, e^(2x) = inf gives 1).  Inline
// on purpose: a library call inside the attention loops costs a full
// register save per call site.
__device__ __forceinline__ float fast_tanh(float x) {
    const float e = fast_exp2(x * (2.0f * kLog2e));
    return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}

// s_waitcnt immediates (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] |
// lgkmcnt[11:8] | vmcnt[5:4] << 14).
#define MXFA_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))
#define MXFA_WAIT_LGKMCNT0() __builtin_amdgcn_s_waitcnt(0xC07F)

typedef __attribute__((address_space(3))) void lds_void;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Direct HBM -> LDS copy of 16 bytes per lane: lane l's bytes land at LDS
// address lds_addr + 16*l (lds_addr must be the same for the whole wave).
//
// Issued as inline assembly on purpose: the compiler's own wait insertion
// treats every LDS read after such a copy as a possible alias and drains
// all outstanding copies (vmcnt(0)) before it, which serialises a
// multi-buffer prefetch.  Callers wait with MXFA_WAIT_VMCNT before reading a
// buffer.  Compiler-generated waits for other vector loads stay correct: a
// copy unknown to the compiler only makes them wait longer (counters retire
// in order).
// The s_nop is the wait state that a scalar write of M0 needs ahead of an LDS
// copy (the compiler keeps it for its own copies, not inside inline assembly).
__device__ __forceinline__ void dma16_at(const void *g, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(g)
                 : "memory", "m0");
}
// The same with 4 bytes per lane (4-byte aligned source): lane l's bytes
// land at lds_addr + 4*l.
__device__ __forceinline__ void dma4_at(const void *g, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(g)
                 : "memory", "m0");
}

// Buffer resource over `bytes` bytes from `base`, offset addressed (stride
// 0): a load at or past `bytes` returns zeros and touches no memory.
__device__ __forceinline__ i32x4 buf_rsrc(const void *base, uint32_t bytes) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    i32x4 r;
    r[0] = (int)__builtin_amdgcn_readfirstlane((uint32_t)b);
    r[1] = (int)((uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) & 0xFFFFu);
    r[2] = (int)__builtin_amdgcn_readfirstlane(bytes);
    r[3] = 0x00020000;   // 32-bit data format, no swizzle, no stride
    return r;
}

// HBM -> LDS copy of 16 bytes per lane through a buffer resource: lane l
// reads base + voff(l) (zeros, and no memory access, when voff(l) + 16
// exceeds the resource's size) and its bytes land at LDS address
// lds_addr + 16*l.  Same wait contract as dma16 (callers wait with
// MXFA_WAIT_VMCNT before reading the buffer).
__device__ __forceinline__ void dma16_buf(const i32x4 &rsrc, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc)
                 : "memory", "m0");
}

// The same with 4 bytes per lane (bytes land at lds_addr + 4*l).
__device__ __forceinline__ void dma4_buf(const i32x4 &rsrc, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc)
                 : "memory", "m0");
}

// 16 bytes stored at agent scope: global_store_dwordx4 with sc1, the
// encoding a relaxed agent-scope atomic store of each element gets on this
// architecture (written through past the XCD's L2), in one transaction
// instead of four.  Complete at device scope once vmcnt drains.
// The s_nop belongs to the store: a store of more than 8 bytes may still be
// reading its data registers when the next instruction writes them (one wait
// state, which the compiler keeps for its own stores but not behind inline
// assembly; without it, lanes 12-15 and 28-31 stored the address arithmetic
// that followed).
__device__ __forceinline__ void st_agent16(float *p, f32x4 v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

__device__ __forceinline__ void st_agent8(float *p, float x, float y) {   // 8-byte aligned
    __hip_atomic_store((uint64_t *)p, ((uint64_t)__builtin_bit_cast(uint32_t, y) << 32) | __builtin_bit_cast(uint32_t, x),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 8 bytes (8-byte aligned) loaded at agent scope, from the coherence point.
__device__ __forceinline__ u32x2 ld_dev2(const float *p) {
    return __builtin_bit_cast(u32x2, __hip_atomic_load((const uint64_t *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// LDS transpose read of four 16-bit values.  Within each group of 16 lanes,
// lane j receives element (j % 4) of the 8-byte chunks addressed by lanes
// j/4 + 4e, e = 0..3 (gfx950 ds_read_b64_tr_b16).
__device__ __forceinline__ u16x4 lds_read_tr16(const void *p) {
    return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p));
}

// XOR swizzles of the 16-byte chunks of a 256-byte K or V row stored in
// LDS (key k, logical chunk c at slot c ^ swz(k)).  K: consecutive keys
// read the same chunk (MFMA A operand), k & 15 spreads them over all banks.
// V: transpose reads fetch 4 consecutive keys x 32 bytes per 16 lanes;
// swz_v keeps those (and the neighbouring 16-lane group) conflict-free.
__device__ __forceinline__ int swz_k(int k) { return k & 15; }
__device__ __forceinline__ int swz_v(int k) { return (((k & 3) << 1) ^ ((k & 1) << 3)) ^ (((k >> 2) & 1) << 1); }

}  // namespace mxfa
