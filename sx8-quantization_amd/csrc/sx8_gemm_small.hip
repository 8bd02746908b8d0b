// sx8_gemm_small.hip -- Y (M, N) = X (M, K) . W^T for a few rows (M <= 128: batched decode,
// short prompts), W in S-X8 blocks.
//
// What bounds it: the decode's VALU work and the packed weights (30 bytes per 32 weights, read
// once); past ~4 row fragments the X operands, which every wave reads through the vector
// cache; for the small layer shapes launch and memory latency (~3.3 us).  The tiled kernels
// of sx8_gemm.hip spend a 128-row tile on these calls, decode through LDS with a barrier per
// K block and split K over work-groups (a second launch adds the partials).  Here a weight
// goes from memory to the matrix core without LDS and K is split over the waves of one
// work-group:
//   * v_mfma_f32_16x16x32_f16 multiplies 32 K values of 16 columns and 16 rows; lane l = 16 g
//     + c supplies 8 consecutive weights of column c, so a lane decodes one 8-weight sub-block
//     straight into the A operand.  The D rows are the columns, the D columns the rows of X;
//   * records are loaded four K blocks at a time: lane (c, t) loads the whole 30-byte record
//     of (column c, block t) -- one wave load per field covers 64 records, where a load per
//     sub-block would need four times the memory instructions -- and does the range
//     arithmetic of its record's four sub-blocks.  MFMA j of a group of four blocks then takes
//     sub-block j of each lane's own block: the K index only has to agree with X, whose
//     packed copy is read in that order.  Plain rows (kRaw) take block t per MFMA instead, as
//     the Z products here take their blocks: 4 x 4 transposes across the wave's 16-lane rows
//     (v_permlane32_swap, v_permlane16_swap) hand lane (c, g) its sub-block of every block;
//   * PCA: one extra MFMA per four blocks, K slots 8 t .. 8 t + 3 = block t's (c0, c0, c1, c1)
//     (lane (c, t) already holds that record) against (Z0 hi, Z0 lo, Z1 hi, Z1 lo);
//   * the waves of a work-group take the four-block groups round-robin, two groups of records
//     in flight per wave, and meet once in LDS (fixed order: deterministic).
// Two forms of input: the packed operands of the prefill GEMM (packed X + Zhl, written by the
// pack pass or by a producer kernel), or plain fp16 rows (kRaw), for which Z is computed on
// the matrix core too: the block's two basis vectors, split into fp16 hi + lo (22 bits of the
// largest element), are four rows of an A operand, so the product with the block's X lands, for
// every row of X, in the lane that feeds it to the PCA MFMA.
// Measured (kernel alone, packed, against k_gemm + k_reduce): 9728 x 2560 at 8 rows 9.9 against
// 17.7 us, 2560 x 9728 at 16 rows 11.6 against 22.5, 4096 x 2560 at 16 / 64 / 128 rows 5.6 / 9.1 /
// 14.5 against 11.9 / 15.1 / 18.7.  One launch from plain rows to fp16 outputs (kRaw): gate
// at 8 / 32 rows 11.6 / 13.8 us, where the pack pass, k_gemm, the sum and the conversion to
// fp16 took 24.3 / 24.2.
#include <algorithm>
#include <type_traits>

#include "sx8_buffer.h"
#include "sx8_device.h"
#include "sx8_gemm_ops.h"
#include "sx8_host.h"

namespace {


struct SmallMat {
    sx8::WeightSrc w;
    const uint32_t* Zhl;
    const float* basis;
    const float* scales;
    const uint16_t* bias;
    void* Y;
    int N;
    int nb;          // column tiles, ceil(N / (16 CF))
};
struct SmallGroup {
    SmallMat m[sx8::kMaxZSets];
    int n_mats;
    int NB;          // column tiles of the group
};

// A whole record as loaded (lane (c, t): column c, block t of a four-block group).
struct Rec {
    uint32_t lohi, hi16, cc, cf;
    uint4 h;      // hi nibbles of the four sub-blocks
    uint2 q;      // lo quads
};

struct RecSrc {
    sx8_rsrc a, b, c, d, e, f;   // v4.4: hdr, levels; split: dmin, dmax, config, coeff, hi, lo
};

template <bool kSplit, int HB>
__device__ __forceinline__ RecSrc rec_src(const sx8::WeightSrc& w, int64_t n_blk) {
    RecSrc r;
    if constexpr (kSplit) {
        r.a = make_rsrc(w.dmin, n_blk * 2);
        r.b = make_rsrc(w.dmax, n_blk * 2);
        r.c = make_rsrc(w.config, n_blk);
        r.d = make_rsrc(w.coeff, n_blk);
        r.e = make_rsrc(w.hi, n_blk * 16);
        r.f = make_rsrc(w.lo, n_blk * 8);
    } else {
        r.a = make_rsrc(w.hdr, n_blk * HB);
        r.b = make_rsrc(w.levels, n_blk * 24);
    }
    return r;
}

// bid past the last block reads zeros (range 0, levels 0: the weights are zero)
template <bool kSplit, int HB>
__device__ __forceinline__ void load_record(Rec& r, const RecSrc& s, uint32_t bid) {
    if constexpr (kSplit) {
        r.lohi = __builtin_amdgcn_raw_buffer_load_b16(s.a, bid * 2, 0, 0);
        r.hi16 = __builtin_amdgcn_raw_buffer_load_b16(s.b, bid * 2, 0, 0);
        r.cc = __builtin_amdgcn_raw_buffer_load_b8(s.c, bid, 0, 0);
        r.cf = __builtin_amdgcn_raw_buffer_load_b8(s.d, bid, 0, 0);
        r.h = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(s.e, bid * 16, 0, 0));
        r.q = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(s.f, bid * 8, 0, 0));
    } else {
        if constexpr (HB == 8) {
            const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(s.a, bid * 8, 0, 0));
            r.lohi = v.x;
            r.cc = v.y;
        } else {
            r.lohi = __builtin_amdgcn_raw_buffer_load_b32(s.a, bid * 6, 0, 0);
            r.cc = __builtin_amdgcn_raw_buffer_load_b16(s.a, bid * 6 + 4, 0, 0);
        }
        r.hi16 = r.cf = 0;
        r.h = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(s.b, bid * 24, 0, 0));
        r.q = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(s.b, bid * 24 + 16, 0, 0));
    }
}

typedef sx8_u32x4 u32x4;

// One column fragment's four blocks, ready to decode.  kT (transposed): element t is this
// lane's sub-block g of block t; otherwise element j is sub-block j of this lane's block.
struct Frag {
    uint32_t h[4], p[4], rlo[4], step[4];
    u32x4 coef;     // PCA operand: (c0, c0), (c1, c1) of this lane's record, two unused words
};

template <bool kSplit, bool kT>
__device__ __forceinline__ void frag_prep(Frag& f, const Rec& r) {
    const uint32_t hi16 = kSplit ? r.hi16 : r.lohi >> 16;
    const float lo = sx8_h2f(r.lohi), hi = sx8_h2f(hi16);
    const float d = hi - lo;
    const float q = d * 0.25f;
    const uint32_t cfg = r.cc & 0xFFu;
    // the sub-block ranges of sx8_gemm.hip's sub_range (rlo = lo + q k1[s], 2^24 step =
    // 2^24 0.015873 d 2^e[s], or the floor for d <= 0), the strategies moved to the bytes of a
    // selector
    uint32_t sel = (cfg << 6) | cfg;
    sel = ((sel << 12) | sel) & 0x03030303u;
    const uint32_t k1b = __builtin_amdgcn_perm(0u, 0x01030000u, sel);
    const bool pos = d > 0.f;
    const uint32_t eb = pos ? __builtin_amdgcn_perm(0u, 0x17161618u, sel) : 0u;   // 24 + e[s]
    const float m = pos ? d * 0.015873f : kStepFloor;
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
        f.rlo[sb] = __builtin_bit_cast(uint32_t, __builtin_fmaf(q, (float)((k1b >> (8 * sb)) & 0xFFu), lo));
        f.step[sb] = __builtin_bit_cast(uint32_t, __builtin_ldexpf(m, (int)((eb >> (8 * sb)) & 0xFFu)));
    }
    f.h[0] = r.h.x;
    f.h[1] = r.h.y;
    f.h[2] = r.h.z;
    f.h[3] = r.h.w;
    if constexpr (kT) {
        sx8_transpose4(f.h);
        sx8_transpose4(f.rlo);
        sx8_transpose4(f.step);
        // quads: words x (sub-blocks 0, 1) and y (2, 3); rows g < 2 need x, g >= 2 y, of every
        // block: one half swap, then each register copied across its row pair
        uint32_t a = r.q.x, b = r.q.y;
        sx8_swap32(a, b);
        f.p[0] = a;
        f.p[1] = a;
        sx8_swap16(f.p[0], f.p[1]);
        f.p[2] = b;
        f.p[3] = b;
        sx8_swap16(f.p[2], f.p[3]);
    } else {
        f.p[0] = f.p[1] = r.q.x;
        f.p[2] = f.p[3] = r.q.y;
    }
    const uint32_t cf = kSplit ? r.cf : r.cc >> 8;
    f.coef = u32x4{sx8_coeff_pair_f16(sx8_sext4(cf)), sx8_coeff_pair_f16(sx8_sext4(cf >> 4)), 0u, 0u};
}

// XCD-aware order (as sx8_gemm.hip): XCD b % 8 gets a contiguous run of column tiles, so
// neighbouring tiles share their header lines in one L2.
__device__ __forceinline__ int xcd_order_small(int b, int G) {
    const int x = b & 7;
    return (b >> 3) + x * (G >> 3) + min(x, G & 7);
}

constexpr uint32_t kOob = 0x80000000u;     // past every buffer (all below 2 GiB): reads zero

// v of lane 4 g + k of this lane's 16-lane row g (row_newbcast, one row at a time)
template <int k>
__device__ __forceinline__ uint32_t from_own_block(uint32_t v) {
    int r = __builtin_amdgcn_update_dpp(0, (int)v, 0x150 + k, 0x1, 0xF, false);
    r = __builtin_amdgcn_update_dpp(r, (int)v, 0x154 + k, 0x2, 0xF, false);
    r = __builtin_amdgcn_update_dpp(r, (int)v, 0x158 + k, 0x4, 0xF, false);
    return (uint32_t)__builtin_amdgcn_update_dpp(r, (int)v, 0x15C + k, 0x8, 0xF, false);
}

// max(|a|, |b|, |c|), NaN left out
__device__ __forceinline__ float abs_max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

constexpr int kMaxWaves = 8;

// Work-group: 64 S threads (S waves); 16 CF columns, all rows (M <= 16 MT).
// kOdd (raw): rows that do not all begin on 4 bytes.  A 16-byte load that is 2 bytes off splits into many
// (32 rows, 4096 columns: K = 4095 34.8 us, 4096 14.3), so these read whole words, one more than they need,
// and shift by half a word where the row begins in the middle of one: 16.9 us (16 rows 19.9 -> 11.7).
template <bool kSplit, int HB, bool kRaw, bool kOdd, int MT, int CF>
__global__ __launch_bounds__(64 * kMaxWaves) void k_gemm_small(const uint16_t* __restrict__ X, int M, int K,
                                                               int64_t ldx, int n_cb, const SmallGroup grp) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = (int)(blockDim.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    int nb = xcd_order_small((int)blockIdx.x, grp.NB);
    int mi = 0;
    while (mi + 1 < grp.n_mats && nb >= grp.m[mi].nb) nb -= grp.m[mi++].nb;
    const SmallMat& mat = grp.m[mi];
    const int N = mat.N;
    const int n0 = nb * 16 * CF;
    const int n_groups = (n_cb + 3) >> 2;

    const RecSrc ws = rec_src<kSplit, HB>(mat.w, (int64_t)N * n_cb);
    sx8_rsrc xs, zs, ss;
    // X's place in its first word, which lies in X's allocation (those begin on 256 bytes)
    const uint32_t x_off = kOdd ? (uint32_t)(reinterpret_cast<uintptr_t>(X) & 3) : 0u;
    if constexpr (kRaw) {
        xs = make_rsrc(kOdd ? reinterpret_cast<const void*>(reinterpret_cast<uintptr_t>(X) & ~(uintptr_t)3) : X,
                       ((int64_t)(M - 1) * ldx + K) * 2 + x_off);
        zs = make_rsrc(mat.basis, (int64_t)n_cb * 256);
        ss = make_rsrc(mat.scales, (int64_t)n_cb * 8);
    } else {
        xs = make_rsrc(X, (int64_t)((M + 31) / 32) * n_cb * 2048);
        zs = make_rsrc(mat.Zhl, (int64_t)M * n_cb * 8);
    }

    // per-lane offsets of group `wave`; one group step adds S of them
    uint32_t bid[CF];
#pragma unroll
    for (int cf = 0; cf < CF; ++cf)
        bid[cf] = (uint32_t)((4 * wave + g) * N + min(n0 + 16 * cf + c, N - 1));
    const uint32_t bid_step = (uint32_t)(4 * S) * (uint32_t)N;
    // X operand t: kRaw: row m, values 32 (kb0 + t) + 8 g ..; packed: chunk (row group, kb0 +
    // g), its 16-byte piece t (k-step t & 1, half t / 2) of row m
    uint32_t xo[MT], zo[MT], x_sh[kOdd ? MT : 1];
    auto x_imm = [](int t) { return kRaw ? 64u * t : 1024u * (t & 1) + 512u * (t >> 1); };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = 16 * mt + c;
        if constexpr (kRaw) {
            xo[mt] = m < M ? (uint32_t)(m * (int)ldx * 2 + 16 * g) + x_off + 256u * wave : kOob;
            if constexpr (kOdd) {
                x_sh[mt] = (xo[mt] & 2) * 8;
                xo[mt] &= ~3u;
            }
        } else {
            xo[mt] = (uint32_t)(((m >> 5) * n_cb + g) * 2048 + (m & 31) * 16) + 8192u * wave;
            if (m - c >= M) xo[mt] = kOob;
            zo[mt] = m < M ? (uint32_t)((m * n_cb + g) * 8) + 32u * wave : kOob;
        }
    }
    // the last element of a row, whose 4-byte word may straddle the end of X (a buffer load of it
    // reads zero): of an odd length, or in a row that begins in the middle of a word
    uint32_t x_last[kRaw ? MT : 1];
    if constexpr (kRaw) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = min(16 * mt + c, M - 1);
            const uint32_t at = (uint32_t)(m * (int)ldx + K - 1) * 2 + x_off;
            x_last[mt] = kOdd || (K & 1) ? __builtin_amdgcn_raw_buffer_load_b16(xs, at, 0, 0) : 0;
        }
    }

    Rec ra[CF], rb[CF];
    // X operands in flight: the whole next group, or two operands ahead past four row fragments
    constexpr int kRing = MT > 4 ? 2 : 4;
    u32x4 x[MT][kRing];
    uint32_t x_more[kOdd ? MT : 1][kRing];
    u32x4 z4[kRaw ? 2 : 1];
    uint2 zp[kRaw ? 1 : MT];
    float2 sc = make_float2(0.f, 0.f);
    auto load_recs = [&](Rec (&r)[CF]) __attribute__((always_inline)) {
#pragma unroll
        for (int cf = 0; cf < CF; ++cf) {
            load_record<kSplit, HB>(r[cf], ws, bid[cf]);
            bid[cf] += bid_step;
        }
    };
    auto load_x = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            x[mt][t % kRing] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, xo[mt] + x_imm(t), 0, 0));
            if constexpr (kOdd) x_more[mt][t % kRing] = __builtin_amdgcn_raw_buffer_load_b32(xs, xo[mt] + x_imm(t) + 16, 0, 0);
        }
    };
    auto next_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xo[mt] += (xo[mt] < kOob ? (kRaw ? 256u : 8192u) * S : 0u);
    };
    // basis operand of block t: A rows 4 t + {0, 1} = b0, b1 (fp16 hi), + {2, 3} the lo parts
    uint32_t zb = 0, sb_off = 0;
    if constexpr (kRaw) {
        zb = (uint32_t)((4 * wave + (c >> 2)) * 256 + (c & 1) * 128 + g * 32);
        sb_off = (uint32_t)((4 * wave + g) * 8);
    }
    auto load_z = [&]() __attribute__((always_inline)) {
        if constexpr (kRaw) {
            z4[0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(zs, zb, 0, 0));
            z4[1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(zs, zb + 16, 0, 0));
            sc = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(ss, sb_off, 0, 0));
            zb += 1024u * S;
            sb_off += 32u * S;
        } else {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                zp[mt] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(zs, zo[mt], 0, 0));
                zo[mt] += (zo[mt] < kOob ? 32u * S : 0u);
            }
        }
    };

    // Two fp16 parts hold 22 bits of a basis vector's largest element while that lies in [2^-3,
    // 2^15); unit vectors of 32 do (2^-2.5 at least).  z_far: the group in z4 has a vector outside
    // (uniform).  z_scale: each vector times a power of two that puts its largest element in [2^14,
    // 2^15), undone in its scale.  Scaling every group costs ~45 instructions, 2560 x 9728 at 2 rows
    // 14.0 -> 15.6 us; the test after the wait for z4 14.5, with the record arithmetic ahead of it to
    // hide its chain 14.1 (1024 x 2560 at 2 / 32 rows 5.58 / 9.10 -> 5.68 / 9.08).
    auto b_max = [&]() __attribute__((always_inline)) {
        float b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) b[i] = __builtin_bit_cast(float, (uint32_t)z4[kRaw ? i >> 2 : 0][i & 3]);
        return abs_max3(abs_max3(b[0], b[1], b[2]), abs_max3(b[3], b[4], b[5]), abs_max3(b[6], b[7], 0.f));
    };
    auto z_far = [&]() __attribute__((always_inline)) {
        const float mx = b_max();
        unsigned long long reach = __ballot(mx >= 0.125f);
        reach |= reach >> 32;
        reach |= reach >> 16;
        return (reach & 0xFFFF) != 0xFFFF || __ballot(mx >= 32768.f) != 0;
    };
    auto z_scale = [&]() __attribute__((always_inline)) {
        uint32_t a = __builtin_bit_cast(uint32_t, b_max()), b = a;      // (non-negative: ordered as integers)
        sx8_swap32(a, b);
        a = b = max(a, b);
        sx8_swap16(a, b);
        const uint32_t ex = min(max(max(a, b) >> 23, 15u), 254u);
        const float down = __builtin_bit_cast(float, (268u - ex) << 23);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            uint32_t w = z4[kRaw ? i >> 2 : 0][i & 3];
            z4[kRaw ? i >> 2 : 0][i & 3] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, w) * down);
        }
        // this lane's scales are of its own block g: lanes 4 g and 4 g + 1 hold its vectors' exponents
        sc.x *= __builtin_bit_cast(float, (from_own_block<0>(ex) - 14u) << 23);
        sc.y *= __builtin_bit_cast(float, (from_own_block<1>(ex) - 14u) << 23);
    };

    sx8_float4 acc[CF][MT];
#pragma unroll
    for (int cf = 0; cf < CF; ++cf)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[cf][mt] = sx8_float4{0.f, 0.f, 0.f, 0.f};

    const uint32_t sel_q = (g & 1) ? kQuadHi : kQuadLo;

    int gi = wave;
    load_recs(ra);
    load_z();
#pragma unroll
    for (int t = 0; t < kRing; ++t) load_x(t);
    if constexpr (kRing == 4) next_x();
    load_recs(rb);
    asm volatile("" ::: "memory");

    auto step = [&](Rec (&r)[CF]) __attribute__((always_inline)) {
        Frag fr[CF];
        if constexpr (kRaw) {
#pragma unroll
            for (int cf = 0; cf < CF; ++cf) frag_prep<kSplit, kRaw>(fr[cf], r[cf]);
            if (z_far()) z_scale();
        }
        // values past K (raw) or blocks past n_cb (packed) count as zero (kOdd: and the last value is
        // put in where its word straddles the end of X, also where no value is past K)
        const int kb0 = 4 * gi;
        const bool last = kb0 * 32 + 128 + (kOdd ? 1 : 0) > (kRaw ? K : n_cb * 32);
        if constexpr (kOdd) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        x[mt][t][i] = __builtin_amdgcn_alignbit(i < 3 ? x[mt][t][i < 3 ? i + 1 : 0] : x_more[mt][t],
                                                                x[mt][t][i], x_sh[mt]);
        }
        if constexpr (kRaw) {
            if (last) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int left = K - (kb0 + t) * 32 - 8 * g;     // values of this lane inside K
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint32_t w = x[mt][t][i];
                            const uint32_t end = kOdd && left == 2 * i + 2 ? (w & 0xFFFFu) | (x_last[mt] << 16) : w;
                            x[mt][t][i] = left >= 2 * i + 2 ? end : left == 2 * i + 1 ? x_last[mt] : 0u;
                        }
                }
            }
        } else if (last) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                if (kb0 + g >= n_cb) zp[mt] = make_uint2(0u, 0u);
        }
        // Z of the four blocks (raw): lane (row, t) gets block t's sums of its row
        u32x4 zop[MT];
        if constexpr (kRaw) {
            const float* b = reinterpret_cast<const float*>(z4);
            uint32_t bw[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const sx8_half2 h2 = {(_Float16)b[2 * i], (_Float16)b[2 * i + 1]};
                const sx8_half2 l2 = {(_Float16)(b[2 * i] - (float)h2.x), (_Float16)(b[2 * i + 1] - (float)h2.y)};
                bw[i] = __builtin_bit_cast(uint32_t, (c & 2) ? l2 : h2);
            }
            sx8_float4 zacc[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) zacc[mt] = sx8_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bool mine = (c >> 2) == t;
                const u32x4 a = {mine ? bw[0] : 0u, mine ? bw[1] : 0u, mine ? bw[2] : 0u, mine ? bw[3] : 0u};
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    zacc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(sx8_half8, a),
                                                                      __builtin_bit_cast(sx8_half8, x[mt][t]),
                                                                      zacc[mt], 0, 0, 0);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                float z0 = sc.x * (zacc[mt][0] + zacc[mt][2]);
                float z1 = sc.y * (zacc[mt][1] + zacc[mt][3]);
                asm volatile("" : "+v"(z0), "+v"(z1));     // rounded to float32 before the split
                zop[mt] = u32x4{sx8_split_hl(z0), sx8_split_hl(z1), 0u, 0u};
            }
        } else {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) zop[mt] = u32x4{zp[mt].x, zp[mt].y, 0u, 0u};
        }
        load_z();
#pragma unroll
        for (int cf = 0; cf < CF; ++cf) {
            if constexpr (!kRaw) frag_prep<kSplit, kRaw>(fr[cf], r[cf]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[cf][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(sx8_half8, fr[cf].coef),
                                                                     __builtin_bit_cast(sx8_half8, zop[mt]),
                                                                     acc[cf][mt], 0, 0, 0);
        }
        load_recs(r);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if constexpr (!kRaw) {
                if (last) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        if (kb0 + g >= n_cb) x[mt][t % kRing] = u32x4{0u, 0u, 0u, 0u};
                }
            }
#pragma unroll
            for (int cf = 0; cf < CF; ++cf) {
                uint32_t lv[4];
                sx8_dec_levels(fr[cf].h[t], fr[cf].p[t], kRaw ? sel_q : (t & 1) ? kQuadHi : kQuadLo, lv);
                const u32x4 a = sx8_dec_weights(lv, __builtin_bit_cast(float, fr[cf].rlo[t]),
                                                __builtin_bit_cast(float, fr[cf].step[t]));
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[cf][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(sx8_half8, a),
                                                                         __builtin_bit_cast(sx8_half8, x[mt][t % kRing]),
                                                                         acc[cf][mt], 0, 0, 0);
            }
            if constexpr (kRing == 2)
                if (t == 2) next_x();
            load_x((t + kRing) & 3);
        }
        if constexpr (kRing == 4) next_x();
        gi += S;
    };
    while (gi < n_groups) {
        step(ra);
        if (gi >= n_groups) break;
        step(rb);
    }

    // sum over the waves in wave order
    sx8_float4* red = reinterpret_cast<sx8_float4*>(smem);
    constexpr int kOut = CF * MT * 64;
#pragma unroll
    for (int cf = 0; cf < CF; ++cf)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red[wave * kOut + (cf * MT + mt) * 64 + lane] = acc[cf][mt];
    __syncthreads();
    for (int o = tid; o < kOut; o += 64 * S) {
        sx8_float4 v = red[o];
        for (int w = 1; w < S; ++w) v += red[w * kOut + o];
        const int l = o & 63, f = o >> 6;
        const int m = 16 * (f % MT) + (l & 15);
        const int n = n0 + 16 * (f / MT) + 4 * (l >> 4);
        if (m >= M || n >= N) continue;
        if constexpr (kRaw) {
            // fp16 output as y.half() + bias gives it: rounded, then the fp16 sum
            uint16_t* y = reinterpret_cast<uint16_t*>(mat.Y) + (int64_t)m * N + n;
            uint16_t h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float s = v[e];
                asm volatile("" : "+v"(s));
                _Float16 t = (_Float16)s;
                if (mat.bias && n + e < N) t = t + __builtin_bit_cast(_Float16, mat.bias[n + e]);
                h[e] = __builtin_bit_cast(uint16_t, t);
            }
            if (n + 3 < N && (reinterpret_cast<uintptr_t>(y) & 7) == 0) {
                *reinterpret_cast<uint2*>(y) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16),
                                                          (uint32_t)h[2] | ((uint32_t)h[3] << 16));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) y[e] = h[e];
            }
        } else {
            float* y = reinterpret_cast<float*>(mat.Y) + (int64_t)m * N + n;
            if (n + 3 < N && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
                *reinterpret_cast<sx8_float4*>(y) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) y[e] = v[e];
            }
        }
    }
}

// Column fragments per wave, waves per work-group and the kernel's estimated time.  A group
// of four blocks costs a SIMD ~0.38 us per column fragment (the decode) plus 0.245 us per
// further row fragment (X comes through the vector cache once per wave), on top of 3.3 us of
// launch, prologue and sum.  Fitted on packed calls, CF = 1: 1024 x 2560 at 16 / 64 / 128 rows 5.1
// / 8.65 / 13.8 us, 2560 x 9728 at 16 / 64 rows 11.3 / 23.7, 512 x 512 at 64 rows 4.5.  Eight row
// fragments in three rounds of work-groups take 3-4 us more than that (12288 x 512 at 128 rows 13.9
// us, the tiled kernel 12.8).  More column fragments only pay where they save a round of work-groups over the CUs: gate_proj (9728
// columns) at 32 rows 13.2 / 13.2 / 11.2 us with CF = 1 / 2 / 3 (608, 304, 203 tiles); with one
// packed row fragment, whose time is all decode, they never do.  Raw rows add the basis
// conversion and the Z products of every tile.
// Eight waves per work-group (two per SIMD) hide the loads where a CU has one work-group and
// the row fragments are few (down at 16 rows 11.6 against 14.3 us with four); else four, so
// that two or three work-groups share a CU (gate at 64 rows 17.5 against 20.7).
struct SmallPlan {
    int cf, S;
    double us;
};

// most column fragments a wave may take: what its registers hold past two row fragments
constexpr int max_cf(int64_t MT, bool raw) { return MT == 1 && !raw ? 1 : MT <= 2 ? 3 : MT <= 5 ? 2 : 1; }

SmallPlan plan_small(int64_t MT, int n_mats, const int64_t* Ns, int64_t n_groups, bool raw) {
    SmallPlan best{1, 8, 1e300};
    for (int cf = 1; cf <= max_cf(MT, raw); ++cf) {
        int64_t tiles = 0;
        for (int i = 0; i < n_mats; ++i) tiles += (Ns[i] + 16 * cf - 1) / (16 * cf);
        const double per = raw ? 0.1 + 0.53 * cf + 0.4 * (double)(MT - 1) : 0.38 * cf + 0.245 * (double)(MT - 1);
        const int64_t rounds = (tiles + 255) / 256;
        const double us = 3.3 + (double)rounds * (double)((n_groups + 3) / 4) * per + (MT == 8 && rounds > 2 ? 3.5 : 0.0);
        if (us < best.us) best = SmallPlan{cf, tiles <= 256 && MT <= 2 ? 8 : 4, us};
    }
    return best;
}

int64_t row_frags(int64_t M) {
    const int64_t MT = (M + 15) / 16;
    return MT == 7 ? 8 : MT;
}

template <bool kSplit, int HB, bool kRaw, bool kOdd, int MT, int CF>
void launch_one(int S, int64_t grid, const uint16_t* X, int64_t M, int64_t K, int64_t ldx, int64_t n_cb,
                const SmallGroup& g, hipStream_t st) {
    const size_t lds = (size_t)S * CF * MT * 1024;
    hipLaunchKernelGGL((k_gemm_small<kSplit, HB, kRaw, kOdd, MT, CF>), dim3((unsigned)grid), dim3(64 * S), lds, st, X,
                       (int)M, (int)K, ldx, (int)n_cb, g);
}

template <bool kSplit, int HB, bool kRaw, bool kOdd = false>
void launch_small(int64_t MT, const SmallPlan& p, int64_t grid, const uint16_t* X, int64_t M, int64_t K,
                  int64_t ldx, int64_t n_cb, const SmallGroup& g, hipStream_t st) {
    auto go = [&](auto mt) {
        constexpr int kMT = decltype(mt)::value;
        constexpr int kCF = max_cf(kMT, kRaw);
        if (kCF >= 3 && p.cf == 3) launch_one<kSplit, HB, kRaw, kOdd, kMT, kCF >= 3 ? 3 : 1>(p.S, grid, X, M, K, ldx, n_cb, g, st);
        else if (kCF >= 2 && p.cf == 2) launch_one<kSplit, HB, kRaw, kOdd, kMT, kCF >= 2 ? 2 : 1>(p.S, grid, X, M, K, ldx, n_cb, g, st);
        else launch_one<kSplit, HB, kRaw, kOdd, kMT, 1>(p.S, grid, X, M, K, ldx, n_cb, g, st);
    };
    if (MT == 1) go(std::integral_constant<int, 1>{});
    else if (kRaw || MT == 2) go(std::integral_constant<int, 2>{});
    if constexpr (!kRaw) {
        switch (MT) {
            case 1: case 2: break;
            case 3: go(std::integral_constant<int, 3>{}); break;
            case 4: go(std::integral_constant<int, 4>{}); break;
            case 5: go(std::integral_constant<int, 5>{}); break;
            case 6: go(std::integral_constant<int, 6>{}); break;
            default: go(std::integral_constant<int, 8>{}); break;
        }
    }
}

int64_t fill_group(SmallGroup& g, int n_mats, const int64_t* Ns, int cf) {
    g.n_mats = n_mats;
    int64_t NB = 0;
    for (int i = 0; i < n_mats; ++i) {
        g.m[i].N = (int)Ns[i];
        g.m[i].nb = (int)((Ns[i] + 16 * cf - 1) / (16 * cf));
        NB += g.m[i].nb;
    }
    g.NB = (int)NB;
    return NB;
}

}  // namespace

namespace sx8 {

double gemm_small_us(int64_t M, int n_mats, const int64_t* Ns, int64_t n_cb) {
    if (M > kSmallRows || n_cb > (1 << 16)) return 1e300;
    // record indices run up to three rounds of 8 waves x 4 blocks past the last block, in 32 bits
    for (int i = 0; i < n_mats; ++i)
        if (Ns[i] * 24 * (n_cb + 3 * 32 + 4) > 0xFFFFFFFF) return 1e300;
    return plan_small(row_frags(M), n_mats, Ns, (n_cb + 3) / 4, false).us;
}

int32_t gemm_small_packed(const char* what, bool split, int32_t hdr_bytes, const uint16_t* Xp, int64_t M,
                          int64_t n_cb, int n_mats, const WeightSrc* ws, const uint32_t* const* Zhl,
                          const int64_t* Ns, float* const* Ys, hipStream_t st) {
    const int64_t MT = row_frags(M);
    const SmallPlan p = plan_small(MT, n_mats, Ns, (n_cb + 3) / 4, false);
    SmallGroup g{};
    const int64_t NB = fill_group(g, n_mats, Ns, p.cf);
    for (int i = 0; i < n_mats; ++i) {
        g.m[i].w = ws[i];
        g.m[i].Zhl = Zhl[i];
        g.m[i].Y = Ys[i];
    }
    if (split) launch_small<true, 6, false>(MT, p, NB, Xp, M, n_cb * 32, 0, n_cb, g, st);
    else if (hdr_bytes == 8) launch_small<false, 8, false>(MT, p, NB, Xp, M, n_cb * 32, 0, n_cb, g, st);
    else launch_small<false, 6, false>(MT, p, NB, Xp, M, n_cb * 32, 0, n_cb, g, st);
    return check_launch(what);
}

int32_t gemm_small_raw(const char* what, int32_t hdr_bytes, const uint16_t* X, int64_t M, int64_t ldx, int64_t K,
                       int64_t n_cb, const WeightSrc& w, const float* basis, const float* scales,
                       const uint16_t* bias, int64_t N, uint16_t* Y, hipStream_t st) {
    const int64_t MT = row_frags(M);
    const SmallPlan p = plan_small(MT, 1, &N, (n_cb + 3) / 4, true);
    SmallGroup g{};
    const int64_t NB = fill_group(g, 1, &N, p.cf);
    g.m[0].w = w;
    g.m[0].basis = basis;
    g.m[0].scales = scales;
    g.m[0].bias = bias;
    g.m[0].Y = Y;
    // word loads where at least two rows begin off 4 bytes; one such row costs less than the extra words
    // (K = 4095, 4096 columns, 2 / 3 / 4 / 8 rows 9.0 / 9.4 / 10.2 / 13.0 us without them, 9.9 / 9.9 / 9.9 / 9.8 with)
    const int64_t off = !aligned(X, 4);
    const bool odd = ((ldx & 1) ? (M + off) / 2 : off * M) >= 2;
    if (hdr_bytes == 8 && odd) launch_small<false, 8, true, true>(MT, p, NB, X, M, K, ldx, n_cb, g, st);
    else if (hdr_bytes == 8) launch_small<false, 8, true>(MT, p, NB, X, M, K, ldx, n_cb, g, st);
    else if (odd) launch_small<false, 6, true, true>(MT, p, NB, X, M, K, ldx, n_cb, g, st);
    else launch_small<false, 6, true>(MT, p, NB, X, M, K, ldx, n_cb, g, st);
    return check_launch(what);
}

}  // namespace sx8

extern "C" int32_t sx8_linear_f16(const uint16_t* X, int64_t M, int64_t ldx, int64_t K, const uint8_t* hdr,
                                  const uint8_t* levels, int32_t hdr_bytes, const float* basis, const float* scales,
                                  const uint16_t* bias, int64_t N, int64_t n_cb, uint16_t* Y, void* stream) {
    using namespace sx8;
    const char* what = "sx8_linear_f16";
    if (!X || !hdr || !levels || !basis || !scales || !Y) return fail(SX8_ERR_INVALID, "%s: null pointer", what);
    if (hdr_bytes != 6 && hdr_bytes != 8)
        return fail(SX8_ERR_INVALID, "%s: hdr_bytes must be 6 or 8, got %d", what, hdr_bytes);
    if (!aligned(hdr, hdr_bytes == 8 ? 8 : 2) || !aligned(levels, 8) || !aligned(X, 2) || !aligned(Y, 2) ||
        !aligned(basis, M == 1 ? 4 : 16) || !aligned(scales, M == 1 ? 4 : 8) || !aligned(bias, 2))
        return fail(SX8_ERR_INVALID, "%s: misaligned pointer", what);
    if (M <= 0 || K <= 0 || N <= 0 || n_cb <= 0 || n_cb * 32 < K || (n_cb - 1) * 32 >= K || ldx < K || N > 0x7FFFFFFF)
        return fail(SX8_ERR_INVALID, "%s: bad shape M=%lld K=%lld ldx=%lld N=%lld n_cb=%lld", what, (long long)M,
                    (long long)K, (long long)ldx, (long long)N, (long long)n_cb);
    if (M == 1 && N <= 0x7FFFFFFF / 2 && n_cb <= 0x7FFFFFFF / 64)
        return gemv_linear(what, hdr_bytes, X, K, hdr, levels, basis, scales, bias, N, n_cb, Y, as_stream(stream));
    if (M > kLinearRows || M * ldx * 2 > 0x7FFFFFFF || N * n_cb * 24 > 0x7FFFFFFF || gemm_small_us(M, 1, &N, n_cb) >= 1e300)
        return fail(SX8_ERR_UNSUPPORTED, "%s: at most %lld rows and operands below 2 GiB", what, (long long)kLinearRows);
    WeightSrc w{};
    w.hdr = hdr;
    w.levels = levels;
    return gemm_small_raw(what, hdr_bytes, X, M, ldx, K, n_cb, w, basis, scales, bias, N, Y, as_stream(stream));
}
