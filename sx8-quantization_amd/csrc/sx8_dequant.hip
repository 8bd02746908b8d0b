// sx8_dequant.hip -- canonical (R64, bit-exact) dequantization kernels:
//   * k_dequant_wave, k_dequant_split: whole tensor from the pkl/container split arrays (n-major);
//     role of kernel_sx8_v43.decode_tensor_gpu_fast (scripts/kernel_sx8_v43.py:109-145).
//   * k_dequant_wave, k_gather_v44: selected rows from the kb-major v4.4 layout; role of the embedding
//     gather sx8_embed_v44 (cuda/sx8_embed_v44.cu:21-94) and, with identity ids, of a
//     whole-tensor dequant from the v4.4 layout.
//
// What bounds them: 30 B in and 64 B out per block, with the binary64 arithmetic (three fused
// multiply-adds and a conversion a weight) close behind.  A wave takes 16 K blocks of four rows
// at a time: lane (c, t) loads the whole record of (row t, block c), one load per field for 64
// records, and the records cross the wave's four 16-lane rows (v_permlane32_swap,
// v_permlane16_swap) so that lane (c, g) decodes sub-block g of block c for each of the four
// rows: its 8 + 8 basis values and scales stay in registers as binary64 for all the wave's
// rows, and every store instruction writes 1 KB of one output row.  One thread per (block,
// sub-block) issues four times the load instructions, re-reads and converts the basis for
// every 16 bytes of output: 9728 x 2560 20.9 us, here 17.8 (a 73 MB copy takes 14.2; with the
// decode replaced by plain moves the kernel takes 14.4).  It stays where it is the faster one
// (wave_wins).
#include <algorithm>

#include "sx8_device.h"
#include "sx8_host.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

// Store 8 fp16 values for columns [col, col+8) of an output row.  Vector store when
// the row pitch allows it, element stores (and the in_f cut) otherwise.
__device__ __forceinline__ void store8(uint16_t* __restrict__ row, int64_t col, int64_t in_f,
                                       bool vec_ok, const uint32_t w[4]) {
    if (vec_ok && col + 8 <= in_f) {
        *reinterpret_cast<uint4*>(row + col) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (col + e < in_f) row[col + e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
}

// basis (n_cb, 64) f32: b0 = [0, 32), b1 = [32, 64); load the sub-block's 8 + 8 values.
__device__ __forceinline__ void load_basis(const float* __restrict__ basis,
                                           const float* __restrict__ scales, int64_t kb, int sb,
                                           double b0[8], double b1[8], double& s0, double& s1) {
    const float4* p0 = reinterpret_cast<const float4*>(basis + kb * 64 + 8 * sb);
    const float4* p1 = reinterpret_cast<const float4*>(basis + kb * 64 + 32 + 8 * sb);
    const float4 a0 = p0[0], a1 = p0[1], c0 = p1[0], c1 = p1[1];
    b0[0] = a0.x; b0[1] = a0.y; b0[2] = a0.z; b0[3] = a0.w;
    b0[4] = a1.x; b0[5] = a1.y; b0[6] = a1.z; b0[7] = a1.w;
    b1[0] = c0.x; b1[1] = c0.y; b1[2] = c0.z; b1[3] = c0.w;
    b1[4] = c1.x; b1[5] = c1.y; b1[6] = c1.z; b1[7] = c1.w;
    const float2 sc = *reinterpret_cast<const float2*>(scales + kb * 2);
    s0 = sc.x;
    s1 = sc.y;
}

// A whole record: dmin | dmax << 16, config | coeff << 8, hi nibbles, lo quads.
struct Rec {
    uint32_t lohi, cc;
    uint32_t h[4];
    uint32_t qx, qy;
};

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

// Fields of (row, kb) from the n-major split arrays (block row n_cb + kb).
struct SplitSrc {
    const uint16_t* dmin;
    const uint16_t* dmax;
    const uint8_t* config;
    const uint8_t* coeff;
    const uint8_t* hi;
    const uint8_t* lo;
    int64_t n_cb;
    __device__ __forceinline__ void load(Rec& o, int64_t row, int kb) const {
        const int64_t bid = row * n_cb + kb;
        o.lohi = (uint32_t)dmin[bid] | ((uint32_t)dmax[bid] << 16);
        o.cc = (uint32_t)config[bid] | ((uint32_t)coeff[bid] << 8);
        const u32x4_a4 h = *reinterpret_cast<const u32x4_a4*>(hi + bid * 16);
        const u32x2_a2 q = *reinterpret_cast<const u32x2_a2*>(lo + bid * 8);
#pragma unroll
        for (int i = 0; i < 4; ++i) o.h[i] = h[i];
        o.qx = q[0];
        o.qy = q[1];
    }
};

// The same from the kb-major v4.4 layout (block kb N + row).
template <int HB>
struct V44Src {
    const uint8_t* hdr;
    const uint8_t* levels;
    int64_t N;
    __device__ __forceinline__ void load(Rec& o, int64_t row, int kb) const {
        const int64_t bid = kb * N + row;
        uint32_t d0, d1, cfg, cf;
        sx8_load_hdr<HB>(hdr, bid, d0, d1, cfg, cf);
        o.lohi = d0 | (d1 << 16);
        o.cc = cfg | (cf << 8);
        const u32x4_a4 h = *reinterpret_cast<const u32x4_a4*>(levels + bid * 24);
        const uint2 q = *reinterpret_cast<const uint2*>(levels + bid * 24 + 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) o.h[i] = h[i];
        o.qx = q.x;
        o.qy = q.y;
    }
};

// v in the lanes of 16-lane row i -> o[i] in every row (all four rows' values of a lane column)
__device__ __forceinline__ void gather_rows(uint32_t v, uint32_t (&o)[4]) {
    uint32_t a = v, b = v;
    sx8_swap32(a, b);            // a: rows 0, 1, 0, 1; b: rows 2, 3, 2, 3
    o[0] = o[1] = a;
    sx8_swap16(o[0], o[1]);
    o[2] = o[3] = b;
    sx8_swap16(o[2], o[3]);
}

// Output rows 4 quad + t (quad = this wave's) of T: row ids[.] of the weight, or row row0 + .
// without ids; rows outside [0, N) are skipped.  blockIdx.x: 16-block column group.
template <typename Src, bool kIds>
__global__ __launch_bounds__(kThreads) void k_dequant_wave(const Src src, const int64_t* __restrict__ ids,
                                                           const float* __restrict__ basis,
                                                           const float* __restrict__ scales, int64_t T, int64_t N,
                                                           int n_cb, int64_t in_f, uint16_t* __restrict__ out, int64_t row0) {
    const int lane = threadIdx.x & 63;
    const int c = lane & 15, g = lane >> 4;
    const int kb = (int)blockIdx.x * 16 + c;
    const int kbc = min(kb, n_cb - 1);
    const int64_t quad = (int64_t)blockIdx.y * kWaves + (threadIdx.x >> 6);
    if (quad * 4 >= T) return;
    // this lane's record: row g of the quad (-1: none)
    const int64_t t = quad * 4 + g;
    int64_t row = t < T ? (kIds ? ids[t] : row0 + t) : -1;
    if (row >= N) row = -1;
    Rec r;
    src.load(r, row < 0 ? 0 : row, kbc);
    double b0[8], b1[8], s0, s1;
    load_basis(basis, scales, kbc, g, b0, b1, s0, s1);
    const unsigned long long ok = __ballot(row >= 0);       // lane 16 i holds row i's
    uint32_t lohi[4], cc[4], p[4];
    gather_rows(r.lohi, lohi);
    gather_rows(r.cc, cc);
    sx8_transpose4(r.h);
    uint32_t a = r.qx, b = r.qy;
    sx8_swap32(a, b);
    p[0] = p[1] = a;
    sx8_swap16(p[0], p[1]);
    p[2] = p[3] = b;
    sx8_swap16(p[2], p[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (!((ok >> (16 * i)) & 1)) continue;          // uniform
        uint32_t w[4];
        sx8_r64_subblock(sx8_h2f(lohi[i]), sx8_h2f(lohi[i] >> 16), cc[i] & 0xFFu, cc[i] >> 8, g, r.h[i],
                         (g & 1) ? p[i] >> 16 : p[i] & 0xFFFFu, b0, b1, s0, s1, w);
        uint16_t* o = out + (quad * 4 + i) * in_f;
        const int64_t col = (int64_t)kb * 32 + 8 * g;
        if (col < in_f) *reinterpret_cast<uint4*>(o + col) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// Whether the wave kernel is the faster one.  A wave's four rows are a chain that few waves do not hide, and
// the lanes past n_cb of the last 16-block group idle.  us, one thread per (block, sub-block) / wave kernel:
//   any rows, output rows off 16 bytes (element stores, which its lane order scatters): 9728 x 2557 38.5 / 50.0
//   rows in order, split arrays: 4096 x 1664 (81% of the lanes used) 7.6 / 8.7; 3300 x 2560 8.9 / 9.4; 6500 x 1472
//     9.7 / 9.5; 9728 x 2560 20.6 / 17.9
//   rows in order, v4.4: 4096 x 1664 9.3 / 9.0; 9728 x 2560 30.3 / 18.2
//   rows by ids, v4.4 (each record a memory access of its own either way): 4096 x 2560 18.7 / 18.9, 8192 x 3584
//     47.3 / 50.6; ahead only for whole sets of four column groups (4096 x 2048 15.4 / 14.9) or many waves (16384
//     x 3072 83.1 / 80.0)
enum class Rows { kSplit, kV44, kV44Ids };
bool wave_wins(Rows r, int64_t T, int64_t n_cb, bool vec_ok) {
    const int64_t quads = (T + 3) / 4, cols = (n_cb + 15) / 16;
    if (!vec_ok || cols > 0x7FFFFFFF / 16) return false;
    switch (r) {
        case Rows::kSplit: return n_cb * 8 >= cols * 16 * 7 && quads * n_cb >= 16 * 4600;
        case Rows::kV44: return n_cb * 5 >= cols * 16 * 4 && quads * cols >= 4096;
        default: return (n_cb % 64 == 0 && quads * cols >= 4096) || quads * n_cb >= 16 * 23000;
    }
}

template <typename Src>
void launch_wave(const Src& src, const int64_t* ids, const float* basis, const float* scales, int64_t T, int64_t N,
                 int64_t n_cb, int64_t in_f, uint16_t* out, hipStream_t st) {
    const int64_t cols = (n_cb + 15) / 16;
    // blockIdx.y takes at most 65535 work-groups: more rows go in several launches
    constexpr int64_t kRows = (int64_t)65535 * kWaves * 4;
    for (int64_t t0 = 0; t0 < T; t0 += kRows) {
        const int64_t Tc = std::min(kRows, T - t0);
        const dim3 grid((unsigned)cols, (unsigned)((Tc + kWaves * 4 - 1) / (kWaves * 4)));
        if (ids)
            hipLaunchKernelGGL((k_dequant_wave<Src, true>), grid, dim3(kThreads), 0, st, src, ids + t0, basis, scales, Tc,
                               N, (int)n_cb, in_f, out + t0 * in_f, t0);
        else
            hipLaunchKernelGGL((k_dequant_wave<Src, false>), grid, dim3(kThreads), 0, st, src, nullptr, basis, scales, Tc,
                               N, (int)n_cb, in_f, out + t0 * in_f, t0);
    }
}

__global__ __launch_bounds__(kThreads) void k_dequant_split(
    const uint16_t* __restrict__ dmin, const uint16_t* __restrict__ dmax,
    const uint8_t* __restrict__ config, const uint8_t* __restrict__ coeff,
    const uint8_t* __restrict__ hi, const uint8_t* __restrict__ lo,
    const float* __restrict__ basis, const float* __restrict__ scales, int64_t n_blocks,
    int64_t n_cb, int64_t in_f, bool vec_ok, uint16_t* __restrict__ out) {
    const int64_t gid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t bid = gid >> 2;
    const int sb = (int)(gid & 3);
    if (bid >= n_blocks) return;
    const int64_t n = bid / n_cb;
    const int64_t kb = bid - n * n_cb;
    double b0[8], b1[8], s0, s1;
    load_basis(basis, scales, kb, sb, b0, b1, s0, s1);
    const uint32_t H = *reinterpret_cast<const uint32_t*>(hi + bid * 16 + 4 * sb);
    const uint32_t P16 = *reinterpret_cast<const uint16_t*>(lo + bid * 8 + 2 * sb);
    uint32_t w[4];
    sx8_r64_subblock(sx8_h2f(dmin[bid]), sx8_h2f(dmax[bid]), config[bid], coeff[bid], sb, H, P16,
                     b0, b1, s0, s1, w);
    store8(out + n * in_f, kb * 32 + 8 * sb, in_f, vec_ok, w);
}

// ids == nullptr: row t of the output is row t of W.  Rows outside [0, N) are skipped.
template <int HB>
__global__ __launch_bounds__(kThreads) void k_gather_v44(
    const int64_t* __restrict__ ids, int64_t T, const uint8_t* __restrict__ hdr,
    const uint8_t* __restrict__ levels, const float* __restrict__ basis,
    const float* __restrict__ scales, int64_t K, int64_t N, int64_t n_cb, bool vec_ok,
    uint16_t* __restrict__ out) {
    const int64_t gid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t per_row = n_cb * 4;
    const int64_t t = gid / per_row;
    if (t >= T) return;
    const int64_t r = gid - t * per_row;
    const int64_t kb = r >> 2;
    const int sb = (int)(r & 3);
    const int64_t row = ids ? ids[t] : t;
    if (row < 0 || row >= N) return;
    const int64_t bid = kb * N + row;
    uint32_t d0, d1, cfg, cf;
    sx8_load_hdr<HB>(hdr, bid, d0, d1, cfg, cf);
    const uint8_t* lv = levels + bid * 24;
    const uint32_t H = *reinterpret_cast<const uint32_t*>(lv + 4 * sb);
    const uint32_t Pw = *reinterpret_cast<const uint32_t*>(lv + 16 + 4 * (sb >> 1));
    const uint32_t P16 = (sb & 1) ? (Pw >> 16) : (Pw & 0xFFFFu);
    double b0[8], b1[8], s0, s1;
    load_basis(basis, scales, kb, sb, b0, b1, s0, s1);
    uint32_t w[4];
    sx8_r64_subblock(sx8_h2f(d0), sx8_h2f(d1), cfg, cf, sb, H, P16, b0, b1, s0, s1, w);
    store8(out + t * K, kb * 32 + 8 * sb, K, vec_ok, w);
}

}  // namespace

extern "C" int32_t sx8_dequant_f16(const uint16_t* dmin, const uint16_t* dmax,
                                   const uint8_t* config, const uint8_t* coeff,
                                   const uint8_t* levels_hi, const uint8_t* levels_lo,
                                   const float* basis, const float* scales, int64_t out_f,
                                   int64_t in_f, int64_t n_cb, uint16_t* out, void* stream) {
    using namespace sx8;
    if (!dmin || !dmax || !config || !coeff || !levels_hi || !levels_lo || !basis || !scales || !out)
        return fail(SX8_ERR_INVALID, "sx8_dequant_f16: null pointer argument");
    if (out_f <= 0 || in_f <= 0 || n_cb <= 0 || n_cb * 32 < in_f || (n_cb - 1) * 32 >= in_f)
        return fail(SX8_ERR_INVALID, "sx8_dequant_f16: bad shape out_f=%lld in_f=%lld n_cb=%lld",
                    (long long)out_f, (long long)in_f, (long long)n_cb);
    if (!aligned(levels_hi, 4) || !aligned(levels_lo, 2) || !aligned(basis, 16) ||
        !aligned(scales, 8) || !aligned(out, 2))
        return fail(SX8_ERR_INVALID, "sx8_dequant_f16: misaligned pointer");
    const int64_t n_blocks = out_f * n_cb;
    const bool vec_ok = aligned(out, 16) && (in_f % 8 == 0);
    if (wave_wins(Rows::kSplit, out_f, n_cb, vec_ok)) {
        launch_wave(SplitSrc{dmin, dmax, config, coeff, levels_hi, levels_lo, n_cb}, nullptr, basis, scales, out_f, out_f,
                    n_cb, in_f, out, as_stream(stream));
        return check_launch("sx8_dequant_f16");
    }
    const int64_t threads = n_blocks * 4;
    const int64_t grid = (threads + kThreads - 1) / kThreads;
    if (grid > 0x7FFFFFFF) return fail(SX8_ERR_UNSUPPORTED, "sx8_dequant_f16: tensor too large");
    hipLaunchKernelGGL(k_dequant_split, dim3((unsigned)grid), dim3(kThreads), 0, as_stream(stream),
                       dmin, dmax, config, coeff, levels_hi, levels_lo, basis, scales, n_blocks,
                       n_cb, in_f, vec_ok, out);
    return check_launch("sx8_dequant_f16");
}

extern "C" int32_t sx8_embed_gather(const int64_t* ids, int64_t T, const uint8_t* hdr,
                                    const uint8_t* levels, int32_t hdr_bytes,
                                    const float* basis, const float* scales, int64_t K,
                                    int64_t N, int64_t n_cb, uint16_t* out, void* stream) {
    using namespace sx8;
    if (!hdr || !levels || !basis || !scales || !out)
        return fail(SX8_ERR_INVALID, "sx8_embed_gather: null pointer argument");
    if (hdr_bytes != 6 && hdr_bytes != 8)
        return fail(SX8_ERR_INVALID, "sx8_embed_gather: hdr_bytes must be 6 or 8, got %d", hdr_bytes);
    if (!ids) T = N;
    if (T < 0 || K <= 0 || N <= 0 || n_cb <= 0 || n_cb * 32 < K || (n_cb - 1) * 32 >= K)
        return fail(SX8_ERR_INVALID, "sx8_embed_gather: bad shape T=%lld K=%lld N=%lld n_cb=%lld",
                    (long long)T, (long long)K, (long long)N, (long long)n_cb);
    if (!aligned(hdr, hdr_bytes == 8 ? 8 : 2) || !aligned(levels, 8) || !aligned(basis, 16) ||
        !aligned(scales, 8) || !aligned(out, 2) || (ids && !aligned(ids, 8)))
        return fail(SX8_ERR_INVALID, "sx8_embed_gather: misaligned pointer");
    if (T == 0) return ok();
    const bool vec_ok = aligned(out, 16) && (K % 8 == 0);
    const hipStream_t st = as_stream(stream);
    if (wave_wins(ids ? Rows::kV44Ids : Rows::kV44, T, n_cb, vec_ok)) {
        if (hdr_bytes == 8) launch_wave(V44Src<8>{hdr, levels, N}, ids, basis, scales, T, N, n_cb, K, out, st);
        else launch_wave(V44Src<6>{hdr, levels, N}, ids, basis, scales, T, N, n_cb, K, out, st);
        return check_launch("sx8_embed_gather");
    }
    const int64_t threads = T * n_cb * 4;
    const int64_t grid = (threads + kThreads - 1) / kThreads;
    if (grid > 0x7FFFFFFF) return fail(SX8_ERR_UNSUPPORTED, "sx8_embed_gather: too many rows");
    if (hdr_bytes == 8)
        hipLaunchKernelGGL(k_gather_v44<8>, dim3((unsigned)grid), dim3(kThreads), 0,
                           as_stream(stream), ids, T, hdr, levels, basis, scales, K, N, n_cb,
                           vec_ok, out);
    else
        hipLaunchKernelGGL(k_gather_v44<6>, dim3((unsigned)grid), dim3(kThreads), 0,
                           as_stream(stream), ids, T, hdr, levels, basis, scales, K, N, n_cb,
                           vec_ok, out);
    return check_launch("sx8_embed_gather");
}
