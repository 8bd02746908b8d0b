// sx8_quant.hip -- the deterministic half of the S-X8 v4.3 quantizer on the GPU: the V6
// encode of every 32-weight block (dmin, dmax, per-sub-block range strategy, 6-bit
// levels) and the level packing, written straight into the pkl / container split arrays.
//
// Role of v6_encode_6bit_gpu and pack_levels_6bit
// (scripts/quantize_qwen35_4b_sx8_v43_gpu.py:22-47, :148-167).  The PCA half (pca_correct_gpu,
// :75-142: per K block the two leading right singular vectors of the residuals, the
// coefficients and their scales) follows below, sx8_quant_pca.
//
// Arithmetic (binary32, every operation rounded, no contraction), per block:
//   dmin, dmax = min, max of the 32 weights; d = max(dmax - dmin, 1e-10); q = d / 4;
//   candidates (lo, hi) = (dmin, dmax), (dmin, dmin + q), (dmax - q, dmax),
//   (dmin + q, dmax - q); per 8-weight sub-block and candidate: step = max((hi - lo) / 63,
//   1e-10), lv = clamp(rint((x - lo) / step), 0, 63), rec = lo + step * lv, mse = (sum of
//   the eight (x - rec)^2 left to right) / 8; the first candidate with the strictly lowest
//   mse wins.  config = s0 | s1 << 2 | s2 << 4 | s3 << 6.
// Packing: qh[t >> 1] holds (lv >> 2) of weight t at bits 4 (t & 1); ql[t >> 2] holds
// (lv & 3) at bits 2 (3 - (t & 3)).
//
// One thread per block, n-major (bid = n * n_cb + kb): a wave reads 64 consecutive
// 64-byte row segments.  Columns past in_f are zero (the reference pads W with zeros).
#include "sx8_device.h"
#include "sx8_host.h"

namespace {

constexpr int kThreads = 256;

__global__ __launch_bounds__(kThreads) void k_v6_encode(
    const uint16_t* __restrict__ W, int64_t out_f, int64_t in_f, int64_t ld, int64_t n_cb,
    uint8_t* __restrict__ levels, uint16_t* __restrict__ dmin_out, uint16_t* __restrict__ dmax_out,
    uint8_t* __restrict__ config_out, uint8_t* __restrict__ hi_out, uint8_t* __restrict__ lo_out, bool vec_out) {
#pragma clang fp contract(off)
    const int64_t bid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (bid >= out_f * n_cb) return;
    const int64_t n = bid / n_cb;
    const int64_t kb = bid - n * n_cb;
    const uint16_t* row = W + n * ld + kb * 32;
    float x[32];
    const bool full = (kb + 1) * 32 <= in_f && (reinterpret_cast<uintptr_t>(row) & 15) == 0;
    if (full) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const uint4 v = reinterpret_cast<const uint4*>(row)[q4];
            const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) x[8 * q4 + i] = sx8_h2f(w4[i >> 1] >> (16 * (i & 1)));
        }
    } else {
#pragma unroll
        for (int t = 0; t < 32; ++t) x[t] = kb * 32 + t < in_f ? sx8_h2f(row[t]) : 0.f;
    }
    float mn = x[0], mx = x[0];
#pragma unroll
    for (int t = 1; t < 32; ++t) {
        mn = x[t] < mn ? x[t] : mn;
        mx = x[t] > mx ? x[t] : mx;
    }
    float d = mx - mn;
    d = d > 1e-10f ? d : 1e-10f;
    const float q = d / 4.0f;
    const float lo_c[4] = {mn, mn, mx - q, mn + q};
    const float hi_c[4] = {mx, mn + q, mx, mx - q};
    uint32_t cfg = 0;
    uint8_t lv_best[32];
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
        float best = __builtin_inff();
        int s_best = 0;
        uint8_t lvb[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float step = (hi_c[c] - lo_c[c]) / 63.0f;
            step = step > 1e-10f ? step : 1e-10f;
            uint8_t lv[8];
            float acc = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float r = __builtin_rintf((x[8 * sb + i] - lo_c[c]) / step);
                r = r < 0.f ? 0.f : (r > 63.f ? 63.f : r);
                lv[i] = (uint8_t)(int)r;
                const float rec = lo_c[c] + step * r;
                const float e = x[8 * sb + i] - rec;
                acc = i == 0 ? e * e : acc + e * e;
            }
            const float mse = acc / 8.0f;
            if (mse < best) {
                best = mse;
                s_best = c;
#pragma unroll
                for (int i = 0; i < 8; ++i) lvb[i] = lv[i];
            }
        }
        cfg |= (uint32_t)s_best << (2 * sb);
#pragma unroll
        for (int i = 0; i < 8; ++i) lv_best[8 * sb + i] = lvb[i];
    }
    dmin_out[bid] = __builtin_bit_cast(uint16_t, (_Float16)mn);
    dmax_out[bid] = __builtin_bit_cast(uint16_t, (_Float16)mx);
    config_out[bid] = (uint8_t)cfg;
    uint32_t h[4] = {0, 0, 0, 0}, l[2] = {0, 0};
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        h[t >> 3] |= (uint32_t)(lv_best[t] >> 2) << (4 * (t & 7));
        l[t >> 4] |= (uint32_t)(lv_best[t] & 3) << (8 * ((t >> 2) & 3) + 2 * (3 - (t & 3)));
    }
    uint8_t* ho = hi_out + bid * 16;
    uint8_t* lo = lo_out + bid * 8;
    if (vec_out) {
        *reinterpret_cast<uint4*>(ho) = make_uint4(h[0], h[1], h[2], h[3]);
        *reinterpret_cast<uint2*>(lo) = make_uint2(l[0], l[1]);
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) ho[k] = (uint8_t)(h[k >> 2] >> (8 * (k & 3)));
#pragma unroll
        for (int k = 0; k < 8; ++k) lo[k] = (uint8_t)(l[k >> 2] >> (8 * (k & 3)));
    }
    if (levels) {
        uint8_t* lvo = levels + bid * 32;
        uint32_t w[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            w[t] = (uint32_t)lv_best[4 * t] | ((uint32_t)lv_best[4 * t + 1] << 8) |
                   ((uint32_t)lv_best[4 * t + 2] << 16) | ((uint32_t)lv_best[4 * t + 3] << 24);
        if (vec_out) {
            reinterpret_cast<uint4*>(lvo)[0] = make_uint4(w[0], w[1], w[2], w[3]);
            reinterpret_cast<uint4*>(lvo)[1] = make_uint4(w[4], w[5], w[6], w[7]);
        } else {
#pragma unroll
            for (int t = 0; t < 32; ++t) lvo[t] = lv_best[t];
        }
    }
}

// ---------------------------------------------------------------- PCA of the residuals
// Six kernels over a tensor of n_rows x n_cb blocks (bid = row * n_cb + kb):
//   k_pca_err     residuals e = x - (lo + step lv) in float32 (every operation rounded, the
//                 steps as products with fp32(1 / 63)), stored K block by K block
//   k_pca_gram    partial Gram matrices E^T E of row ranges, float64 on the matrix core
//   k_pca_eig     their sum's two leading eigenvectors by repeated squaring on the matrix core
//   k_pca_coeff   c = basis . e (float64 sums of the float32 values, rounded to float32)
//   k_pca_scale   the lower median of |c| by radix selection; scale = max(median / 3, 1e-10)
//   k_pca_byte    c / scale rounded to signed 4 bits
// The eigenproblems bounded this: a few hundred 32 x 32 matrices took a library's batched solver
// 13.3 of the 14.7 ms of a 2560 x 4096 tensor (its tridiagonalisation runs column by column,
// ~430 us a launch) and the median 60 us.  Measured here on that tensor (128 K blocks): V6 encode
// 36 us (byte stores: 38), residuals 14.5, Gram 14, eigenvectors 33, coefficients 8.4, medians
// 6.6, bytes 3.5; the rest of a call's 0.55 ms is the copy of 9.8 MB to host memory.

constexpr int kPcaSplits = 8;        // row ranges of the Gram sums
constexpr float kInv63 = 1.0f / 63.0f;

// One thread per (block, sub-block): 8 residuals, contiguous 32-byte stores.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_pca_err(const T* __restrict__ blocks,
                                                      const uint8_t* __restrict__ levels,
                                                      const T* __restrict__ dmin, const T* __restrict__ dmax,
                                                      const uint8_t* __restrict__ config, int64_t n_rows,
                                                      int64_t n_cb, float* __restrict__ err) {
#pragma clang fp contract(off)
    const int64_t gid = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t bid = gid >> 2;
    const int sb = (int)(gid & 3);
    if (bid >= n_rows * n_cb) return;
    const int64_t row = bid / n_cb;
    const int64_t kb = bid - row * n_cb;
    const float mn = (float)dmin[bid], mx = (float)dmax[bid];
    float d = mx - mn;
    d = d < 1e-10f ? 1e-10f : d;                     // (NaN stays, as torch.clamp leaves it)
    const float q = d / 4.0f;
    const int s = (config[bid] >> (2 * sb)) & 3;
    float w = d - 2.0f * q;
    w = w < 1e-10f ? 1e-10f : w;
    const float lo = s == 2 ? mx - q : s == 3 ? mn + q : mn;
    const float step = (s == 0 ? d : s == 3 ? w : q) * kInv63;
    const T* x = blocks + bid * 32 + 8 * sb;
    const uint2 lv = *reinterpret_cast<const uint2*>(levels + bid * 32 + 8 * sb);
    float e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float l = (float)(((i < 4 ? lv.x : lv.y) >> (8 * (i & 3))) & 0xFFu);
        const float r = lo + step * l;
        e[i] = (float)x[i] - r;
    }
    float4* o = reinterpret_cast<float4*>(err + (kb * n_rows + row) * 32 + 8 * sb);
    o[0] = make_float4(e[0], e[1], e[2], e[3]);
    o[1] = make_float4(e[4], e[5], e[6], e[7]);
}

typedef double sx8_double4 __attribute__((ext_vector_type(4)));

// Work-group (split, kb): its rows' Gram matrix as three 16 x 16 tiles (00, 01, 11) of
// v_mfma_f64_16x16x4: lane l supplies e[row l / 16][l % 16] of four rows, so both operands
// of a tile are the same loads (products of float32 values are exact in float64).
__global__ __launch_bounds__(256) void k_pca_gram(const float* __restrict__ err, int n_rows, int rows_per,
                                                  double* __restrict__ part) {
    const int kb = blockIdx.x, split = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r0 = split * rows_per, r1 = min(r0 + rows_per, n_rows);
    const float* e = err + (int64_t)kb * n_rows * 32;
    sx8_double4 acc[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) acc[t] = sx8_double4{0.0, 0.0, 0.0, 0.0};
    for (int r = r0 + wave * 4; r < r1; r += 16 * 4) {
        float x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = r + 16 * u + (lane >> 4);
            const float* p = e + (int64_t)min(row, n_rows - 1) * 32 + (lane & 15);
            x[u] = p[0];
            y[u] = p[16];
            if (row >= r1) x[u] = y[u] = 0.f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double a = x[u], b = y[u];
            acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, a, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, b, acc[2], 0, 0, 0);
        }
    }
    __shared__ sx8_double4 red[4][3][64];
#pragma unroll
    for (int t = 0; t < 3; ++t) red[wave][t][lane] = acc[t];
    __syncthreads();
    if (threadIdx.x < 192) {
        const int t = threadIdx.x / 64, l = threadIdx.x & 63;
        const sx8_double4 v = ((red[0][t][l] + red[1][t][l]) + red[2][t][l]) + red[3][t][l];
        // element i of lane l: row l / 16 + 4 i, column l % 16
        double* o = part + (((int64_t)split * gridDim.x + kb) * 3 + t) * 256 + (l & 15);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[((l >> 4) + 4 * i) * 16] = v[i];
    }
}

// One work-group of three waves per K block: the two leading eigenvectors of the 32 x 32 Gram
// matrix by repeated squaring in float64.  B^(2^k) of a positive semi-definite B tends to the
// projector on its largest eigenvalue, whose longest column is the vector; the second vector is
// the same of the deflated matrix A - v w^T - w v^T + (v.w) v v^T, w = A v.  A squaring is one
// 16 x 16 tile a wave (tiles 00, 01, 11 of a symmetric result; 8 f64 MFMAs whose two operands
// are both rows of B), with one barrier: the result goes to the other of two buffers, scaled by
// a power of two that the trace of B gives.  tr(B)^2 - tr(B^2) is twice the share of the other
// eigenvalues to first order, so once it is below 1e-8 one more squaring leaves 1e-16; the
// rounding errors shrink with the powers like the gap grows, so the vectors are good to a few
// 2^-53 / (relative gap).  Gaps below 1e-12 end after 45 squarings with a vector of the two's
// plane.  Residuals of trained or random weights take 9 to 17 squarings a vector, each ~0.4 us
// of LDS, MFMA and barrier latency: 33 us for the 128 K blocks of a 2560 x 4096 tensor, where
// cyclic Jacobi rotations (some 8 sweeps of 31 dependent rounds) took 157 and were good to
// 1e-13 / gap.
constexpr int kEigThreads = 192;
constexpr int kEigLd = 36;           // doubles: the operand reads spread over all banks
constexpr int kEigSquarings = 45;

struct EigSmem {
    double A[32 * kEigLd];
    __attribute__((aligned(16))) double B[2][32 * kEigLd], dg[2][32], v[2][32], w[32];
};

__device__ __forceinline__ double eig_sum(const double* d) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 32; ++i) s[i & 3] += d[i];
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// index of the largest of f(d[0]) .. f(d[31]), the first of equals
template <typename F>
__device__ __forceinline__ int eig_argmax(const double* d, F f) {
    int j = 0;
    double best = f(d[0]);
#pragma unroll
    for (int i = 1; i < 32; ++i) {
        const double x = f(d[i]);
        if (x > best) {
            best = x;
            j = i;
        }
    }
    return j;
}

// The leading vector of B[0] (positive trace, diagonal in dg[0], both behind a barrier), made
// orthogonal to v[0] if second, into v[second].
__device__ __forceinline__ void eig_lead(EigSmem& sm, int second) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ra = wave == 2 ? 16 : 0, rb = wave == 0 ? 0 : 16;
    const int row = lane >> 4, col = lane & 15;
    int cur = 0;
    double prev = 0.0;
    bool last = false;
    for (int k = 0; k < kEigSquarings && !last; ++k) {       // the same for every thread
        const double* a = sm.B[cur] + (ra + col) * kEigLd + row;
        const double* b = sm.B[cur] + (rb + col) * kEigLd + row;
        sx8_double4 acc[2];
        acc[0] = acc[1] = sx8_double4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 8; ++s)
            acc[s & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[4 * s], b[4 * s], acc[s & 1], 0, 0, 0);
        const double t = eig_sum(sm.dg[cur]);
        last = k > 0 && prev * prev - t <= 1e-8 * (prev * prev);
        const int ex = __builtin_amdgcn_frexp_exp(t);
        prev = __builtin_amdgcn_ldexp(t, -ex);
        double* o = sm.B[cur ^ 1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double d = __builtin_amdgcn_ldexp(acc[0][i] + acc[1][i], -2 * ex);
            const int r = ra + row + 4 * i, c = rb + col;
            o[r * kEigLd + c] = d;
            if (wave == 1) o[c * kEigLd + r] = d;
            else if (r == c) sm.dg[cur ^ 1][r] = d;
        }
        __syncthreads();
        cur ^= 1;
    }
    if (wave == 0) {
        const int j = eig_argmax(sm.dg[cur], [](double d) { return d; });
        double* v = sm.v[second];
        const int i = lane & 31;
        double x = sm.B[cur][j * kEigLd + i];
        auto unit = [&]() {                                   // v = x / |x|, in every lane's x
            if (lane < 32) sm.w[i] = x * x;
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            x /= sqrt(eig_sum(sm.w));
        };
        unit();
        if (second) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            if (lane < 32) sm.w[i] = x * sm.v[0][i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            x -= eig_sum(sm.w) * sm.v[0][i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            unit();
        }
        if (lane < 32) v[i] = x;
    }
    __syncthreads();
}

__global__ __launch_bounds__(kEigThreads) void k_pca_eig(const double* __restrict__ part, int n_splits, int n_cb,
                                                         float* __restrict__ data) {
    __shared__ EigSmem sm;
    const int kb = blockIdx.x, tid = threadIdx.x;
#pragma unroll
    for (int i = tid; i < 768; i += kEigThreads) {
        const int t = i >> 8, r = (i >> 4) & 15, c = i & 15;
        double v = 0.0;
#pragma unroll 8
        for (int s = 0; s < n_splits; ++s) v += part[(((int64_t)s * n_cb + kb) * 3 + t) * 256 + (i & 255)];
        const int rr = r + (t == 2 ? 16 : 0), cc = c + (t >= 1 ? 16 : 0);
        sm.A[rr * kEigLd + cc] = sm.B[0][rr * kEigLd + cc] = v;
        if (t == 1) sm.A[cc * kEigLd + rr] = sm.B[0][cc * kEigLd + rr] = v;
        if (rr == cc) sm.dg[0][rr] = v;
    }
    __syncthreads();
    const double tr = eig_sum(sm.dg[0]);
    float* out = data + (int64_t)kb * 64;
    if (!(tr < 1e150)) {                              // infinities or NaN in the weights
        if (tid < 64) out[tid] = __builtin_nanf("");
        return;
    }
    if (tr > 0.0) {
        eig_lead(sm, 0);
    } else {                                          // no residual at all
        if (tid < 32) sm.v[0][tid] = tid == 0 ? 1.0 : 0.0;
        __syncthreads();
    }
    if (tid < 32) {
        double w = 0.0;
#pragma unroll
        for (int i = 0; i < 32; ++i) w = __builtin_fma(sm.A[tid * kEigLd + i], sm.v[0][i], w);
        sm.w[tid] = w;
    }
    __syncthreads();
    double c = 0.0;
#pragma unroll
    for (int i = 0; i < 32; ++i) c = __builtin_fma(sm.w[i], sm.v[0][i], c);
    for (int i = tid; i < 1024; i += kEigThreads) {
        const int x = i >> 5, y = i & 31;
        const double vx = sm.v[0][x], vy = sm.v[0][y];
        const double d = sm.A[x * kEigLd + y] - (vx * sm.w[y] + sm.w[x] * vy) + c * vx * vy;
        sm.B[0][x * kEigLd + y] = d;
        if (x == y) sm.dg[0][x] = d;
    }
    __syncthreads();
    if (eig_sum(sm.dg[0]) > 1e-13 * tr) {
        eig_lead(sm, 1);
    } else if (tid < 32) {                            // one direction only: any unit vector beside it
        const int j = eig_argmax(sm.v[0], [](double d) { return -fabs(d); });
        const double p = sm.v[0][j];                  // e_j - p v, of squared length 1 - p^2
        sm.v[1][tid] = ((tid == j ? 1.0 : 0.0) - p * sm.v[0][tid]) / sqrt(1.0 - p * p);
    }
    __syncthreads();
    if (tid < 64) {                                   // the largest-magnitude component positive
        const double* v = sm.v[tid >> 5];
        const int arg = eig_argmax(v, [](double d) { return fabs(d); });
        out[tid] = (float)(v[arg] < 0.0 ? -v[tid & 31] : v[tid & 31]);
    }
}

// craw[kb][k][row] = basis_k . e, one thread per row of a K block.
__global__ __launch_bounds__(kThreads) void k_pca_coeff(const float* __restrict__ err,
                                                        const float* __restrict__ data, int n_rows,
                                                        float* __restrict__ craw) {
    const int kb = blockIdx.y;
    const int row = (int)blockIdx.x * kThreads + (int)threadIdx.x;
    if (row >= n_rows) return;
    const float4* e = reinterpret_cast<const float4*>(err + ((int64_t)kb * n_rows + row) * 32);
    const float* b = data + (int64_t)kb * 64;
    double c0 = 0.0, c1 = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float4 v = e[i];
        const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            c0 = __builtin_fma((double)b[4 * i + j], (double)x[j], c0);
            c1 = __builtin_fma((double)b[32 + 4 * i + j], (double)x[j], c1);
        }
    }
    craw[((int64_t)kb * 2) * n_rows + row] = (float)c0;
    craw[((int64_t)kb * 2 + 1) * n_rows + row] = (float)c1;
}

// The lower median of |craw| over the rows of one (kb, k), by radix selection on the float bits
// (non-negative floats order as integers): three passes of 11, 11 and 10 bits.  NaN sorts last
// here and is then the answer, as in torch.median.
__global__ __launch_bounds__(1024) void k_pca_scale(const float* __restrict__ craw, int n_rows,
                                                    float* __restrict__ scales) {
    __shared__ uint32_t hist[2048];
    __shared__ uint32_t sel_prefix, sel_rank, any_nan;
    __shared__ uint32_t wsum[16];
    const int tid = threadIdx.x;
    const float* c = craw + (int64_t)blockIdx.x * n_rows;
    uint32_t prefix = 0, rank = (uint32_t)(n_rows - 1) / 2;
    if (tid == 0) any_nan = 0;
#pragma unroll
    for (int pass = 0; pass < 3; ++pass) {
        const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0;
        const uint32_t mask = pass == 2 ? 0x3FFu : 0x7FFu;
        for (int i = tid; i < 2048; i += 1024) hist[i] = 0;
        __syncthreads();
        for (int i = tid; i < n_rows; i += 1024) {
            const uint32_t v = __builtin_bit_cast(uint32_t, c[i]) & 0x7FFFFFFFu;
            if (pass == 0 && v > 0x7F800000u) any_nan = 1;
            const bool in = pass == 0 || (v >> (pass == 1 ? 21 : 10)) == prefix;
            if (in) atomicAdd(&hist[(v >> shift) & mask], 1u);
        }
        __syncthreads();
        // bin of the rank: two bins per thread, sums over the waves, then the owner says
        const uint32_t h0 = hist[2 * tid], h1 = hist[2 * tid + 1];
        uint32_t incl = h0 + h1;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(incl, o);
            if ((tid & 63) >= o) incl += t;
        }
        if ((tid & 63) == 63) wsum[tid >> 6] = incl;
        __syncthreads();
        uint32_t base = 0;
        for (int w = 0; w < (tid >> 6); ++w) base += wsum[w];
        const uint32_t lo = base + incl - (h0 + h1);
        if (rank >= lo && rank < lo + h0 + h1) {
            const bool second = rank >= lo + h0;
            sel_prefix = (prefix << (pass == 2 ? 10 : 11)) | (uint32_t)(2 * tid + (second ? 1 : 0));
            sel_rank = rank - (second ? lo + h0 : lo);
        }
        __syncthreads();
        prefix = sel_prefix;
        rank = sel_rank;
        __syncthreads();
    }
    if (tid == 0) {
        const float med = any_nan ? __builtin_nanf("") : __builtin_bit_cast(float, prefix);
        const float s = med * (1.0f / 3.0f);          // (torch's form of a division by a number)
        scales[blockIdx.x] = s < 1e-10f ? 1e-10f : s;
    }
}

// Coefficient bytes, four K blocks of a row per thread, rows along the lanes.
__global__ __launch_bounds__(kThreads) void k_pca_byte(const float* __restrict__ craw,
                                                       const float* __restrict__ scales, int n_rows, int n_cb,
                                                       uint8_t* __restrict__ coeff) {
    const int row = (int)blockIdx.x * kThreads + (int)threadIdx.x;
    if (row >= n_rows) return;
    const int kb0 = blockIdx.y * 4;
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int kb = min(kb0 + j, n_cb - 1);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float v = __builtin_rintf(craw[((int64_t)kb * 2 + k) * n_rows + row] / scales[kb * 2 + k]);
            v = v < -8.f ? -8.f : (v > 7.f ? 7.f : v);
            w |= ((uint32_t)(int)v & 0xFu) << (8 * j + 4 * k);
        }
    }
    uint8_t* o = coeff + (int64_t)row * n_cb + kb0;
    if (kb0 + 4 <= n_cb && (reinterpret_cast<uintptr_t>(o) & 3) == 0) {
        *reinterpret_cast<uint32_t*>(o) = w;
    } else {
        for (int j = 0; j < 4 && kb0 + j < n_cb; ++j) o[j] = (uint8_t)(w >> (8 * j));
    }
}

struct PcaLayout {
    int64_t err, part, craw, total;
};
PcaLayout pca_layout(int64_t n_rows, int64_t n_cb) {
    PcaLayout l;
    l.err = 0;
    l.part = l.err + n_rows * n_cb * 128;
    l.craw = l.part + (int64_t)kPcaSplits * n_cb * 768 * 8;
    l.total = l.craw + n_rows * n_cb * 8;
    return l;
}

}  // namespace

extern "C" int32_t sx8_v6_encode(const uint16_t* W, int64_t out_f, int64_t in_f, int64_t ld,
                                 uint8_t* levels, uint16_t* dmin, uint16_t* dmax, uint8_t* config,
                                 uint8_t* levels_hi, uint8_t* levels_lo, void* stream) {
    using namespace sx8;
    if (!W || !dmin || !dmax || !config || !levels_hi || !levels_lo)
        return fail(SX8_ERR_INVALID, "sx8_v6_encode: null pointer argument");
    if (out_f <= 0 || in_f <= 0 || ld < in_f)
        return fail(SX8_ERR_INVALID, "sx8_v6_encode: bad shape out_f=%lld in_f=%lld ld=%lld",
                    (long long)out_f, (long long)in_f, (long long)ld);
    if (!aligned(W, 2) || !aligned(dmin, 2) || !aligned(dmax, 2))
        return fail(SX8_ERR_INVALID, "sx8_v6_encode: misaligned pointer");
    const int64_t n_cb = (in_f + 31) / 32;
    const int64_t grid = (out_f * n_cb + kThreads - 1) / kThreads;
    if (grid > 0x7FFFFFFF) return fail(SX8_ERR_UNSUPPORTED, "sx8_v6_encode: tensor too large");
    const bool vec_out = aligned(levels_hi, 16) && aligned(levels_lo, 8) && aligned(levels, 16);
    hipLaunchKernelGGL(k_v6_encode, dim3((unsigned)grid), dim3(kThreads), 0, as_stream(stream), W,
                       out_f, in_f, ld, n_cb, levels, dmin, dmax, config, levels_hi, levels_lo, vec_out);
    return check_launch("sx8_v6_encode");
}

extern "C" int64_t sx8_quant_pca_workspace_bytes(int64_t n_rows, int64_t n_cb) {
    if (n_rows <= 0 || n_cb <= 0 || n_rows > ((int64_t)1 << 36) / n_cb) return -1;
    return pca_layout(n_rows, n_cb).total;
}

extern "C" int32_t sx8_quant_pca(const void* blocks, const void* dmin, const void* dmax, int32_t is_f16,
                                 const uint8_t* levels, const uint8_t* config, int64_t n_rows, int64_t n_cb,
                                 uint8_t* coeff, float* data, float* scales, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
    using namespace sx8;
    const char* what = "sx8_quant_pca";
    if (!blocks || !dmin || !dmax || !levels || !config || !coeff || !data || !scales || !workspace)
        return fail(SX8_ERR_INVALID, "%s: null pointer argument", what);
    const int64_t need = sx8_quant_pca_workspace_bytes(n_rows, n_cb);
    if (need < 0) return fail(SX8_ERR_INVALID, "%s: bad shape n_rows=%lld n_cb=%lld", what, (long long)n_rows,
                              (long long)n_cb);
    const int esz = is_f16 ? 2 : 4;
    if (!aligned(blocks, esz) || !aligned(dmin, esz) || !aligned(dmax, esz) || !aligned(levels, 8) ||
        !aligned(data, 4) || !aligned(scales, 4) || !aligned(workspace, 16))
        return fail(SX8_ERR_INVALID, "%s: misaligned pointer", what);
    if (workspace_bytes < need)
        return fail(SX8_ERR_INVALID, "%s: workspace needs %lld bytes, got %lld", what, (long long)need,
                    (long long)workspace_bytes);
    const int64_t err_grid = (n_rows * n_cb * 4 + kThreads - 1) / kThreads;
    const int64_t row_grid = (n_rows + kThreads - 1) / kThreads;
    // grid limits: 65535 work-groups in y; 32-bit row numbers
    if (err_grid > 0x7FFFFFFF || n_rows > 0x3FFFFFFF || n_cb > 65535 || 2 * n_cb > 0x7FFFFFFF)
        return fail(SX8_ERR_UNSUPPORTED, "%s: tensor too large", what);
    const PcaLayout l = pca_layout(n_rows, n_cb);
    uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
    float* err = reinterpret_cast<float*>(ws + l.err);
    double* part = reinterpret_cast<double*>(ws + l.part);
    float* craw = reinterpret_cast<float*>(ws + l.craw);
    const hipStream_t st = as_stream(stream);
    if (is_f16)
        hipLaunchKernelGGL(k_pca_err<_Float16>, dim3((unsigned)err_grid), dim3(kThreads), 0, st,
                           reinterpret_cast<const _Float16*>(blocks), levels, reinterpret_cast<const _Float16*>(dmin),
                           reinterpret_cast<const _Float16*>(dmax), config, n_rows, n_cb, err);
    else
        hipLaunchKernelGGL(k_pca_err<float>, dim3((unsigned)err_grid), dim3(kThreads), 0, st,
                           reinterpret_cast<const float*>(blocks), levels, reinterpret_cast<const float*>(dmin),
                           reinterpret_cast<const float*>(dmax), config, n_rows, n_cb, err);
    const int rows_per = (int)((n_rows + kPcaSplits - 1) / kPcaSplits);
    hipLaunchKernelGGL(k_pca_gram, dim3((unsigned)n_cb, kPcaSplits), dim3(256), 0, st, err, (int)n_rows, rows_per,
                       part);
    hipLaunchKernelGGL(k_pca_eig, dim3((unsigned)n_cb), dim3(kEigThreads), 0, st, part, kPcaSplits, (int)n_cb, data);
    hipLaunchKernelGGL(k_pca_coeff, dim3((unsigned)row_grid, (unsigned)n_cb), dim3(kThreads), 0, st, err, data,
                       (int)n_rows, craw);
    hipLaunchKernelGGL(k_pca_scale, dim3((unsigned)(2 * n_cb)), dim3(1024), 0, st, craw, (int)n_rows, scales);
    hipLaunchKernelGGL(k_pca_byte, dim3((unsigned)row_grid, (unsigned)((n_cb + 3) / 4)), dim3(kThreads), 0, st, craw,
                       scales, (int)n_rows, (int)n_cb, coeff);
    return check_launch(what);
}
