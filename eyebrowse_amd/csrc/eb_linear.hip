// linear_f16w for gfx950: y[m, o] = sum_k x[m, k] * w[o, k], x and y f32, w IEEE half.
//
// Replaces linear_f16w (crates/eyebrowse-kernels/src/matmul.rs:84-144), a 16x16-tiled
// scalar GEMM that unpacks two halves per u32 word. The weight layout is the reference's:
// the logical [out, in] matrix flattened row-major, two halves per 32-bit word, low half
// first (crates/eyebrowse-gpu/src/tensor.rs:6-23); read as little-endian 16-bit units it
// is a plain half array, which is how the kernels address it.
//
// Two regimes:
//  - Few rows (decode, m <= kLinearGemvRows): HBM-bound on the weight (2*in*out bytes per
//    launch). One wave per kRowsPerWave output features (one per wave below 16384
//    features), or, for long rows, a workgroup per 4 or 8 features; lanes stride the
//    contraction in 16-byte chunks (8 halves), each chunk reused for every x row; the
//    multiply-adds read the halves directly (v_fma_mix_f32) and accumulate in f32. A wave
//    reduction (and a sum of the four waves) ends it.
//  - Many rows (prefill): matrix cores. The weight is exactly representable in f16, so
//    only x needs care: each x row is scaled by a power of two 2^-e (its largest
//    magnitude lands in [2^14, 2^15)) and split into x_hi = f16(x') and
//    x_lo = f16(x' - x_hi). Then x' = x_hi + x_lo to about 2^-22 relative, every product
//    x_hi*w and x_lo*w is exact in f32, and two v_mfma_f32_32x32x16_f16 per 32x32x16
//    block accumulate them in f32. The output is multiplied back by 2^e (ldexp). This
//    runs on the f16 matrix cores (2.5 PFLOP/s dense) at about f32 accuracy, where an
//    FP32-MFMA GEMM would be capped at 157 TFLOP/s. A pre-pass writes the row exponents.
//    Rows whose largest magnitude is not finite keep e = 0 and so give a non-finite
//    result, as the f32 product would.
//    With a workspace for the split rows (every recorder call), a pre-pass writes x_hi and
//    x_lo once and linear_tile_kernel copies both and the weight memory-to-LDS; without one
//    (raw launches, contractions not a multiple of 64) linear_gemm_kernel splits the rows it
//    stages in every workgroup.
// A scalar kernel covers shapes the vector paths do not (in % 8 != 0, unaligned
// pointers), like the reference's odd-width test (matmul.rs:255-272).
//
// Up to three (weight, output) pairs that share x run in one launch: q/k/v projections
// of one layer read the normalised hidden state once per tile instead of three times.
#include "eb_common.h"
#include "eb_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <climits>
#include <mutex>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

struct LinearSegs {
    const _Float16 *w[eb::kLinearMaxSegs];
    float *y[eb::kLinearMaxSegs];
    int n[eb::kLinearMaxSegs];      // output features of each pair
    int first[eb::kLinearMaxSegs + 1];  // first work unit of each pair; first[nseg] = total
    int nseg;
};

// The pair that owns work unit u (units are numbered pair by pair).
__device__ __forceinline__ int seg_of(const LinearSegs &s, int u) {
    int i = 0;
#pragma unroll
    for (int j = 1; j < eb::kLinearMaxSegs; ++j) i += (j < s.nseg && u >= s.first[j]) ? 1 : 0;
    return i;
}

__device__ __forceinline__ float wave_sum(float v) {
    v = eb::group_sum<16>(v);
    v += eb::lane_xor16(v);
    v += eb::lane_xor32(v);
    return v;
}

// ---------------------------------------------------------------- few rows ------------
constexpr int kRowsPerWave = 4;   // output features per wave
// Fewer output features than this many waves' worth (at kRowsPerWave each, i.e. below
// 16384 features) run one feature per wave, so that the launch still spreads over the
// chip. A feature's sum is the same either way (the same lanes, chunks and reduction), so
// the results are bit-identical. Measured (us per launch, 64 launches per graph, one box;
// four -> one feature per wave): Qwen q_proj 2.85 -> 2.28, k/v_proj 2.82 -> 2.19, a 4096-row
// head 3.08 -> 2.86. The Qwen LM head (151936 features) keeps four: one measured 44.1 ->
// 72.0, and two / eight 50.6 / 47.9 against four's 43.5.
#ifndef EB_GEMV_ONE_ROW_UNITS
#define EB_GEMV_ONE_ROW_UNITS 4096
#endif
constexpr int kGemvOneRowUnits = EB_GEMV_ONE_ROW_UNITS;
// Rows of up to this many halves are one wave's, a 16-byte chunk per lane and feature at a time:
// the Qwen LM head (in 1024) read at 5.0 TB/s with 4 chunks in flight (half of them clamped
// repeats of the row's last chunk), 6.3 TB/s with 2 and 6.9 TB/s with 1; 8 features per wave at 1
// or 2 chunks measured 6.1-6.3. Longer rows are linear_gemv_long_kernel's.
constexpr int kGemvShortRow = 1024;

// MR: capacity in x rows (the launch passes m <= MR). Requires in % 8 == 0 and 16-byte
// aligned x, w and rows (in % 8 == 0 keeps every row start aligned).
template <int MR, int RPW>
__global__ __launch_bounds__(kThreads) void linear_gemv_kernel(const float *__restrict__ x,
                                                               LinearSegs s, int m, int K) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int unit = blockIdx.x * kWaves + wave;  // a group of RPW features
    if (unit >= s.first[s.nseg]) return;          // whole waves only; no barriers below
    const int sg = seg_of(s, unit);
    const int N = s.n[sg];
    const int o0 = (unit - s.first[sg]) * RPW;
    const _Float16 *w = s.w[sg];
    const int k8 = K / 8;

    float acc[RPW][MR];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int i = 0; i < MR; ++i) acc[r][i] = 0.0f;

    for (int c0 = 0; c0 < k8; c0 += 64) {
        // All weight loads of the step first (clamped addresses, masked values), non-temporal:
        // each weight is read once per launch (the Qwen LM head, 311 MB: 4.78 -> 5.07 TB/s).
        f16x8 wv[RPW];
        const int c = c0 + lane;
        const int cc = c < k8 ? c : k8 - 1;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const int o = min(o0 + r, N - 1);
            wv[r] = __builtin_nontemporal_load(
                reinterpret_cast<const f16x8 *>(w + (size_t)o * K + (size_t)cc * 8));
        }
        if (c >= k8) break;
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            if (i >= m) break;
            const f32x4 xa = *reinterpret_cast<const f32x4 *>(x + (size_t)i * K + c * 8);
            const f32x4 xb = *reinterpret_cast<const f32x4 *>(x + (size_t)i * K + c * 8 + 4);
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                const f16x8 h = wv[r];
                float t = acc[r][i];
                t += xa.x * (float)h[0];
                t += xa.y * (float)h[1];
                t += xa.z * (float)h[2];
                t += xa.w * (float)h[3];
                t += xb.x * (float)h[4];
                t += xb.y * (float)h[5];
                t += xb.z * (float)h[6];
                t += xb.w * (float)h[7];
                acc[r][i] = t;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            const float v = wave_sum(acc[r][i]);
            if (lane == 0 && i < m && o0 + r < N) s.y[sg][(size_t)i * N + o0 + r] = v;
        }
}

template <int RPW>
void launch_gemv(unsigned blocks, hipStream_t st, const float *x, const LinearSegs &s, int m,
                 int K) {
    if (m <= 1)
        linear_gemv_kernel<1, RPW><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else if (m <= 2)
        linear_gemv_kernel<2, RPW><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else if (m <= 4)
        linear_gemv_kernel<4, RPW><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else
        linear_gemv_kernel<(int)eb::kLinearGemvRows, RPW><<<blocks, kThreads, 0, st>>>(x, s, m, K);
}

// Rows of more than kGemvShortRow halves: the workgroup's four waves share F features, thread t
// taking chunks t, t + 256, ... of every row. The threads' sums meet in LDS, where thread l of a
// wave adds those of threads l, 64 + l, 128 + l and 192 + l before the wave's sum: one wave sum
// per value, where one in each wave cost 8 rows over 100000 features 5 %. What bounded the
// one-wave-per-row form was not the weight but x, which every wave read whole (16 KB for 8 KB of
// weights at in 4096); here a wave reads a quarter of it for F features, and a thread has F loads
// of 16 bytes in flight. Measured (us, launches in a layer or a head, one wave per row or per four
// -> this form): Mistral token at 6000 keys 31.5 -> 29.0, Mistral 8 rows 78.4 -> 59.8, Qwen 8 rows
// 44.2 -> 35.5 (F 4; F 8 0.2 to 8 % slower). Weights of 16384 features and more: 2560 x 60000 at 2
// rows 68.1 -> 51.9, 3 rows 78.2 -> 74.2, 8 rows 135.4 -> 138.3; 4096 x 32768 at 4 rows 64.9 ->
// 59.6, 8 rows 96.5 -> 92.6; 1152 x 130000, where a row is 144 chunks for 256 threads, 3 rows 92.9
// -> 94.5, 8 rows 193.4 -> 193.3. Those take F 8 up to 4 rows (1 row 2560 x 60000 49.6, F 4 54.6;
// 4 rows 80.7, F 4 87.3), F 4 from 5 on (8 rows 138.4, F 8 148.2: the registers leave two waves
// per SIMD).
// The order of a sum depends on K alone (here, and above for K up to kGemvShortRow): not on the
// rows of the call, on F, or on the launch's other outputs.
template <int MR, int F>
__global__ __launch_bounds__(kThreads) void linear_gemv_long_kernel(const float *__restrict__ x,
                                                                    LinearSegs s, int m, int K) {
    __shared__ float part[F * MR][kThreads];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sg = seg_of(s, blockIdx.x);
    const int N = s.n[sg];
    const int o0 = (blockIdx.x - s.first[sg]) * F;
    const _Float16 *w = s.w[sg];
    const int k8 = K / 8;

    float acc[F][MR];
#pragma unroll
    for (int r = 0; r < F; ++r)
#pragma unroll
        for (int i = 0; i < MR; ++i) acc[r][i] = 0.0f;

    for (int c = tid; c < k8; c += kThreads) {
        f16x8 wv[F];  // (non-temporal as above; features past the last repeat it)
#pragma unroll
        for (int r = 0; r < F; ++r)
            wv[r] = __builtin_nontemporal_load(reinterpret_cast<const f16x8 *>(
                w + (size_t)min(o0 + r, N - 1) * K + (size_t)c * 8));
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            if (i >= m) break;
            const f32x4 xa = *reinterpret_cast<const f32x4 *>(x + (size_t)i * K + c * 8);
            const f32x4 xb = *reinterpret_cast<const f32x4 *>(x + (size_t)i * K + c * 8 + 4);
#pragma unroll
            for (int r = 0; r < F; ++r) {
                const f16x8 h = wv[r];
                float t = acc[r][i];
                t += xa.x * (float)h[0];
                t += xa.y * (float)h[1];
                t += xa.z * (float)h[2];
                t += xa.w * (float)h[3];
                t += xb.x * (float)h[4];
                t += xb.y * (float)h[5];
                t += xb.z * (float)h[6];
                t += xb.w * (float)h[7];
                acc[r][i] = t;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < F; ++r)
#pragma unroll
        for (int i = 0; i < MR; ++i)
            if (i < m) part[r * MR + i][tid] = acc[r][i];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < F * MR / kWaves; ++v) {
        const int f = v * kWaves + wave;
        if (f % MR >= m) continue;
        const float t = (part[f][lane] + part[f][64 + lane]) + (part[f][128 + lane] + part[f][192 + lane]);
        const float sum = wave_sum(t);
        if (lane == 0 && o0 + f / MR < N) s.y[sg][(size_t)(f % MR) * N + o0 + f / MR] = sum;
    }
}

template <int F>
void launch_gemv_long(unsigned blocks, hipStream_t st, const float *x, const LinearSegs &s, int m,
                      int K) {
    if (m <= 1)
        linear_gemv_long_kernel<1, F><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else if (m <= 2)
        linear_gemv_long_kernel<2, F><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else if (m <= 3)
        linear_gemv_long_kernel<3, F><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else if (m <= 4 || F > 4)  // (F 8 takes up to 4 rows)
        linear_gemv_long_kernel<4, F><<<blocks, kThreads, 0, st>>>(x, s, m, K);
    else
        linear_gemv_long_kernel<(int)eb::kLinearGemvRows, 4><<<blocks, kThreads, 0, st>>>(x, s, m, K);
}

// ---------------------------------------------------------------- any shape -----------
// One thread per output element, k ascending: the reference's order of summation.
__global__ __launch_bounds__(kThreads) void linear_scalar_kernel(const float *__restrict__ x,
                                                                 LinearSegs s, int m, int K) {
    const size_t idx = (size_t)blockIdx.x * kThreads + threadIdx.x;
    int sg = 0;
    size_t base = 0;
    for (; sg < s.nseg; ++sg) {
        const size_t cnt = (size_t)m * s.n[sg];
        if (idx < base + cnt) break;
        base += cnt;
    }
    if (sg >= s.nseg) return;
    const int N = s.n[sg];
    const size_t e = idx - base;
    const int i = (int)(e / N);
    const int o = (int)(e % N);
    const _Float16 *wr = s.w[sg] + (size_t)o * K;
    const float *xr = x + (size_t)i * K;
    float acc = 0.0f;
    for (int k = 0; k < K; ++k) acc += xr[k] * (float)wr[k];
    s.y[sg][(size_t)i * N + o] = acc;
}

// ---------------------------------------------------------------- many rows -----------
// Row exponents: ex[i] = e_i (as a float), e_i such that the row's largest magnitude
// times 2^-e_i lies in [2^14, 2^15) (e_i = 0 for zero or non-finite rows). One wave per
// row. Scaling uses ldexp (one rounding, no intermediate overflow), so e_i may exceed the
// exponent range of a single f32 scale factor (rows of subnormals need 2^163).
// With zero_out, the wave also zeroes its row of every output (for the split-contraction
// GEMM, whose halves add into y).
__global__ __launch_bounds__(kThreads) void linear_row_scale_kernel(const float *__restrict__ x,
                                                                    float *__restrict__ ex,
                                                                    int M, int K, LinearSegs s,
                                                                    bool zero_out) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= M) return;
    if (zero_out) {
        for (int g = 0; g < s.nseg; ++g) {
            float *yr = s.y[g] + (size_t)row * s.n[g];
            for (int c = lane; c < s.n[g]; c += 64) yr[c] = 0.0f;
        }
    }
    const float *xr = x + (size_t)row * K;
    float mx = 0.0f;
    float bad = 0.0f;  // becomes NaN (and stays NaN) once a NaN or inf is seen
    for (int c = lane; c < K / 4; c += 64) {  // K % 8 == 0 on this path
        const f32x4 v = *reinterpret_cast<const f32x4 *>(xr + 4 * c);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        bad += 0.0f * ((v.x + v.y) + (v.z + v.w));
    }
    mx = eb::class_reduce<1, true>(mx);
    bad = eb::class_reduce<1, false>(bad);
    int e = 0;
    if (bad == 0.0f && mx > 0.0f) e = ilogbf(mx) - 14;
    if (lane == 0) ex[row] = (float)e;
}

constexpr int kBM = 128;  // x rows per workgroup tile
#ifndef EB_LINEAR_BK
#define EB_LINEAR_BK 32
#endif
constexpr int kBK = EB_LINEAR_BK;  // contraction per LDS stage
// Shortest contraction cut in two halves when the 128 x 128 tiles alone leave CUs idle.
#ifndef EB_LINEAR_KSPLIT_MIN
#define EB_LINEAR_KSPLIT_MIN 1024
#endif
constexpr int kLdsRow = kBK + 8;  // halves per LDS row (16-byte pad against bank conflicts)
constexpr int kXcds = 8;  // MI355X: workgroup ids are dealt round-robin to 8 XCDs

template <int WNB>
struct GemmShape {
    static constexpr int BN = 64 * WNB;  // features per workgroup tile
    static constexpr int BUF = (2 * kBM + BN) * kLdsRow;  // halves: x_hi, x_lo, w
};
template <int WNB, int NBUF>
constexpr size_t gemm_lds_bytes() {
    return (size_t)NBUF * GemmShape<WNB>::BUF * 2;
}

__device__ __forceinline__ floatx16 mfma16(f16x8 a, f16x8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Requires in % 8 == 0 and 16-byte aligned x and w. Tile t: m-tile t / ntn, n-unit
// t % ntn (n-units numbered pair by pair). Workgroup ids are remapped so that each XCD
// works on a contiguous range of tiles (the same x rows), which its own L2 then keeps.
// WNB: 32-feature blocks per wave (the workgroup tile is 128 rows x 64*WNB features);
// NBUF: LDS buffers per stage (2: double buffered, one barrier per stage; 1: two
// barriers, half the LDS); MINB: workgroups per CU the registers must allow.
// ksplit 2: the contraction is cut in two halves, workgroups ids [tiles, 2*tiles) taking
// the second; each half adds its (scaled) partial into y, which the row-scale pre-pass
// zeroes first.
// Two addends onto zero give the same bits in either order (0 + a + b = a + b = b + a).
template <int WNB, int NBUF, int MINB>
__global__ __launch_bounds__(kThreads, MINB) void linear_gemm_kernel(const float *__restrict__ x,
                                                               const float *__restrict__ ex,
                                                               LinearSegs s, int M, int K,
                                                               int ksplit) {
    using Sh = GemmShape<WNB>;
    constexpr int BN = Sh::BN;
    extern __shared__ _Float16 lds[];
    __shared__ int s_ex[kBM];  // row exponents of the tile (read by the epilogue)
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int nt = gridDim.x / ksplit;
    const int bid = blockIdx.x % nt;
    const int half = blockIdx.x / nt;
    const int full = (nt / kXcds) * kXcds;
    const int t = bid < full ? (bid % kXcds) * (nt / kXcds) + bid / kXcds : bid;
    const int ntn = s.first[s.nseg];
    const int mt = t / ntn;
    const int nu = t % ntn;
    const int sg = seg_of(s, nu);
    const int N = s.n[sg];
    const int m0 = mt * kBM;
    const int n0 = (nu - s.first[sg]) * BN;
    const _Float16 *w = s.w[sg];
    if (tid < kBM) s_ex[tid] = (int)ex[min(m0 + tid, M - 1)];

    // Staging assignment: x tile kBM x kBK f32 (NX f32x4 per thread); w tile BN x kBK
    // halves (NW f16x8 per thread).
    constexpr int X4 = kBK / 4, W8 = kBK / 8;  // vectors per tile row
    constexpr int NX = kBM * X4 / kThreads, NW = BN * W8 / kThreads;
    f32x4 rx[NX];
    f16x8 rw[NW];
    int rs[NX];  // -e of the row each staged f32x4 belongs to
#pragma unroll
    for (int j = 0; j < NX; ++j) {
        const int idx = tid + j * kThreads;
        const int row = min(m0 + idx / X4, M - 1);
        rs[j] = -(int)ex[row];
    }
    // Whole contraction stages and buffers below 2 GiB (every model's projections): raw
    // buffer loads, the lane's byte offset computed once and the stage's as a scalar; rows
    // past M (x) or N (w) lie past the buffer's end and read as zeros. Otherwise clamped,
    // selected loads.
    const bool fast = K % kBK == 0 && (size_t)M * K * 4 <= (size_t)INT_MAX &&
                      (size_t)N * K * 2 <= (size_t)INT_MAX;
    const __amdgpu_buffer_rsrc_t xres = eb::make_rsrc(x, fast ? M * K * 4 : 0);
    const __amdgpu_buffer_rsrc_t wres = eb::make_rsrc(w, fast ? N * K * 2 : 0);
    unsigned xoff[NX], woff[NW];
#pragma unroll
    for (int j = 0; j < NX; ++j) {
        const int idx = tid + j * kThreads;
        xoff[j] = ((unsigned)(m0 + idx / X4) * (unsigned)K + (unsigned)(idx % X4) * 4u) * 4u;
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        const int idx = tid + j * kThreads;
        woff[j] = ((unsigned)(n0 + idx / W8) * (unsigned)K + (unsigned)(idx % W8) * 8u) * 2u;
    }
    auto load_stage = [&](int k0) {
        if (fast) {
            const int kx = __builtin_amdgcn_readfirstlane(4 * k0);  // (uniform: scalar)
            const int kw = __builtin_amdgcn_readfirstlane(2 * k0);
#pragma unroll
            for (int j = 0; j < NX; ++j)
                rx[j] = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(xres, (int)xoff[j], kx, 0));
#pragma unroll
            for (int j = 0; j < NW; ++j)
                rw[j] = __builtin_bit_cast(
                    f16x8, __builtin_amdgcn_raw_buffer_load_b128(wres, (int)woff[j], kw, 0));
            return;
        }
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int idx = tid + j * kThreads;
            const int r = idx / X4, c4 = idx % X4;
            const int row = m0 + r, k = k0 + c4 * 4;
            const bool ok = row < M && k < K;
            const f32x4 v = *reinterpret_cast<const f32x4 *>(
                x + (size_t)min(row, M - 1) * K + (ok ? k : 0));
            rx[j] = ok ? v : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int j = 0; j < NW; ++j) {
            const int idx = tid + j * kThreads;
            const int r = idx / W8, c8 = idx % W8;
            const int o = n0 + r, k = k0 + c8 * 8;
            const bool ok = o < N && k < K;
            const f16x8 v = *reinterpret_cast<const f16x8 *>(
                w + (size_t)min(o, N - 1) * K + (ok ? k : 0));
            rw[j] = ok ? v : f16x8{};
        }
    };
    auto store_stage = [&](int buf) {
        _Float16 *hi = lds + buf * Sh::BUF;
        _Float16 *lo = hi + kBM * kLdsRow;
        _Float16 *wt = lo + kBM * kLdsRow;
#pragma unroll
        for (int j = 0; j < NX; ++j) {
            const int idx = tid + j * kThreads;
            const int r = idx / X4, c4 = idx % X4;
            const f32x4 v = {ldexpf(rx[j].x, rs[j]), ldexpf(rx[j].y, rs[j]),
                             ldexpf(rx[j].z, rs[j]), ldexpf(rx[j].w, rs[j])};
            const f16x4 h = __builtin_convertvector(v, f16x4);
            const f16x4 l = __builtin_convertvector(v - __builtin_convertvector(h, f32x4), f16x4);
            *reinterpret_cast<f16x4 *>(hi + r * kLdsRow + c4 * 4) = h;
            *reinterpret_cast<f16x4 *>(lo + r * kLdsRow + c4 * 4) = l;
        }
#pragma unroll
        for (int j = 0; j < NW; ++j) {
            const int idx = tid + j * kThreads;
            const int r = idx / W8, c8 = idx % W8;
            *reinterpret_cast<f16x8 *>(wt + r * kLdsRow + c8 * 8) = rw[j];
        }
    };

    // Wave (wm, wn) computes rows wm*64..+64 and features wn*32*WNB..+32*WNB of the tile:
    // 2 x WNB blocks of 32 x 32.
    const int wm = wave >> 1, wn = wave & 1;
    floatx16 acc[2][WNB];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < WNB; ++b) acc[a][b] = floatx16{};

    auto compute = [&](int buf) {
        const _Float16 *hi = lds + buf * Sh::BUF;
        const _Float16 *lo = hi + kBM * kLdsRow;
        const _Float16 *wt = lo + kBM * kLdsRow;
#pragma unroll
        for (int kk = 0; kk < kBK / 16; ++kk) {
            const int kof = kk * 16 + (lane >> 5) * 8;
            f16x8 ah[2], al[2], bw[WNB];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int r = wm * 64 + a * 32 + (lane & 31);
                ah[a] = *reinterpret_cast<const f16x8 *>(hi + r * kLdsRow + kof);
                al[a] = *reinterpret_cast<const f16x8 *>(lo + r * kLdsRow + kof);
            }
#pragma unroll
            for (int b = 0; b < WNB; ++b) {
                const int r = wn * 32 * WNB + b * 32 + (lane & 31);
                bw[b] = *reinterpret_cast<const f16x8 *>(wt + r * kLdsRow + kof);
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < WNB; ++b) {
                    acc[a][b] = mfma16(ah[a], bw[b], acc[a][b]);
                    acc[a][b] = mfma16(al[a], bw[b], acc[a][b]);
                }
        }
    };

    // This workgroup's stages: all of them, or one half of the contraction.
    const int nst_all = (K + kBK - 1) / kBK;
    const int per = (nst_all + ksplit - 1) / ksplit;
    const int st0 = half * per;
    const int nst = min(nst_all - st0, per);
    load_stage(st0 * kBK);
    store_stage(0);
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
        if (st + 1 < nst) load_stage((st0 + st + 1) * kBK);
        if constexpr (NBUF == 2) {
            compute(st & 1);
            if (st + 1 < nst) store_stage((st & 1) ^ 1);
            __syncthreads();
        } else {
            compute(0);
            if (st + 1 < nst) {
                __syncthreads();  // every wave is done reading the buffer
                store_stage(0);
                __syncthreads();
            }
        }
    }

    // Epilogue: lane holds feature j = lane % 32 of each block, rows
    // 8*(r/4) + 4*(lane/32) + r%4; scale back and store (32 consecutive features per row).
    float *y = s.y[sg];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < WNB; ++b) {
            const int o = n0 + wn * 32 * WNB + b * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int rt = wm * 64 + a * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                const int row = m0 + rt;
                if (row < M && o < N) {
                    const float v = ldexpf(acc[a][b][r], s_ex[rt]);
                    if (ksplit == 1)
                        y[(size_t)row * N + o] = v;
                    else
                        atomicAdd(y + (size_t)row * N + o, v);
                }
            }
        }
}

// ---------------------------------------------------------------- many rows, split once -
// Split pass: row i of x scaled by 2^-e_i (linear_row_scale_kernel's exponent, into ex) and
// split, x_hi into xs row i and x_lo into xs row M + i. One wave per row; rows of up to NC * 512
// elements stay in registers between the maximum and the split (NC 0: read twice).
// Bytes: 4 + 4 per element; 4096 x 4096 takes 19.9 us (6.7 TB/s), 64 x 1024 2.5 us (a launch).
template <int NC>
__global__ __launch_bounds__(kThreads) void linear_split_kernel(const float *__restrict__ x,
                                                                _Float16 *__restrict__ xs,
                                                                float *__restrict__ ex, int M,
                                                                int K) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= M) return;
    const float *xr = x + (size_t)row * K;
    const int k8 = K / 8;
    struct Oct {
        f32x4 a, b;
    };
    auto load = [&](int c) {
        const float *p = xr + (size_t)(c < k8 ? c : 0) * 8;  // (clamped: a repeat moves no max)
        return Oct{*reinterpret_cast<const f32x4 *>(p), *reinterpret_cast<const f32x4 *>(p + 4)};
    };
    float mx = 0.0f, bad = 0.0f;
    auto scan = [&](const Oct &v) {
        mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(v.a.x), fabsf(v.a.y)), fmaxf(fabsf(v.a.z), fabsf(v.a.w))),
                             fmaxf(fmaxf(fabsf(v.b.x), fabsf(v.b.y)), fmaxf(fabsf(v.b.z), fabsf(v.b.w)))));
        bad += 0.0f * ((v.a.x + v.a.y) + (v.a.z + v.a.w));
        bad += 0.0f * ((v.b.x + v.b.y) + (v.b.z + v.b.w));
    };
    Oct v[NC > 0 ? NC : 1];
    if constexpr (NC > 0) {
#pragma unroll
        for (int j = 0; j < NC; ++j) v[j] = load(j * 64 + lane);
#pragma unroll
        for (int j = 0; j < NC; ++j) scan(v[j]);
    } else {
        for (int c = lane; c < k8; c += 64) scan(load(c));
    }
    mx = eb::class_reduce<1, true>(mx);
    bad = eb::class_reduce<1, false>(bad);
    int e = 0;
    if (bad == 0.0f && mx > 0.0f) e = ilogbf(mx) - 14;
    if (lane == 0) ex[row] = (float)e;
    _Float16 *hi = xs + (size_t)row * K, *lo = hi + (size_t)M * K;
    auto store = [&](int c, const Oct &o) {
        typedef float f32x8 __attribute__((ext_vector_type(8)));
        const f32x8 q = {ldexpf(o.a.x, -e), ldexpf(o.a.y, -e), ldexpf(o.a.z, -e), ldexpf(o.a.w, -e),
                         ldexpf(o.b.x, -e), ldexpf(o.b.y, -e), ldexpf(o.b.z, -e), ldexpf(o.b.w, -e)};
        const f16x8 h = __builtin_convertvector(q, f16x8);
        *reinterpret_cast<f16x8 *>(hi + (size_t)c * 8) = h;
        *reinterpret_cast<f16x8 *>(lo + (size_t)c * 8) =
            __builtin_convertvector(q - __builtin_convertvector(h, f32x8), f16x8);
    };
    if constexpr (NC > 0) {
#pragma unroll
        for (int j = 0; j < NC; ++j)
            if (j * 64 + lane < k8) store(j * 64 + lane, v[j]);
    } else {
        for (int c = lane; c < k8; c += 64) store(c, load(c));
    }
}

// Tile shape: WM x WN waves of TM x TN blocks of 32 x 32, times KW waves that share the 16-deep
// steps of a stage (wave kw takes steps kw, kw + KW, ...), BK of the contraction per stage,
// NBUF stages in LDS.
template <int WM_, int WN_, int TM_, int TN_, int KW_, int BK_, int NBUF_>
struct TileShape {
    static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, KW = KW_, BK = BK_, NBUF = NBUF_;
    static constexpr int NW = WM * WN * KW, THREADS = NW * 64;
    static constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    static constexpr int ROWB = BK * 2;                  // bytes of an LDS row
    static constexpr int STAGE = (2 * BM + BN) * ROWB;   // x_hi rows, x_lo rows, w rows
    static constexpr int NI = STAGE / 1024 / NW;         // 1 KiB copies per wave and stage
    // One wave per output: the contraction's halves are summed apart where the registers hold two
    // sums (see linear_tile_kernel).
    static constexpr bool HALVES = KW == 1 && TM * TN <= 2;
    static constexpr int RED = KW > 1 ? NW * TM * TN * 16 * 256 : 0;  // the waves' partial sums
    static constexpr int LDS = NBUF * STAGE > RED ? NBUF * STAGE : RED;
    static_assert(STAGE % (1024 * NW) == 0, "every wave issues NI copies per stage");
    // Waves per SIMD that the LDS allows (the compiler does not see the dynamic LDS).
    static constexpr int WGS = 160 * 1024 / (LDS + BM * 4);
    static constexpr int WAVES = WGS * NW / 4 < 1 ? 1 : WGS * NW / 4 > 8 ? 8 : WGS * NW / 4;
};
// Chunk c (16 bytes) of LDS row r lies at chunk c ^ tile_swizzle(r) of the row, so that eight
// consecutive rows' chunks c, read together as an MFMA operand, meet eight different bank groups.
// The copies keep whole 64- or 128-byte pieces of a row on consecutive lanes.
template <int BK>
__device__ __forceinline__ int tile_swizzle(int r) {
    return BK == 32 ? (r >> 1) & 3 : r & 7;
}

template <int N>
__device__ __forceinline__ void wait_copies() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// y tile = x tile . w tile^T from the split rows xs and exponents ex. Requires K % BK == 0, M * K
// below 2^30, N * K below 2^31 (as every launch's weight is), 16-byte aligned xs and w.
//
// The operands go memory-to-LDS (global_load_lds: no registers, no arithmetic), NBUF - 1 stages
// ahead, one barrier per stage. As inline assembly, which the compiler's wait counting does not
// see; they complete in issue order, so a stage is there when at most the later stages' copies
// are outstanding. Past the last stage they repeat it (into buffers that nobody reads).
// What bounds it: tiles of 128 x 256 and up the matrix cores at the clock that the power limit
// leaves (1.1-1.2 PFLOP/s of f16 products at 4096 x 4096 x 4096; a library f16 product of 8192^3
// reaches 1.23 here); smaller ones the bytes that a CU can fetch from L2 (about 50 B/ns), hence
// tiles that balance 2 BM against BN, and as many of them as there are CUs. Against
// linear_gemm_kernel, which splits x in every workgroup and has no shape for few rows (us, split
// pass included, q/k/v then o_proj): Qwen 64 rows 22.5 -> 7.9, 32.2 -> 9.7, 1000 rows 52 -> 28,
// 37.5 -> 23.5; Mistral 64 rows 59 -> 18, 57 -> 16, 500 rows 88 -> 65, 74 -> 48, 4096 rows
// 420 -> 375, 280 -> 249.
//
// With KW > 1 the waves' partial sums meet in LDS, in the order of kw. With one wave per output
// (KW 1) and up to two blocks of accumulators, the first half of the contraction is set aside
// half way and added at the end: the roundings of a sum are half as many, of half the size
// (relative error against 64 bits 2.9e-7 in one chain, 2.1e-7 in two at K 1024, 5.8e-7 and
// 4.1e-7 at 4096). linear_gemm_kernel cuts the contraction at the sizes that these shapes take;
// the larger shapes keep one chain, as its wide tiles do. A result's bits depend on KW, HALVES,
// BK and K, not otherwise on the tile. With the eight-wave shapes (kTileFewRows) they are the same
// whatever the launch's other outputs; beyond, the tile (so HALVES) is chosen for all outputs
// together, and a fused and a separate projection of many rows may differ in their last bits
// (linear_gemm_kernel's wide tiles and cut contraction do so too).
// Workgroups: each XCD gets a contiguous range of tiles, in groups of kGroupM row tiles by all
// feature tiles, row tile fastest, so that the tiles in flight on an XCD share rows and features.
constexpr int kGroupM = 4;
template <class C>
__global__ __attribute__((amdgpu_flat_work_group_size(C::THREADS, C::THREADS),
                          amdgpu_waves_per_eu(C::WAVES, C::WAVES))) void
linear_tile_kernel(const _Float16 *__restrict__ xs, const float *__restrict__ ex, LinearSegs s,
                   int M, int K) {
    constexpr int BM = C::BM, BN = C::BN, BK = C::BK, TM = C::TM, TN = C::TN, KW = C::KW;
    constexpr int ROWB = C::ROWB, CPR = BK / 8;  // 16-byte chunks per LDS row
    extern __shared__ char tile_lds[];
    __shared__ int s_ex[BM];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt = gridDim.x, bid = blockIdx.x;
    const int full = (nt / kXcds) * kXcds;
    const int t = bid < full ? (bid % kXcds) * (nt / kXcds) + bid / kXcds : bid;
    const int ntn = s.first[s.nseg], ntm = nt / ntn;
    const int g0 = t / (kGroupM * ntn) * kGroupM, r0 = t % (kGroupM * ntn);
    const int gm = min(kGroupM, ntm - g0);  // row tiles of this group
    const int nu = r0 / gm;
    const int sg = seg_of(s, nu);
    const int N = s.n[sg];
    const int m0 = __builtin_amdgcn_readfirstlane((g0 + r0 % gm) * BM);
    const int n0 = __builtin_amdgcn_readfirstlane((nu - s.first[sg]) * BN);
    const _Float16 *w = s.w[sg];
    for (int i = tid; i < BM; i += C::THREADS) s_ex[i] = (int)ex[min(m0 + i, M - 1)];

    // Copy i of this wave fills KiB block i * NW + wave of the stage; the lane's byte offset
    // within xs (or w). Rows past the end repeat the last one; they are not stored.
    unsigned voff[C::NI];
#pragma unroll
    for (int i = 0; i < C::NI; ++i) {
        const int q = (i * C::NW + wave) * 64 + lane;
        const int row = q / CPR, c = (q % CPR) ^ tile_swizzle<BK>(row);
        const int xr = min(m0 + (row < BM ? row : row - BM), M - 1) + (row < BM ? 0 : M);
        const int wr = min(n0 + row - 2 * BM, N - 1);
        voff[i] = (unsigned)(row < 2 * BM ? xr : wr) * (unsigned)K * 2u + c * 16u;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)tile_lds;
    auto copy_stage = [&](int buf, bool more) {
#pragma unroll
        for (int i = 0; i < C::NI; ++i) {
            const int b = i * C::NW + wave;  // (uniform; 2 BM rows are whole blocks)
            const void *base = b >= 2 * BM * ROWB / 1024 ? static_cast<const void *>(w)
                                                         : static_cast<const void *>(xs);
            const unsigned dst = __builtin_amdgcn_readfirstlane(lds0 + buf * C::STAGE + b * 1024);
            // (s_nop: a copy to LDS may read m0 one wait state after its write at the soonest.)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :
                         : "s"(dst), "v"(voff[i]), "s"(base)
                         : "memory", "m0");
        }
#pragma unroll
        for (int i = 0; i < C::NI; ++i) voff[i] += more ? 2 * BK : 0;
    };

    const int kw = wave / (C::WM * C::WN), slot = wave % (C::WM * C::WN);
    const int wm = slot / C::WN, wn = slot % C::WN;
    const int hf = lane >> 5, l32 = lane & 31;
    floatx16 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = floatx16{};

    const int nst = K / BK;
#pragma unroll
    for (int p = 0; p < C::NBUF - 1; ++p) copy_stage(p, p + 1 < nst);
    constexpr int STEPS = BK / 16 / KW;
    unsigned off[STEPS];  // the lane's chunk of row l32 in each of its steps
#pragma unroll
    for (int j = 0; j < STEPS; ++j)
        off[j] = l32 * ROWB + ((((j * KW + kw) * 2 + hf) ^ tile_swizzle<BK>(l32)) * 16);
    int buf = 0, nb = C::NBUF - 1;
    floatx16 first[C::HALVES ? TM : 1][C::HALVES ? TN : 1] = {};
    // (Two loops: a test in one cost a move per accumulator register and stage, a 1000-row Qwen
    // layer 95 -> 100 us.)
    auto stages = [&](int st0, int st1) {
        for (int st = st0; st < st1; ++st) {
            wait_copies<(C::NBUF - 2) * C::NI>();
            __syncthreads();  // stage st is there, and nobody reads buffer nb any more
            copy_stage(nb, st + C::NBUF < nst);
            const char *xb = tile_lds + buf * C::STAGE + wm * TM * 32 * ROWB;
            const char *wb = tile_lds + buf * C::STAGE + (2 * BM + wn * TN * 32) * ROWB;
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                f16x8 ah[TM], al[TM], bw[TN];
#pragma unroll
                for (int b = 0; b < TN; ++b)
                    bw[b] = *reinterpret_cast<const f16x8 *>(wb + off[j] + b * 32 * ROWB);
#pragma unroll
                for (int a = 0; a < TM; ++a) {
                    ah[a] = *reinterpret_cast<const f16x8 *>(xb + off[j] + a * 32 * ROWB);
                    al[a] = *reinterpret_cast<const f16x8 *>(xb + off[j] + (BM + a * 32) * ROWB);
                }
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) acc[a][b] = mfma16(ah[a], bw[b], acc[a][b]);
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b) acc[a][b] = mfma16(al[a], bw[b], acc[a][b]);
            }
            buf = buf == C::NBUF - 1 ? 0 : buf + 1;
            nb = nb == C::NBUF - 1 ? 0 : nb + 1;
        }
    };
    if constexpr (C::HALVES) {
        stages(0, nst / 2);
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b) first[a][b] = acc[a][b], acc[a][b] = floatx16{};
        stages(nst / 2, nst);
    } else {
        stages(0, nst);
    }
    wait_copies<0>();  // (the repeated last stages)
    if constexpr (C::HALVES) {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b) acc[a][b] = first[a][b] + acc[a][b];
    }

    // Register r of block (a, b): feature l32 of the block, row 8*(r/4) + 4*hf + r%4.
    float *y = s.y[sg];
    auto put = [&](int a, int b, int r, float v) {
        const int o = n0 + (wn * TN + b) * 32 + l32;
        const int rt = (wm * TM + a) * 32 + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (m0 + rt < M && o < N) y[(size_t)(m0 + rt) * N + o] = ldexpf(v, s_ex[rt]);
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) put(a, b, r, acc[a][b][r]);
    } else {
        constexpr int NR = TM * TN * 16;  // registers of a wave; wave kw sums NR / KW of them
        __syncthreads();                  // every wave's copies and reads are done
        float *red = reinterpret_cast<float *>(tile_lds);
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    red[(wave * NR + (a * TN + b) * 16 + r) * 64 + lane] = acc[a][b][r];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NR / KW; ++i) {
            const int f = kw * (NR / KW) + i;
            float v = red[(slot * NR + f) * 64 + lane];
#pragma unroll
            for (int k = 1; k < KW; ++k) v += red[((k * C::WM * C::WN + slot) * NR + f) * 64 + lane];
            put(f / 16 / TN, f / 16 % TN, f % 16, v);
        }
    }
}

template <class C>
eb_status launch_tile(hipStream_t st, const _Float16 *xs, const float *ex, LinearSegs s,
                      const size_t *out_f, int nseg, size_t m, size_t in_f) {
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(&linear_tile_kernel<C>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    });
    if (attr_err != hipSuccess) return eb::hip_fail(attr_err, "hipFuncSetAttribute(linear)");
    s.first[0] = 0;
    for (int i = 0; i < nseg; ++i)
        s.first[i + 1] = s.first[i] + (int)((out_f[i] + C::BN - 1) / C::BN);
    const size_t tiles = (m + C::BM - 1) / C::BM * (size_t)s.first[nseg];
    linear_tile_kernel<C><<<(unsigned)tiles, C::THREADS, C::LDS, st>>>(xs, ex, s, (int)m, (int)in_f);
    return eb::check_launch("linear_f16w");
}

// The tile shapes, and the time of one round of tiles (one per CU) as fixed + per_k * K us, fitted
// to a sweep of 9 to 4096 rows at the Qwen and Mistral widths (made before the shapes with HALVES
// cut their sums in two; not fitted again since). tile_cost takes the rounds of the fullest CU, or
// half way to the average where two workgroups share a CU and overlap.
struct TileModel {
    int bm, bn;
    bool shared;  // two workgroups per CU
    float fixed, per_k;
};
// Up to kTileFewRows rows and whole 128-deep stages: eight waves share each stage's steps, which
// keeps a CU's copies in flight on the small tiles that few rows need. Beyond, one wave sums an
// output. The line is a number of rows, so that it does not move with the launch's other outputs.
// Both sides of it (us, split pass included, eight waves / one): Mistral o_proj 128 rows 18.8 /
// 29.9, 256 rows 27.5 / 31.3; q/k/v 24.9 / 29.8, 45.5 / 44.8; Qwen o_proj 10.2 / 17.8, 10.4 /
// 18.9; 1536 -> 6144, the worst for eight waves, 14.0 / 15.2, 23.6 / 21.5.
using TileK8a = TileShape<1, 1, 1, 1, 8, 128, 4>;
using TileK8b = TileShape<1, 1, 1, 2, 8, 128, 4>;
using TileK8c = TileShape<1, 1, 2, 2, 8, 128, 3>;
using TileA = TileShape<2, 2, 1, 1, 1, 64, 3>;
using TileB = TileShape<2, 4, 1, 1, 1, 64, 2>;
using TileC = TileShape<4, 2, 1, 2, 1, 64, 3>;
using TileD = TileShape<2, 4, 2, 2, 1, 32, 2>;
using TileE = TileShape<4, 2, 2, 4, 1, 32, 3>;
constexpr size_t kTileFewRows = 256;
constexpr TileModel kTilesK8[] = {{32, 32, false, 1.5f, 2.33e-3f},
                                  {32, 64, false, 2.2f, 2.9e-3f},
                                  {64, 64, false, 3.6f, 4.75e-3f}};
constexpr TileModel kTiles[] = {{64, 64, true, 3.0f, 5.2e-3f},
                                {64, 128, true, 4.0f, 8.0e-3f},
                                {128, 128, false, 5.0f, 15.2e-3f},
                                {128, 256, true, 6.0f, 27.5e-3f},
                                {256, 256, false, 12.0f, 53.0e-3f}};
float tile_cost(const TileModel &t, const size_t *out_f, int nseg, size_t m, size_t in_f, float cus) {
    size_t units = 0;
    for (int i = 0; i < nseg; ++i) units += (out_f[i] + t.bn - 1) / t.bn;
    const float avg = (float)((m + t.bm - 1) / t.bm * units) / cus;
    float rounds = std::ceil(avg);
    if (t.shared && avg > 1.0f) rounds = 0.5f * (rounds + avg);
    return rounds * (t.fixed + t.per_k * (float)in_f);
}
template <size_t NT>
int best_tile(const TileModel (&tiles)[NT], const size_t *out_f, int nseg, size_t m, size_t in_f) {
    const float cus = (float)eb::current_cu_count();
    int best = 0;
    float cost = 0.0f;
    for (int i = 0; i < (int)NT; ++i) {
        const float c = tile_cost(tiles[i], out_f, nseg, m, in_f, cus);
        if (i == 0 || c < cost) cost = c, best = i;
    }
    return best;
}

// Floats ahead of the split rows: the row exponents, to whole 256-byte lines.
size_t tile_ex_floats(size_t m) { return (m + 63) / 64 * 64; }

eb_status launch_tiles(hipStream_t st, const float *x, const LinearSegs &s, const size_t *out_f,
                       int nseg, size_t m, size_t in_f, float *ws) {
    float *ex = ws;
    _Float16 *xs = reinterpret_cast<_Float16 *>(ws + tile_ex_floats(m));
    const unsigned grid = (unsigned)((m + kWaves - 1) / kWaves);
    const int M = (int)m, K = (int)in_f;
    if (K <= 1024) linear_split_kernel<2><<<grid, kThreads, 0, st>>>(x, xs, ex, M, K);
    else if (K <= 2048) linear_split_kernel<4><<<grid, kThreads, 0, st>>>(x, xs, ex, M, K);
    else if (K <= 4096) linear_split_kernel<8><<<grid, kThreads, 0, st>>>(x, xs, ex, M, K);
    else linear_split_kernel<0><<<grid, kThreads, 0, st>>>(x, xs, ex, M, K);
    const eb_status err = eb::check_launch("linear_f16w (split pass)");
    if (err != EB_OK) return err;
    if (m <= kTileFewRows && in_f % 128 == 0) {
        switch (best_tile(kTilesK8, out_f, nseg, m, in_f)) {
            case 0: return launch_tile<TileK8a>(st, xs, ex, s, out_f, nseg, m, in_f);
            case 1: return launch_tile<TileK8b>(st, xs, ex, s, out_f, nseg, m, in_f);
            default: return launch_tile<TileK8c>(st, xs, ex, s, out_f, nseg, m, in_f);
        }
    }
    switch (best_tile(kTiles, out_f, nseg, m, in_f)) {
        case 0: return launch_tile<TileA>(st, xs, ex, s, out_f, nseg, m, in_f);
        case 1: return launch_tile<TileB>(st, xs, ex, s, out_f, nseg, m, in_f);
        case 2: return launch_tile<TileC>(st, xs, ex, s, out_f, nseg, m, in_f);
        case 3: return launch_tile<TileD>(st, xs, ex, s, out_f, nseg, m, in_f);
        default: return launch_tile<TileE>(st, xs, ex, s, out_f, nseg, m, in_f);
    }
}

// ksplit 2 expects the outputs zeroed (linear_row_scale_kernel's zero_out).
template <int WNB, int NBUF, int MINB>
eb_status launch_gemm(hipStream_t st, const float *x, const float *ex, LinearSegs s,
                      const size_t *out_f, int nseg, size_t m, size_t in_f, int ksplit = 1) {
    constexpr int BN = GemmShape<WNB>::BN;
    constexpr size_t lds_bytes = gemm_lds_bytes<WNB, NBUF>();
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [] {
        attr_err = hipFuncSetAttribute(
            reinterpret_cast<const void *>(&linear_gemm_kernel<WNB, NBUF, MINB>),
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    });
    if (attr_err != hipSuccess) return eb::hip_fail(attr_err, "hipFuncSetAttribute(linear)");
    s.first[0] = 0;
    for (int i = 0; i < nseg; ++i)
        s.first[i + 1] = s.first[i] + (int)((out_f[i] + BN - 1) / BN);
    const size_t tiles = (size_t)((m + kBM - 1) / kBM) * (size_t)s.first[nseg];
    linear_gemm_kernel<WNB, NBUF, MINB><<<(unsigned)(tiles * ksplit), kThreads, lds_bytes, st>>>(
        x, ex, s, (int)m, (int)in_f, ksplit);
    return eb::check_launch("linear_f16w");
}

__global__ __launch_bounds__(kThreads) void zero_fill_kernel(float *__restrict__ y, size_t n) {
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) y[i] = 0.0f;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

namespace eb {

size_t linear_workspace_floats(size_t m, size_t in_f) {
    return (m > kLinearGemvRows && in_f % 8 == 0) ? m : 0;
}

// (M * K below 2^30: the split rows' byte offsets are 32 bits.)
size_t linear_split_workspace_floats(size_t m, size_t in_f) {
    if (m <= kLinearGemvRows || in_f == 0 || in_f % 64 != 0 || m > ((size_t)1 << 30) / in_f - 1)
        return linear_workspace_floats(m, in_f);
    return tile_ex_floats(m) + m * in_f;
}

size_t linear_usable_workspace_floats(const float *x, const uint16_t *const *w,
                                      const size_t *out_f, int nseg, size_t m, size_t in_f) {
    bool split = aligned16(x);
    size_t total_out = 0;
    for (int i = 0; i < nseg; ++i) {
        split = split && aligned16(w[i]);
        total_out += out_f[i];
    }
    return split && total_out > 0 ? linear_split_workspace_floats(m, in_f)
                                  : linear_workspace_floats(m, in_f);
}

eb_status launch_linear_f16w_multi(hipStream_t st, const float *x, const uint16_t *const *w,
                                   float *const *y, const size_t *out_f, int nseg, size_t m,
                                   size_t in_f, float *ws, size_t ws_floats) {
    if (nseg < 1 || nseg > kLinearMaxSegs) return fail(EB_OTHER, "linear: 1..3 weights");
    if (m == 0) return ok();
    bool vec = in_f % 8 == 0 && aligned16(x);
    size_t total_out = 0;
    for (int i = 0; i < nseg; ++i) {
        vec = vec && aligned16(w[i]);
        total_out += out_f[i];
    }
    if (total_out == 0) return ok();
    if (in_f == 0) {  // empty sums: zeros (a kernel, not a memset, so graphs may hold it)
        for (int i = 0; i < nseg; ++i) {
            const size_t n = m * out_f[i];
            if (n == 0) continue;
            zero_fill_kernel<<<(unsigned)std::min<size_t>((n + kThreads - 1) / kThreads, 4096),
                               kThreads, 0, st>>>(y[i], n);
        }
        return check_launch("linear_f16w");
    }
    LinearSegs s{};
    s.nseg = nseg;
    for (int i = 0; i < nseg; ++i) {
        s.w[i] = reinterpret_cast<const _Float16 *>(w[i]);
        s.y[i] = y[i];
        s.n[i] = (int)out_f[i];
    }
    if (!vec) {
        const size_t elems = m * total_out;
        linear_scalar_kernel<<<(unsigned)((elems + kThreads - 1) / kThreads), kThreads, 0, st>>>(
            x, s, (int)m, (int)in_f);
        return check_launch("linear_f16w");
    }
    if (m <= kLinearGemvRows) {
        size_t units4 = 0;
        for (int i = 0; i < nseg; ++i) units4 += (out_f[i] + kRowsPerWave - 1) / kRowsPerWave;
        const bool few = units4 < (size_t)kGemvOneRowUnits, longer = in_f > (size_t)kGemvShortRow;
        // Features per unit: a workgroup's (longer rows) or a wave's.
        const size_t per = longer ? (few || m > 4 ? 4 : 8) : (few ? 1 : kRowsPerWave);
        s.first[0] = 0;
        for (int i = 0; i < nseg; ++i) s.first[i + 1] = s.first[i] + (int)((out_f[i] + per - 1) / per);
        const unsigned units = (unsigned)s.first[nseg], blocks = (units + kWaves - 1) / kWaves;
        const int mi = (int)m, k = (int)in_f;
        if (longer && per == 4) launch_gemv_long<4>(units, st, x, s, mi, k);
        else if (longer) launch_gemv_long<8>(units, st, x, s, mi, k);
        else if (few) launch_gemv<1>(blocks, st, x, s, mi, k);
        else launch_gemv<kRowsPerWave>(blocks, st, x, s, mi, k);
        return check_launch("linear_f16w");
    }
    if (ws == nullptr || ws_floats < m) return fail(EB_SHAPE_MISMATCH, "linear: workspace too small");
    const size_t split = linear_split_workspace_floats(m, in_f);
    if (split > linear_workspace_floats(m, in_f) && ws_floats >= split && aligned16(ws))
        return launch_tiles(st, x, s, out_f, nseg, m, in_f, ws);
    // Without a workspace for the split rows.
    // Wide tiles (64 x 128 per wave: 0.5 LDS fragment reads per MFMA instead of 0.75) when
    // they still give every CU two workgroups; otherwise 128 x 128 tiles, whose twice as
    // many workgroups keep more of the chip busy. With at most one 128 x 128 tile per CU
    // (o_proj-like shapes: many rows, few features), long contractions are cut in two
    // halves, doubling the workgroups; the pre-pass then zeroes the outputs they add into.
    const size_t mtiles = (m + kBM - 1) / kBM;
    size_t wide_units = 0, units = 0;
    for (int i = 0; i < nseg; ++i) {
        wide_units += (out_f[i] + GemmShape<4>::BN - 1) / GemmShape<4>::BN;
        units += (out_f[i] + GemmShape<2>::BN - 1) / GemmShape<2>::BN;
    }
    const size_t cus = (size_t)current_cu_count();
    const bool wide = mtiles * wide_units >= 2 * cus;
    const int ksplit =
        (!wide && mtiles * units <= cus && in_f >= (size_t)EB_LINEAR_KSPLIT_MIN) ? 2 : 1;
    linear_row_scale_kernel<<<(unsigned)((m + kWaves - 1) / kWaves), kThreads, 0, st>>>(
        x, ws, (int)m, (int)in_f, s, ksplit > 1);
    if (wide) return launch_gemm<4, 1, 2>(st, x, ws, s, out_f, nseg, m, in_f);
    return launch_gemm<2, 2, 1>(st, x, ws, s, out_f, nseg, m, in_f, ksplit);
}

}  // namespace eb
