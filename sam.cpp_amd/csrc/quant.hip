// Activation staging (the per-call RHS packing of the mul_mat path), row
// quantizers in ggml wire format, and to_float / get_rows, for gfx950.
//
// Staging turns F32 activation rows into the fp16 MFMA A operand:
//   Q8_0 mode : value = fp16(to_float(q8_0 block) * 2^-e)  (Q8_0 weights)
//   Q8_K mode : value = fp16(to_float(q8_K block) * 2^-e)  (K-quant weights)
//   F16 mode  : value = fp16(x * 2^-e)
// where the Q8 blocks are bit-exact with ggml's CPU from_float for the
// weight's vec_dot_type (src/runtime/ggml/backends/cpu.hpp:13-23) and 2^e is
// a per-row power of two that keeps the row maximum inside fp16's range; the
// GEMM epilogue multiplies it back exactly.
#include <algorithm>

#include "internal.hpp"
#include "q8stage.hpp"

#pragma clang fp contract(off)

namespace samhip {

namespace {

// Staging with each lane owning 8 consecutive values (a Q8_0 block spans 4
// lanes, a Q8_K block 32 lanes).  The row stays in registers (K <= 512*CH),
// so X is read once; every cross-lane reduction runs with all lanes active
// (lanes past K hold zeros).
template <int MODE, int CH, bool X86, int PRE = PRE_NONE>
__device__ __forceinline__ void stage8_row(const float* __restrict__ x, int64_t x_stride, int m, int K, int kp,
                                           _Float16* __restrict__ a, int64_t lda, float* __restrict__ row_scale,
                                           int lane, const RowPre& pre = RowPre{}) {
    const float* xr = x + int64_t(m) * x_stride;
    floatx8 v[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int k = 512 * c + 8 * lane;
        if (k < K) {
            const floatx4 lo = load4f_stream(xr + k), hi = load4f_stream(xr + k + 4);
            v[c] = floatx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
            v[c] = floatx8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
    int64_t dst = m;
    if (PRE == PRE_GELU) {
        // the F32 erf-GELU of the producing graph node, before packing
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i) v[c][i] = gelu_erf(v[c][i]);   // gelu(0) = 0 keeps the padding
    } else if (PRE == PRE_LAYER_NORM) {
        // ggml_norm(x, eps) * w + b of the producing node, the row leaving in
        // window order when pre.ws > 0
        float s = 0.f;
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i) s += v[c][i];
        const float mean = wave_sum(s) / float(K);
        float s2 = 0.f;
        if (K == 512 * CH) {   // every lane's values lie in the row
#pragma unroll
            for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float d = v[c][i] - mean;
                    v[c][i] = d;
                    s2 += d * d;
                }
        } else {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const bool live = 512 * c + 8 * lane < K;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float d = live ? v[c][i] - mean : 0.f;
                    v[c][i] = d;
                    s2 += d * d;
                }
            }
        }
        const float variance = wave_sum(s2) / float(K);
        const float scale = 1.0f / sqrtf(variance + pre.eps);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int k = 512 * c + 8 * lane;
            if (k < K) {
                const floatx4 w0 = load4f(pre.w + k), w1 = load4f(pre.w + k + 4);
                const floatx4 b0 = load4f(pre.b + k), b1 = load4f(pre.b + k + 4);
                const floatx8 w{w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
                const floatx8 b{b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
#pragma unroll
                for (int i = 0; i < 8; ++i) v[c][i] = (v[c][i] * scale) * w[i] + b[i];
            }
        }
        if (pre.ws > 0) {
            const int gy = m / pre.gw, gx = m - gy * pre.gw;
            const int win = (gy / pre.ws) * (pre.gw / pre.ws) + gx / pre.ws;
            dst = int64_t(win) * pre.ws * pre.ws + (gy % pre.ws) * pre.ws + gx % pre.ws;
        }
    }
    // the blocks' extremes give the row's largest magnitude and, unless a
    // NaN, an infinity or a tie of signs sends the wave the ordered way, the
    // blocks' scales
    uint32_t ext[CH], top = 0;
    bool odd = false;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        ext[c] = quant8_extreme<MODE>(v[c], odd);
        top = umax(top, ext[c] & 0x7fffffffu);
    }
    _Float16* ar = a + dst * lda;
    if (!__any(odd)) {
        const int e = row_exponent(quant8_wave_max<MODE>(top));
        const float down = exp2i(-e);
        if (lane == 0) row_scale[dst] = exp2i(e);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int k = 512 * c + 8 * lane;
            float d = 0.f, mul = 0.f;
            if (MODE != T_F16) quant8_scale_of<MODE, X86>(ext[c], d, mul);
            const half8 o = quant8_operand<MODE, X86, false>(v[c], d, mul, down);
            if (k < kp) *reinterpret_cast<half8*>(ar + k) = o;   // lanes in [K, kp) hold zeros
        }
        return;
    }
    float rmax = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) rmax = fmaxf(rmax, fabsf(v[c][i]));
    const float r32 = max32_lanes(rmax);
    rmax = fmaxf(r32, __shfl_xor(r32, 32, 64));
    const int e = row_exponent(rmax);
    const float down = exp2i(-e);
    if (lane == 0) row_scale[dst] = exp2i(e);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int k = 512 * c + 8 * lane;
        float d = 0.f, mul = 0.f;
        if (MODE != T_F16) quant8_scale_ordered<MODE, X86>(v[c], lane, d, mul);
        const half8 o = quant8_operand<MODE, X86, true>(v[c], d, mul, down);
        if (k < kp) *reinterpret_cast<half8*>(ar + k) = o;
    }
}

// Rows of up to 5120 values (fc2's 4736), optionally through erf-GELU: two
// waves per row (values [0, 2560) and [2560, K)), the row maximum combined
// through LDS, so each wave holds half the row in registers and the
// workgroup stages two rows.  Every wave of the workgroup must call it (one
// barrier).  Measured against the alternatives at K = 4736: 39 us without
// a PRE (one wave per row, 97 VGPRs: 41 us), 42 us with the erf-GELU (a
// chunked pass parking the Q8 codes in LDS until the row maximum is known:
// 43-44 us).
template <int MODE, bool X86, int PRE>
__device__ __forceinline__ void stage8_half_row(const float* __restrict__ x, int64_t x_stride, int m, int M, int K, int kp,
                                                _Float16* __restrict__ a, int64_t lda, float* __restrict__ row_scale,
                                                int lane, int wave, float* pair_max) {
    constexpr int CHH = 5;
    const int half = wave & 1;
    const bool live = m < M;
    const float* xr = x + int64_t(live ? m : 0) * x_stride;
    floatx8 v[CHH];
#pragma unroll
    for (int c = 0; c < CHH; ++c) {
        const int k = 2560 * half + 512 * c + 8 * lane;
        if (live && k < K) {
            const floatx4 lo = load4f_stream(xr + k), hi = load4f_stream(xr + k + 4);
            v[c] = floatx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
            v[c] = floatx8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
    if (PRE == PRE_GELU)
#pragma unroll
        for (int c = 0; c < CHH; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i) v[c][i] = gelu_erf(v[c][i]);   // gelu(0) = 0 keeps the padding
    // as in stage8_row; the two halves meet on the largest magnitude
    uint32_t ext[CHH], top = 0;
    bool odd = false;
#pragma unroll
    for (int c = 0; c < CHH; ++c) {
        ext[c] = quant8_extreme<MODE>(v[c], odd);
        top = umax(top, ext[c] & 0x7fffffffu);
    }
    float rmax = quant8_wave_max<MODE>(top);
    odd = __any(odd);
    if (odd) {   // the largest magnitude without the NaNs
        rmax = 0.f;
#pragma unroll
        for (int c = 0; c < CHH; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i) rmax = fmaxf(rmax, fabsf(v[c][i]));
        const float r32 = max32_lanes(rmax);
        rmax = fmaxf(r32, __shfl_xor(r32, 32, 64));
    }
    if (lane == 0) pair_max[wave] = rmax;
    __syncthreads();
    rmax = fmaxf(pair_max[wave & ~1], pair_max[wave | 1]);
    const int e = row_exponent(rmax);
    const float down = exp2i(-e);
    if (live && half == 0 && lane == 0) row_scale[m] = exp2i(e);
    _Float16* ar = a + int64_t(live ? m : 0) * lda;
    if (odd) {
#pragma unroll
        for (int c = 0; c < CHH; ++c) {
            const int k = 2560 * half + 512 * c + 8 * lane;
            float d = 0.f, mul = 0.f;
            if (MODE != T_F16) quant8_scale_ordered<MODE, X86>(v[c], lane, d, mul);
            const half8 o = quant8_operand<MODE, X86, true>(v[c], d, mul, down);
            if (live && k < kp) *reinterpret_cast<half8*>(ar + k) = o;
        }
        return;
    }
#pragma unroll
    for (int c = 0; c < CHH; ++c) {
        const int k = 2560 * half + 512 * c + 8 * lane;
        float d = 0.f, mul = 0.f;
        if (MODE != T_F16) quant8_scale_of<MODE, X86>(ext[c], d, mul);
        const half8 o = quant8_operand<MODE, X86, false>(v[c], d, mul, down);
        if (live && k < kp) *reinterpret_cast<half8*>(ar + k) = o;
    }
}

template <int MODE, int CH, bool X86>
__global__ __launch_bounds__(256) void stage8_kernel(const float* __restrict__ x, int64_t x_stride, int M, int K, int kp,
                                                     _Float16* __restrict__ a, int64_t lda,
                                                     float* __restrict__ row_scale) {
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= M) return;
    stage8_row<MODE, CH, X86>(x, x_stride, m, K, kp, a, lda, row_scale, threadIdx.x & 63);
}

// thread t: half (t & 1) of 32-value step of one weight row -> 16 fp16
// values; the steps past K, up to kp, are zeros
template <int WT>
__device__ __forceinline__ void dequant_piece(const uint8_t* __restrict__ W, int64_t w_stride, int K, int kp,
                                              int64_t t, _Float16* __restrict__ out, int64_t ldo) {
    const int steps = kp / 32;
    const int h = int(t & 1);
    const int64_t rs = t >> 1;
    const int row = int(rs / steps), step = int(rs % steps);
    if (32 * step >= K) {   // Q8_0 rows only: a K-quant row ends on a multiple of 256
        half8* o = reinterpret_cast<half8*>(out + int64_t(row) * ldo + 32 * step + 16 * h);
        o[0] = o[1] = half8{0, 0, 0, 0, 0, 0, 0, 0};
        return;
    }
    WeightPiece<WT> piece;
    piece.load(W + int64_t(row) * w_stride, step, h);
    _Float16 v[16];
    piece.dequant(step, h, v);
    half8* o = reinterpret_cast<half8*>(out + int64_t(row) * ldo + 32 * step + 16 * h);
    o[0] = half8{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
    o[1] = half8{v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15]};
}

// Both per-call preparations of a tall product in one launch: workgroups
// [0, stage_blocks) pack four activation rows each, the rest decode 256
// weight pieces each (the two roles touch disjoint memory).
template <int MODE, int CH, bool X86, int WT, int PRE = PRE_NONE>
__global__ __launch_bounds__(256) void prep_kernel(const float* __restrict__ x, int64_t x_stride, int M, int K, int kp,
                                                   _Float16* __restrict__ a, int64_t lda, float* __restrict__ row_scale,
                                                   int stage_blocks, const uint8_t* __restrict__ W, int64_t w_stride,
                                                   int N, _Float16* __restrict__ wout, int64_t ldo, RowPre pre) {
    // rows past 2048 values without a layer norm: two waves per row
    constexpr bool PAIR = CH > 4 && (PRE == PRE_NONE || PRE == PRE_GELU);
    if constexpr (PAIR) {
        if (int(blockIdx.x) < stage_blocks) {
            __shared__ float pair_max[4];
            const int wave = threadIdx.x >> 6;
            stage8_half_row<MODE, X86, PRE>(x, x_stride, blockIdx.x * 2 + (wave >> 1), M, K, kp, a, lda, row_scale,
                                       threadIdx.x & 63, wave, pair_max);
            return;
        }
    }
    if (!PAIR && int(blockIdx.x) < stage_blocks) {
        const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
        if (m < M) {
            stage8_row<MODE, CH, X86, PRE>(x, x_stride, m, K, kp, a, lda, row_scale, threadIdx.x & 63, pre);
        }
        return;
    }
    const int64_t t = int64_t(blockIdx.x - stage_blocks) * 256 + threadIdx.x;
    if (t < int64_t(N) * (kp / 32) * 2) dequant_piece<WT>(W, w_stride, K, kp, t, wout, ldo);
}

// One wave per row, 4 rows per 256-thread block.
template <int MODE>
__global__ __launch_bounds__(256) void stage_rows_kernel(const float* __restrict__ x, int64_t x_stride, int M, int K, int kp,
                                                         _Float16* __restrict__ a, int64_t lda,
                                                         float* __restrict__ row_scale, int x86) {
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= M) return;
    const float* xr = x + int64_t(m) * x_stride;
    float rmax = 0.f;
    for (int k = 4 * lane; k < K; k += 256) {
        const floatx4 v = load4f(xr + k);
        rmax = fmaxf(rmax, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    }
    rmax = wave_max(rmax);
    const int e = row_exponent(rmax);
    const float down = exp2i(-e);
    if (lane == 0) row_scale[m] = exp2i(e);
    _Float16* ar = a + int64_t(m) * lda;
    for (int k = 4 * lane; k < K; k += 256) {
        const floatx4 v = load4f(xr + k);
        _Float16 out[4];
        if (MODE == T_F16) {
            for (int i = 0; i < 4; ++i) out[i] = (_Float16)(v[i] * down);
        } else {
            float d;
            int q[4];
            if (MODE == T_Q8_0) {
                q8_0_codes(v, x86, d, q);
                d = half_bits_to_float(float_to_half_bits(d));   // stored fp16 scale
            } else {
                q8_k_codes(v, lane, d, q);
            }
            const float dd = d * down;
            for (int i = 0; i < 4; ++i) out[i] = (_Float16)((float)q[i] * dd);
        }
        typedef _Float16 half4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<half4*>(ar + k) = half4{out[0], out[1], out[2], out[3]};
    }
    for (int k = K + lane; k < kp; k += 64) ar[k] = (_Float16)0.f;
}

// Weight rows -> fp16(to_float(W)) [N][K]: thread (row, 32-element step,
// half) writes 16 consecutive halves, so a wave stores 1 KB contiguously.
template <int WT>
__global__ __launch_bounds__(256) void dequant_w_f16_kernel(const uint8_t* __restrict__ W, int64_t w_stride, int N,
                                                            int K, int kp, _Float16* __restrict__ out, int64_t ldo) {
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t >= int64_t(N) * (kp / 32) * 2) return;
    dequant_piece<WT>(W, w_stride, K, kp, t, out, ldo);
}

// Scalar-load variant for rows that are not 16-byte aligned.
template <int MODE>
__global__ __launch_bounds__(256) void stage_rows_unaligned_kernel(const float* __restrict__ x, int64_t x_stride, int M,
                                                                   int K, int kp, _Float16* __restrict__ a, int64_t lda,
                                                                   float* __restrict__ row_scale, int x86) {
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= M) return;
    const float* xr = x + int64_t(m) * x_stride;
    auto load = [&](int k) { return floatx4{xr[k], xr[k + 1], xr[k + 2], xr[k + 3]}; };
    float rmax = 0.f;
    for (int k = 4 * lane; k < K; k += 256) {
        const floatx4 v = load(k);
        rmax = fmaxf(rmax, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    }
    rmax = wave_max(rmax);
    const int e = row_exponent(rmax);
    const float down = exp2i(-e);
    if (lane == 0) row_scale[m] = exp2i(e);
    _Float16* ar = a + int64_t(m) * lda;
    for (int k = 4 * lane; k < K; k += 256) {
        const floatx4 v = load(k);
        float d = 0.f;
        int q[4];
        if (MODE == T_Q8_0) {
            q8_0_codes(v, x86, d, q);
            d = half_bits_to_float(float_to_half_bits(d));
        } else if (MODE == T_Q8_K) {
            q8_k_codes(v, lane, d, q);
        }
        const float dd = d * down;
        for (int i = 0; i < 4; ++i)
            ar[k + i] = MODE == T_F16 ? (_Float16)(v[i] * down) : (_Float16)((float)q[i] * dd);
    }
    for (int k = K + lane; k < kp; k += 64) ar[k] = (_Float16)0.f;
}

// Q8_K rows in ggml wire format.  One wave per row.
__global__ __launch_bounds__(256) void quantize_q8_k_kernel(const float* __restrict__ x, int64_t x_stride, int rows,
                                                            int K, uint8_t* __restrict__ dst) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const float* xr = x + int64_t(r) * x_stride;
    uint8_t* out = dst + int64_t(r) * (K / 256) * 292;
    for (int k = 4 * lane; k < K; k += 256) {
        const floatx4 v = floatx4{xr[k], xr[k + 1], xr[k + 2], xr[k + 3]};
        float d;
        int q[4];
        q8_k_codes(v, lane, d, q);
        uint8_t* blk = out + (k / 256) * 292;
        const int within = k % 256;
        if (within == 0) *reinterpret_cast<float*>(blk) = d;
        for (int i = 0; i < 4; ++i) blk[4 + within + i] = uint8_t(int8_t(q[i]));
        const int s = group_sum<4>(q[0] + q[1] + q[2] + q[3]);
        if ((lane & 3) == 0) {
            const int16_t s16 = int16_t(s);
            blk[260 + 2 * (within / 16)] = uint8_t(uint16_t(s16) & 0xff);
            blk[260 + 2 * (within / 16) + 1] = uint8_t(uint16_t(s16) >> 8);
        }
    }
}

// Q8_0 rows in ggml wire format.  Packed rows follow one another without
// padding, so the kernel walks the blocks of all rows as one sequence: a wave
// takes 16 of them (8 values a lane, a block on a lane quad), puts their 544
// bytes together in LDS and stores them as dwords.  (With a wave per row and
// a store per code byte, the 34-byte blocks cost five stores a lane and 256
// values.)  Bound by HBM: 82 944 rows of 256 values 20.7 -> 16.8 us.
constexpr int kQ8WaveBlocks = 16, kQ8WaveBytes = 34 * kQ8WaveBlocks;

template <bool X86, bool XVEC>
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float* __restrict__ x, int64_t x_stride,
                                                            int64_t blocks, int nb, uint8_t* __restrict__ dst) {
    __shared__ __attribute__((aligned(16))) uint8_t buf[4][kQ8WaveBytes];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t first = (int64_t(blockIdx.x) * 4 + wave) * kQ8WaveBlocks;
    if (first >= blocks) return;   // (no barrier below: a wave's bytes are its own)
    const int i = lane >> 2;
    // lanes past the last block repeat it; their bytes are not stored
    const int64_t g = min(first + i, blocks - 1);
    const int64_t r = uint32_t(g) / uint32_t(nb);   // (a launch has at most 2^28 blocks)
    const float* xb = x + r * x_stride + 32 * (g - r * nb) + 8 * (lane & 3);
    floatx8 v;
    if (XVEC) {
        const floatx4 a = load4f(xb), c = load4f(xb + 4);
        v = floatx8{a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]};
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = xb[j];
    }
    // as quant8_icodes, except that a block of NaNs keeps a NaN scale
    float amax = fabsf(v[0]);
#pragma unroll
    for (int j = 1; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    amax = max4_lanes(amax);
    const float d = div127(amax);
    float mul;
    if (X86) mul = amax != 0.f ? 127.f / amax : 0.f;
    else mul = d != 0.f ? 1.f / d : 0.f;
    int q[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = cvt_i32_nan0(quant8_round<T_Q8_0, X86>(v[j] * mul));
    uint16_t* o = reinterpret_cast<uint16_t*>(buf[wave] + 34 * i);
    if ((lane & 3) == 0) o[0] = float_to_half_bits(d);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[1 + 4 * (lane & 3) + j] = uint16_t((q[2 * j] & 0xff) | ((q[2 * j + 1] & 0xff) << 8));
    wave_lds_handoff();   // 16-bit stores above, 32-bit loads below
    const int bytes = int(min(int64_t(kQ8WaveBlocks), blocks - first)) * 34;
    uint8_t* out = dst + first * 34;
    if (reinterpret_cast<uintptr_t>(dst) % 4 == 0) {
        for (int k = 4 * lane; k + 4 <= bytes; k += 256)
            *reinterpret_cast<uint32_t*>(out + k) = *reinterpret_cast<const uint32_t*>(buf[wave] + k);
        const int left = bytes & 3, at = bytes - left;
        if (lane < left) out[at + lane] = buf[wave][at + lane];
    } else {
        for (int k = lane; k < bytes; k += 64) out[k] = buf[wave][k];
    }
}

// to_float of values 4c .. 4c + 3 of a packed row (within one Q8_0 block,
// one Q4_K / Q5_K sub-block, one Q6_K half sub-block, one Q8_K block).
template <int TYPE>
__device__ __forceinline__ floatx4 dequant4(const uint8_t* row, int c) {
    floatx4 y;
    if (TYPE == T_F32) {
        const float* f = reinterpret_cast<const float*>(row) + 4 * c;
        y = floatx4{f[0], f[1], f[2], f[3]};
    } else if (TYPE == T_F16) {
        const uint32_t lo = load4_a2(row + 8 * int64_t(c)), hi = load4_a2(row + 8 * int64_t(c) + 4);
        y = floatx4{half_bits_to_float(lo & 0xffffu), half_bits_to_float(lo >> 16), half_bits_to_float(hi & 0xffffu),
                    half_bits_to_float(hi >> 16)};
    } else if (TYPE == T_Q8_0 || TYPE == T_Q8_K) {
        const uint8_t* b = TYPE == T_Q8_0 ? row + 34 * int64_t(c >> 3) : row + 292 * int64_t(c >> 6);
        const float d = TYPE == T_Q8_0 ? half_bits_to_float(load2_a2(b)) : __builtin_bit_cast(float, load4_a2(b));
        const uint32_t q = TYPE == T_Q8_0 ? load4_a2(b + 2 + 4 * (c & 7)) : load4_a2(b + 4 + 4 * (c & 63));
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = d * (float)(int8_t)(q >> (8 * i));
    } else if (TYPE == T_Q4_K || TYPE == T_Q5_K) {
        const uint8_t* b = row + (TYPE == T_Q4_K ? 144 : 176) * int64_t(c >> 6);
        const int j = (c >> 3) & 7, l = 4 * (c & 7);   // sub-block, first value in it
        const uint32_t sc[3] = {load4_a2(b + 4), load4_a2(b + 8), load4_a2(b + 12)};
        int s, m;
        k4_scale_min(j, sc, s, m);
        const uint32_t h = load4_a2(b);
        const float dj = half_bits_to_float(h & 0xffffu) * (float)s;
        const float mj = half_bits_to_float(h >> 16) * (float)m;
        uint32_t q = (load4_a2(b + (TYPE == T_Q4_K ? 16 : 48) + 32 * (j >> 1) + l) >> (4 * (j & 1))) & 0x0f0f0f0fu;
        if (TYPE == T_Q5_K) q |= ((load4_a2(b + 16 + l) >> j) & 0x01010101u) << 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = dj * (float)((q >> (8 * i)) & 0xffu) - mj;
    } else {
        const uint8_t* b = row + 210 * int64_t(c >> 6);
        const int j = (c >> 3) & 7, l = 4 * (c & 7), half = j >> 2, q4 = j & 3;
        const float ds = half_bits_to_float(load2_a2(b + 208)) * (float)(int8_t)b[192 + 8 * half + 2 * q4 + (l >> 4)];
        const uint32_t lo = (load4_a2(b + 64 * half + 32 * (q4 & 1) + l) >> (4 * (q4 >> 1))) & 0x0f0f0f0fu;
        const uint32_t q = lo | (((load4_a2(b + 128 + 32 * half + l) >> (2 * q4)) & 0x03030303u) << 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = ds * (float)(int((q >> (8 * i)) & 0xffu) - 32);
    }
    return y;
}

// A lane decodes four consecutive values, so a wave's stores are whole
// 1 KB runs of the row (VEC: 16 bytes a lane; a lane per 32 values left each
// lane storing its own 128 bytes).  A workgroup covers 256 such quads: whole
// rows while they are shorter than that, else one run of a row (grid y), and
// walks the rows in steps of the grid.  Bound by HBM: 82 944 rows of 256
// values from Q8_0 31.3 -> 17.5 us (6.1 TB/s, the values partly in the MALL).
template <int TYPE, bool VEC>
__global__ __launch_bounds__(256) void dequant_rows_kernel(const uint8_t* __restrict__ src, int64_t src_stride,
                                                           const int32_t* __restrict__ ids, int64_t src_rows,
                                                           float* __restrict__ dst, int64_t dst_stride, int rows,
                                                           int K, int* __restrict__ bad_id) {
    const unsigned quads = unsigned(K) / 4;
    const unsigned per = quads < 256 ? 256 / quads : 1;   // rows per workgroup
    const unsigned sub = quads < 256 ? threadIdx.x / quads : 0;
    const unsigned c = quads < 256 ? threadIdx.x - sub * quads : blockIdx.y * 256 + threadIdx.x;
    if (sub >= per || c >= quads) return;
    for (int64_t r = int64_t(blockIdx.x) * per + sub; r < rows; r += int64_t(gridDim.x) * per) {
        int64_t sr = r;
        if (ids) {
            sr = ids[r];
            if (sr < 0 || sr >= src_rows) {
                if (c == 0) *bad_id = 1;   // (host memory: a plain store, every writer's the same)
                continue;
            }
        }
        const floatx4 v = dequant4<TYPE>(src + sr * src_stride, int(c));
        float* y = dst + r * dst_stride + 4 * int64_t(c);
        if (VEC) {
            *reinterpret_cast<floatx4*>(y) = v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = v[i];
        }
    }
}

// Staging of a product whose activation rows arrive as Q8_0 codes and F32
// block maxima (Epilogue::q8 of the producing GEMM): the fp16 operand and
// row scale that staging the F32 rows gives, bit for bit, since the row
// maximum is the largest block maximum, the block scale fp16(amax / 127) and
// each value fp16(q * (d * 2^-e)).  One wave per row, four rows per
// workgroup; lane l takes values 8l .. 8l + 7 of each 512-value chunk.  The
// workgroups past stage_blocks decode the weight as prep_kernel's do.
template <int WT>
__global__ __launch_bounds__(256) void prep_codes_kernel(const int8_t* __restrict__ codes,
                                                         const float* __restrict__ amax, int64_t ldc, int M, int K,
                                                         _Float16* __restrict__ a, int64_t lda,
                                                         float* __restrict__ row_scale, int stage_blocks,
                                                         const uint8_t* __restrict__ W, int64_t w_stride, int N,
                                                         _Float16* __restrict__ wout, int64_t ldo) {
#pragma clang fp contract(off)
    if (int(blockIdx.x) < stage_blocks) {
        const int lane = threadIdx.x & 63;
        const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
        if (m >= M) return;
        const float* am = amax + int64_t(m) * (ldc >> 5);
        float rmax = 0.f;
        for (int b = lane; b < K / 32; b += 64) rmax = fmaxf(rmax, am[b]);
        rmax = wave_max(rmax);
        const int e = row_exponent(rmax);
        const float down = exp2i(-e);
        if (lane == 0) row_scale[m] = exp2i(e);
        const int8_t* cr = codes + int64_t(m) * ldc;
        _Float16* ar = a + int64_t(m) * lda;
        for (int k = 8 * lane; k < K; k += 512) {
            const u32x2 w = *reinterpret_cast<const u32x2*>(cr + k);
            const float dd = half_bits_to_float(float_to_half_bits(am[k >> 5] / 127.f)) * down;
            half8 o;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int q = int(int8_t(uint8_t(w[i >> 2] >> (8 * (i & 3)))));
                o[i] = (_Float16)(float(q) * dd);
            }
            *reinterpret_cast<half8*>(ar + k) = o;
        }
        return;
    }
    const int64_t t = int64_t(blockIdx.x - stage_blocks) * 256 + threadIdx.x;
    if (t < int64_t(N) * (K / 32) * 2) dequant_piece<WT>(W, w_stride, K, K, t, wout, ldo);
}

}  // namespace

void launch_dequant_w_f16(int wtype, const void* w, int64_t w_stride, int N, int K, int kp, _Float16* out,
                          int64_t ldo, hipStream_t stream) {
    const int64_t threads = int64_t(N) * (kp / 32) * 2;
    const dim3 grid(unsigned((threads + 255) / 256)), block(256);
    const uint8_t* wb = static_cast<const uint8_t*>(w);
    switch (wtype) {
        case T_Q8_0: hipLaunchKernelGGL(dequant_w_f16_kernel<T_Q8_0>, grid, block, 0, stream, wb, w_stride, N, K, kp, out, ldo); break;
        case T_Q4_K: hipLaunchKernelGGL(dequant_w_f16_kernel<T_Q4_K>, grid, block, 0, stream, wb, w_stride, N, K, kp, out, ldo); break;
        case T_Q5_K: hipLaunchKernelGGL(dequant_w_f16_kernel<T_Q5_K>, grid, block, 0, stream, wb, w_stride, N, K, kp, out, ldo); break;
        case T_Q6_K: hipLaunchKernelGGL(dequant_w_f16_kernel<T_Q6_K>, grid, block, 0, stream, wb, w_stride, N, K, kp, out, ldo); break;
        default: break;
    }
}

bool launch_prep(int mode, int wtype, const float* x, int64_t x_stride, int M, int K, int kp, _Float16* a, int64_t lda,
                 float* row_scale, int x86, const void* w, int64_t w_stride, int N, _Float16* wout, int64_t ldo,
                 hipStream_t stream, const RowPre& pre) {
    if (kp > 512 * 10 || reinterpret_cast<uintptr_t>(x) % 16 || x_stride % 4) return false;
    if (pre.kind == PRE_LAYER_NORM && (!pre.w || !pre.b || reinterpret_cast<uintptr_t>(pre.w) % 16 ||
                                       reinterpret_cast<uintptr_t>(pre.b) % 16 || K % 8))
        return false;
    const int64_t db = (int64_t(N) * (kp / 32) * 2 + 255) / 256;
    const dim3 block(256);
    const uint8_t* wb = static_cast<const uint8_t*>(w);
#define SAMHIP_PREP(MODE, CH, X86, WT)                                                                               \
    do {                                                                                                             \
        /* staging workgroups: four rows each, two for long rows with no PRE */                                    \
        const int sb = (CH > 4 && pre.kind != PRE_LAYER_NORM) ? (M + 1) / 2 : (M + 3) / 4;                                  \
        const dim3 grid(unsigned(sb + db));                                                                          \
        if (pre.kind == PRE_GELU)                                                                                    \
            hipLaunchKernelGGL((prep_kernel<MODE, CH, X86, WT, PRE_GELU>), grid, block, 0, stream, x, x_stride, M, K, \
                               kp, a, lda, row_scale, sb, wb, w_stride, N, wout, ldo, pre);                              \
        else if (pre.kind == PRE_LAYER_NORM)                                                                         \
            hipLaunchKernelGGL((prep_kernel<MODE, CH, X86, WT, PRE_LAYER_NORM>), grid, block, 0, stream, x, x_stride, \
                               M, K, kp, a, lda, row_scale, sb, wb, w_stride, N, wout, ldo, pre);                        \
        else                                                                                                         \
            hipLaunchKernelGGL((prep_kernel<MODE, CH, X86, WT>), grid, block, 0, stream, x, x_stride, M, K, kp, a, lda,  \
                               row_scale, sb, wb, w_stride, N, wout, ldo, pre);                                      \
    } while (0)
#define SAMHIP_PREP_CH(MODE, X86, WT)                    \
    do {                                                 \
        if (kp <= 1024) SAMHIP_PREP(MODE, 2, X86, WT);    \
        else if (kp <= 2048) SAMHIP_PREP(MODE, 4, X86, WT); \
        else SAMHIP_PREP(MODE, 10, X86, WT);             \
    } while (0)
    switch (wtype) {
        case T_Q8_0:
            if (mode == T_F16) SAMHIP_PREP_CH(T_F16, false, T_Q8_0);
            else if (x86) SAMHIP_PREP_CH(T_Q8_0, true, T_Q8_0);
            else SAMHIP_PREP_CH(T_Q8_0, false, T_Q8_0);
            break;
        case T_Q4_K:
            if (mode == T_F16) SAMHIP_PREP_CH(T_F16, false, T_Q4_K);
            else SAMHIP_PREP_CH(T_Q8_K, false, T_Q4_K);
            break;
        case T_Q5_K:
            if (mode == T_F16) SAMHIP_PREP_CH(T_F16, false, T_Q5_K);
            else SAMHIP_PREP_CH(T_Q8_K, false, T_Q5_K);
            break;
        case T_Q6_K:
            if (mode == T_F16) SAMHIP_PREP_CH(T_F16, false, T_Q6_K);
            else SAMHIP_PREP_CH(T_Q8_K, false, T_Q6_K);
            break;
        default: return false;
    }
#undef SAMHIP_PREP_CH
#undef SAMHIP_PREP
    return true;
}

bool launch_prep_codes(const int8_t* codes, const float* amax, int64_t ldc, int M, int K, _Float16* a, int64_t lda,
                       float* row_scale, int wtype, const void* w, int64_t w_stride, int N, _Float16* wout,
                       int64_t ldo, hipStream_t stream) {
    // 8-byte code loads and 16-byte operand stores
    if (wtype != T_Q8_0 || M < 1 || N < 1 || K < 32 || K % 32 || ldc % 32 || K > ldc || lda % 8 ||
        reinterpret_cast<uintptr_t>(codes) % 8 || reinterpret_cast<uintptr_t>(amax) % 4 ||
        reinterpret_cast<uintptr_t>(a) % 16)
        return false;
    const int sb = (M + 3) / 4;
    const int64_t db = (int64_t(N) * (K / 32) * 2 + 255) / 256;
    hipLaunchKernelGGL(prep_codes_kernel<T_Q8_0>, dim3(unsigned(sb + db)), dim3(256), 0, stream, codes, amax, ldc, M,
                       K, a, lda, row_scale, sb, static_cast<const uint8_t*>(w), w_stride, N, wout, ldo);
    return true;
}

void launch_stage_rows(int mode, bool aligned, const float* x, int64_t x_stride, int M, int K, int kp, _Float16* a,
                       int64_t lda, float* row_scale, int x86, hipStream_t stream) {
    const dim3 grid((M + 3) / 4), block(256);
    if (aligned && kp <= 512 * 10) {
#define SAMHIP_STAGE8(MODE, CH)                                                                                 \
    do {                                                                                                        \
        if (MODE == T_Q8_0 && x86)                                                                              \
            hipLaunchKernelGGL((stage8_kernel<MODE, CH, true>), grid, block, 0, stream, x, x_stride, M, K, kp, a, \
                               lda, row_scale);                                                                 \
        else                                                                                                    \
            hipLaunchKernelGGL((stage8_kernel<MODE, CH, false>), grid, block, 0, stream, x, x_stride, M, K, kp, a, \
                               lda, row_scale);                                                                 \
    } while (0)
#define SAMHIP_STAGE8_MODE(MODE)                  \
    if (kp <= 1024) SAMHIP_STAGE8(MODE, 2);       \
    else if (kp <= 2048) SAMHIP_STAGE8(MODE, 4);   \
    else SAMHIP_STAGE8(MODE, 10);
        switch (mode) {
            case T_F16: SAMHIP_STAGE8_MODE(T_F16) break;
            case T_Q8_0: SAMHIP_STAGE8_MODE(T_Q8_0) break;
            case T_Q8_K: SAMHIP_STAGE8_MODE(T_Q8_K) break;
            default: break;
        }
#undef SAMHIP_STAGE8_MODE
#undef SAMHIP_STAGE8
        return;
    }
#define SAMHIP_STAGE(MODE)                                                                                      \
    if (aligned) hipLaunchKernelGGL(stage_rows_kernel<MODE>, grid, block, 0, stream, x, x_stride, M, K, kp, a, lda, \
                                    row_scale, x86);                                                           \
    else hipLaunchKernelGGL(stage_rows_unaligned_kernel<MODE>, grid, block, 0, stream, x, x_stride, M, K, kp, a, lda, \
                            row_scale, x86);
    switch (mode) {
        case T_F16: SAMHIP_STAGE(T_F16) break;
        case T_Q8_0: SAMHIP_STAGE(T_Q8_0) break;
        case T_Q8_K: SAMHIP_STAGE(T_Q8_K) break;
        default: break;
    }
#undef SAMHIP_STAGE
}

// F32 -> F16 rows (ggml_cast to F16: round to nearest even, overflow to inf).
__global__ __launch_bounds__(256) void cast_f16_kernel(const float* __restrict__ x, int64_t x_stride, int rows, int K,
                                                       _Float16* __restrict__ dst) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= int64_t(rows) * K) return;
    const int64_t r = i / K, c = i - r * K;
    dst[i] = (_Float16)x[r * x_stride + c];
}

void launch_cast_f16(const float* x, int64_t x_stride, int rows, int K, _Float16* dst, hipStream_t stream) {
    const int64_t n = int64_t(rows) * K;
    hipLaunchKernelGGL(cast_f16_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, stream, x, x_stride, rows, K,
                       dst);
}

void launch_quantize_act(int type, const float* x, int64_t x_stride, int rows, int K, void* dst, int x86,
                         hipStream_t stream) {
    uint8_t* d = static_cast<uint8_t*>(dst);
    if (type != T_Q8_0) {
        hipLaunchKernelGGL(quantize_q8_k_kernel, dim3((rows + 3) / 4), dim3(256), 0, stream, x, x_stride, rows, K, d);
        return;
    }
    const int nb = K / 32;
    const bool xvec = reinterpret_cast<uintptr_t>(x) % 16 == 0 && x_stride % 4 == 0;
    // (a dispatch counts its work-items in 32 bits: four per block here)
    const int step = int(std::max<int64_t>(1, (int64_t(1) << 28) / nb));
    for (int64_t r0 = 0; r0 < rows; r0 += step) {
        const int64_t blocks = std::min<int64_t>(step, rows - r0) * nb;
        const dim3 grid(unsigned((blocks + 4 * kQ8WaveBlocks - 1) / (4 * kQ8WaveBlocks)));
        const float* xs = x + r0 * x_stride;
        uint8_t* ds = d + r0 * nb * 34;
#define SAMHIP_Q8_0(X86, XVEC) \
    hipLaunchKernelGGL((quantize_q8_0_kernel<X86, XVEC>), grid, dim3(256), 0, stream, xs, x_stride, blocks, nb, ds)
        if (x86 && xvec) SAMHIP_Q8_0(true, true);
        else if (x86) SAMHIP_Q8_0(true, false);
        else if (xvec) SAMHIP_Q8_0(false, true);
        else SAMHIP_Q8_0(false, false);
#undef SAMHIP_Q8_0
    }
}

// ---------------------------------------------------------------------------
// ggml-cuda's right-operand formats and the native-activation range rule.
// One lane per value, 32 lanes (half a wave) per 32-value block, so every
// reduction stays inside a lane group and whole groups leave together.
// ---------------------------------------------------------------------------

// 1 when a block of F32 values is outside the native activation's range:
// a non-finite value, or a nonzero block maximum outside [1e-30, 1e30],
// compared as bit patterns so subnormals are not flushed
// (cmake/patches/ggml-native-activation.patch:148-171).
__device__ __forceinline__ bool block_out_of_range(float v) {
    uint32_t bits = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
    uint32_t bad = bits >= 0x7f800000u;
    for (int off = 16; off > 0; off >>= 1) {
        bits = max(bits, uint32_t(__shfl_xor(int(bits), off, 32)));
        bad |= uint32_t(__shfl_xor(int(bad), off, 32));
    }
    constexpr uint32_t lower = 0x0da24260u, upper = 0x7149f2cau;   // bits of 1e-30f, 1e30f
    return bad || bits > upper || (bits != 0 && bits < lower);
}

__device__ __forceinline__ float group32_absmax(float v) {
    float a = fabsf(v);
    for (int off = 16; off > 0; off >>= 1) a = fmaxf(a, __shfl_xor(a, off, 32));
    return a;
}

// quantize_q8_1 (MMVQ right operand): d = amax/127, q = roundf(x/d), half d
// and half of the original values' sum in the 32-lane xor-butterfly order.
__global__ __launch_bounds__(256) void quantize_q8_1_kernel(const float* __restrict__ x, int64_t x_stride, int rows,
                                                            int K, uint8_t* __restrict__ dst) {
#pragma clang fp contract(off)
    const int64_t nb = K / 32;
    const int64_t blk = (int64_t(blockIdx.x) * 256 + threadIdx.x) >> 5;
    const int lane = threadIdx.x & 31;
    if (blk >= int64_t(rows) * nb) return;
    const int64_t r = blk / nb, b = blk - r * nb;
    const float v = x[r * x_stride + b * 32 + lane];
    const float amax = group32_absmax(v);
    float s = v;
    for (int off = 16; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 32);
    const float d = amax / 127.f;
    const float qr = amax == 0.f ? 0.f : __builtin_roundf(v / d);
    const float q = qr == qr ? qr : 0.f;   // NaN -> code 0
    uint8_t* out = dst + blk * 36;
    out[4 + lane] = uint8_t(int8_t(q));
    if (lane == 0) {
        *reinterpret_cast<uint16_t*>(out) = float_to_half_bits(d);
        *reinterpret_cast<uint16_t*>(out + 2) = float_to_half_bits(s);
    }
}

// quantize_mmq_q8_1, D4 layout, for Q8_0 products: rows padded with zeros to
// kp (a multiple of 512) values, tile t of 128 values of row r at
// dst + (t*rows + r)*144 = 4 F32 scales, then 128 codes.  d_inv = 127/amax
// correctly rounded, q = roundf(x*d_inv), scale 1/d_inv.  Blocks outside the
// native range set *invalid.
__global__ __launch_bounds__(256) void quantize_q8_1_mmq_kernel(const float* __restrict__ x, int64_t x_stride,
                                                                int rows, int K, int kp, uint8_t* __restrict__ dst,
                                                                int* __restrict__ invalid) {
#pragma clang fp contract(off)
    const int64_t nb = kp / 32;
    const int64_t blk = (int64_t(blockIdx.x) * 256 + threadIdx.x) >> 5;
    const int lane = threadIdx.x & 31;
    if (blk >= int64_t(rows) * nb) return;
    const int64_t r = blk / nb, kb = blk - r * nb;
    const int64_t k = kb * 32 + lane;
    const float v = k < K ? x[r * x_stride + k] : 0.f;
    if (block_out_of_range(v) && lane == 0) atomicOr(invalid, 1);
    const float amax = group32_absmax(v);
    float q = 0.f, d = 0.f;
    if (amax != 0.f) {
        const float d_inv = 127.f / amax;
        const float r = __builtin_roundf(v * d_inv);
        q = r == r ? r : 0.f;   // NaN -> code 0 (such blocks also raise *invalid)
        d = 1.f / d_inv;
    }
    uint8_t* out = dst + ((kb >> 2) * rows + r) * 144;
    out[16 + 32 * (kb & 3) + lane] = uint8_t(int8_t(q));
    if (lane == 0) *reinterpret_cast<float*>(out + 4 * (kb & 3)) = d;
}

// The range rule alone over F32 rows (mul_mat's opt-in activation check).
__global__ __launch_bounds__(256) void q8_rhs_check_kernel(const float* __restrict__ x, int64_t x_stride, int rows,
                                                           int K, int* __restrict__ invalid) {
    const int64_t nb = K / 32;
    const int64_t blk = (int64_t(blockIdx.x) * 256 + threadIdx.x) >> 5;
    const int lane = threadIdx.x & 31;
    if (blk >= int64_t(rows) * nb) return;
    const int64_t r = blk / nb, b = blk - r * nb;
    if (block_out_of_range(x[r * x_stride + b * 32 + lane]) && lane == 0) atomicOr(invalid, 1);
}

void launch_quantize_q8_1(const float* x, int64_t x_stride, int rows, int K, void* dst, hipStream_t stream) {
    const int64_t lanes = int64_t(rows) * K;
    hipLaunchKernelGGL(quantize_q8_1_kernel, dim3(unsigned((lanes + 255) / 256)), dim3(256), 0, stream, x, x_stride,
                       rows, K, static_cast<uint8_t*>(dst));
}

void launch_quantize_q8_1_mmq(const float* x, int64_t x_stride, int rows, int K, void* dst, int* invalid,
                              hipStream_t stream) {
    const int kp = (K + 511) / 512 * 512;
    const int64_t lanes = int64_t(rows) * kp;
    hipLaunchKernelGGL(quantize_q8_1_mmq_kernel, dim3(unsigned((lanes + 255) / 256)), dim3(256), 0, stream, x,
                       x_stride, rows, K, kp, static_cast<uint8_t*>(dst), invalid);
}

void launch_q8_rhs_check(const float* x, int64_t x_stride, int rows, int K, int* invalid, hipStream_t stream) {
    const int64_t lanes = int64_t(rows) * K;
    hipLaunchKernelGGL(q8_rhs_check_kernel, dim3(unsigned((lanes + 255) / 256)), dim3(256), 0, stream, x, x_stride,
                       rows, K, invalid);
}

void launch_dequant_rows(int type, const void* src, int64_t src_stride, const int32_t* ids, int64_t src_rows,
                         float* dst, int64_t dst_stride, int rows, int K, int* bad_id, hipStream_t stream) {
    const int64_t quads = K / 4, per = quads < 256 ? 256 / quads : 1;
    // enough workgroups for every CU to hold its eight; each takes further rows
    const int64_t cols = (quads + 255) / 256;
    const int64_t groups = std::min<int64_t>((rows + per - 1) / per, std::max<int64_t>(1, 16384 / cols));
    const dim3 grid{unsigned(groups), unsigned(cols)}, block(256);
    const uint8_t* s = static_cast<const uint8_t*>(src);
    const bool vec = reinterpret_cast<uintptr_t>(dst) % 16 == 0 && dst_stride % 4 == 0;
#define SAMHIP_DQ(T)                                                                                                  \
    if (vec)                                                                                                          \
        hipLaunchKernelGGL((dequant_rows_kernel<T, true>), grid, block, 0, stream, s, src_stride, ids, src_rows, dst, \
                           dst_stride, rows, K, bad_id);                                                              \
    else                                                                                                              \
        hipLaunchKernelGGL((dequant_rows_kernel<T, false>), grid, block, 0, stream, s, src_stride, ids, src_rows,     \
                           dst, dst_stride, rows, K, bad_id)
    switch (type) {
        case T_F32: SAMHIP_DQ(T_F32); break;
        case T_F16: SAMHIP_DQ(T_F16); break;
        case T_Q8_0: SAMHIP_DQ(T_Q8_0); break;
        case T_Q4_K: SAMHIP_DQ(T_Q4_K); break;
        case T_Q5_K: SAMHIP_DQ(T_Q5_K); break;
        case T_Q6_K: SAMHIP_DQ(T_Q6_K); break;
        case T_Q8_K: SAMHIP_DQ(T_Q8_K); break;
        default: break;
    }
#undef SAMHIP_DQ
}

}  // namespace samhip
