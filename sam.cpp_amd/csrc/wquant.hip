// K-quant weight packing on the device: ggml_quantize_chunk for Q4_K, Q5_K
// and Q6_K without importance weights, i.e. quantize_row_q{4,5,6}_K_ref
// (the path tools/quantize/quantize_rows.cpp:210 takes to pack SAM weights).
// One lane packs one sub-block with the same serial scale search ggml runs on
// the CPU; contraction is disabled and division/sqrt are
// correctly rounded so the bytes match the CPU packer exactly.
#include "internal.hpp"

#pragma clang fp contract(off)

namespace samhip {

namespace {

__device__ __forceinline__ int round_even(float v) { return int(__builtin_rintf(v)); }

// The integer nearest to v in [0, nmax], and in [-32, 31], as a float: what
// converting to int and clamping gives, for a NaN too (0; v_med3_f32 then
// takes its other operands' minimum).  A -0 makes no difference to the sums.
__device__ __forceinline__ float code_asym(float v, float nmax) {
    return __builtin_amdgcn_fmed3f(__builtin_rintf(v), 0.f, nmax);
}
__device__ __forceinline__ float code_sym(float v) {
    const float r = __builtin_rintf(v);
    return __builtin_amdgcn_fmed3f(r == r ? r : 0.f, -32.f, 31.f);
}

__device__ __forceinline__ float half_round(float v) { return half_bits_to_float(float_to_half_bits(v)); }

// Weighted asymmetric fit of a sub-block's 32 values to [0, nmax] (see the
// CPU restatement).  The codes themselves are not kept: trial codes follow
// from (iscale, base), those of the best trial.
struct AsymFit {
    float scale, neg_min;
    float iscale, base;   // code i = round(iscale * (x[i] - base)) clamped; iscale 0: every code 0
};

template <int NMAX, int NSTEP>
__device__ __forceinline__ AsymFit fit_scale_min(const float (&x)[32], const float (&w)[32], float rmin) {
    constexpr float nmax = NMAX;
    float lo = x[0], hi = x[0];
    float sum_w = w[0], sum_x = w[0] * x[0];
#pragma unroll
    for (int i = 1; i < 32; ++i) {
        if (x[i] < lo) lo = x[i];
        if (x[i] > hi) hi = x[i];
        sum_w += w[i];
        sum_x += w[i] * x[i];
    }
    if (lo > 0) lo = 0;
    AsymFit f;
    if (hi == lo) {
        f.scale = 0.f;
        f.neg_min = -lo;
        f.iscale = 0.f;
        f.base = 0.f;
        return f;
    }
    f.iscale = nmax / (hi - lo);
    f.base = lo;
    f.scale = 1 / f.iscale;
    float best = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const float l = code_asym(f.iscale * (x[i] - lo), nmax);
        const float diff = f.scale * l + lo - x[i];
        best += w[i] * diff * diff;
    }
#pragma unroll 1
    for (int step = 0; step <= NSTEP; ++step) {
        const float iscale = (rmin + 0.1f * step + nmax) / (hi - lo);
        float sum_l = 0, sum_l2 = 0, sum_xl = 0;
        float l[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            l[i] = code_asym(iscale * (x[i] - lo), nmax);
            const float wl = w[i] * l[i];
            sum_l += wl;
            sum_l2 += wl * l[i];
            sum_xl += wl * x[i];
        }
        const float det = sum_w * sum_l2 - sum_l * sum_l;
        if (det > 0) {
            float this_scale = (sum_w * sum_xl - sum_x * sum_l) / det;
            float this_min = (sum_l2 * sum_x - sum_l * sum_xl) / det;
            if (this_min > 0) {
                this_min = 0;
                this_scale = sum_xl / sum_l2;
            }
            float err = 0;
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const float diff = this_scale * l[i] + this_min - x[i];
                err += w[i] * diff * diff;
            }
            if (err < best) {
                f.iscale = iscale;
                f.base = lo;
                best = err;
                f.scale = this_scale;
                lo = this_min;
            }
        }
    }
    f.neg_min = -lo;
    return f;
}

// Symmetric fit of 16 values to [-32, 31] with x^2 weights, 19 candidates;
// code i = round(best_iscale * x[i]) clamped to the range, of the best one;
// `tiny` values all get code 0.
__device__ __forceinline__ float fit_scale_sym16(const float (&x)[16], float& best_iscale, bool& tiny) {
    constexpr float nmax = 32.f;
    float amax = 0, smax = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float a = fabsf(x[i]);
        if (a > amax) { amax = a; smax = x[i]; }
    }
    best_iscale = 0.f;
    tiny = amax < 1e-15f;
    if (tiny) return 0.f;
    float iscale = -nmax / smax;
    float sum_lx = 0, sum_l2 = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float l = code_sym(iscale * x[i]);
        const float w = x[i] * x[i];
        sum_lx += w * x[i] * l;
        sum_l2 += w * l * l;
    }
    float scale = sum_l2 ? sum_lx / sum_l2 : 0.f;
    float best = scale * sum_lx;
    best_iscale = iscale;
#pragma unroll 1
    for (int step = -9; step <= 9; ++step) {
        if (step == 0) continue;
        iscale = -(nmax + 0.1f * step) / smax;
        sum_lx = sum_l2 = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float l = code_sym(iscale * x[i]);
            const float w = x[i] * x[i];
            sum_lx += w * x[i] * l;
            sum_l2 += w * l * l;
        }
        if (sum_l2 > 0 && sum_lx * sum_lx > best * sum_l2) {
            best_iscale = iscale;
            scale = sum_lx / sum_l2;
            best = scale * sum_lx;
        }
    }
    return scale;
}

// Four codes (small non-negative floats) in the bytes of a dword.
__device__ __forceinline__ uint32_t code_bytes(float a, float b, float c, float d) {
    return uint32_t(a) | (uint32_t(b) << 8) | (uint32_t(c) << 16) | (uint32_t(d) << 24);
}

__device__ __forceinline__ uint32_t lane_xor(uint32_t v, int mask) { return uint32_t(__shfl_xor(int(v), mask, 64)); }

// A lane packs one sub-block (32 values of Q4_K / Q5_K, 16 of Q6_K), so the
// 8 or 16 lanes of a super-block meet only for the super-block's scales and
// the packed bytes, and each sum keeps ggml's serial order.  The scale
// search bounds it: 21 (16, 18) trials of 32 (16) values at 16 (10) VALU
// operations each, ~12k instructions per wave, with the values, weights and
// trial codes in registers.  4736 x 1024 values take 56 us (Q4_K), 49 (Q5_K)
// and 31 (Q6_K); with one lane per super-block, which left three quarters of
// the SIMDs without a wave and kept the codes in scratch, 243, 292 and 166.
// A wave's super-blocks are contiguous in dst; they are assembled in LDS and
// leave as whole dwords when dst allows it.
template <int TYPE>
__global__ __launch_bounds__(64) void quantize_weights_kernel(const float* __restrict__ x, int64_t x_stride, int rows,
                                                              int K, uint8_t* __restrict__ dst) {
    constexpr int BB = block_bytes(TYPE);
    constexpr int SUB = TYPE == T_Q6_K ? 16 : 32, LANES = 256 / SUB, PER = 64 / LANES;
    __shared__ __attribute__((aligned(16))) uint8_t buf[PER * BB];
    const int nb = K / 256;
    const int64_t total = int64_t(rows) * nb, first = int64_t(blockIdx.x) * PER;
    const int lane = threadIdx.x, slot = lane / LANES, j = lane % LANES;
    // lanes past the last super-block repeat it; their bytes are not stored
    const int64_t t = min(first + slot, total - 1);
    const int64_t r = t / nb;
    const float* xb = x + r * x_stride + 256 * (t - r * nb) + SUB * j;
    uint8_t* out = buf + slot * BB;
    float v[SUB];
    if (reinterpret_cast<uintptr_t>(x) % 16 == 0 && x_stride % 4 == 0) {
#pragma unroll
        for (int i = 0; i < SUB; i += 4) {
            const floatx4 q = *reinterpret_cast<const floatx4*>(xb + i);
            v[i] = q[0], v[i + 1] = q[1], v[i + 2] = q[2], v[i + 3] = q[3];
        }
    } else {
#pragma unroll
        for (int i = 0; i < SUB; ++i) v[i] = xb[i];
    }
    if constexpr (TYPE == T_Q4_K || TYPE == T_Q5_K) {
        constexpr int NMAX = TYPE == T_Q4_K ? 15 : 31;
        float sum_x2 = 0;
#pragma unroll
        for (int i = 0; i < 32; ++i) sum_x2 += v[i] * v[i];
        const float av_x = __builtin_sqrtf(sum_x2 / 32);
        float w[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) w[i] = av_x + fabsf(v[i]);
        const AsymFit f = TYPE == T_Q4_K ? fit_scale_min<NMAX, 20>(v, w, -1.f) : fit_scale_min<NMAX, 15>(v, w, -0.5f);
        // the super-block's largest scale and min (a NaN never wins)
        float max_scale = __builtin_fmaxf(f.scale, 0.f), max_min = __builtin_fmaxf(f.neg_min, 0.f);
#pragma unroll
        for (int m = 1; m < 8; m <<= 1) {
            max_scale = __builtin_fmaxf(max_scale, __shfl_xor(max_scale, m, 64));
            max_min = __builtin_fmaxf(max_min, __shfl_xor(max_min, m, 64));
        }
        const float inv_scale = max_scale > 0 ? 63.f / max_scale : 0.f;
        const float inv_min = max_min > 0 ? 63.f / max_min : 0.f;
        uint32_t ls = uint8_t(round_even(inv_scale * f.scale));
        uint32_t lm = uint8_t(round_even(inv_min * f.neg_min));
        ls = ls < 63 ? ls : 63;
        lm = lm < 63 ? lm : 63;
        const uint32_t ls4 = lane_xor(ls, 4), lm4 = lane_xor(lm, 4);   // sub-block j ^ 4's
        if (j < 4) {
            out[4 + j] = uint8_t(ls | ((ls4 >> 4) << 6));
            out[8 + j] = uint8_t(lm | ((lm4 >> 4) << 6));
        } else {
            out[8 + j] = uint8_t((ls & 0x0f) | ((lm & 0x0f) << 4));
        }
        const float hd = max_scale / 63.f, hm = max_min / 63.f;
        if (j == 0)
            *reinterpret_cast<uint32_t*>(out) = uint32_t(float_to_half_bits(hd)) | (uint32_t(float_to_half_bits(hm)) << 16);
        const float dj = half_round(hd) * int(ls), mj = half_round(hm) * int(lm);
        float c[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            // scale 0: the codes of the fit
            c[i] = code_asym(dj != 0.f ? (v[i] + mj) / dj : f.iscale * (v[i] - f.base), float(NMAX));
        }
        // the pair of sub-blocks 2c, 2c + 1 shares 32 bytes (low and high
        // nibbles): the even lane writes the first 16, the odd the rest
        constexpr int QS = TYPE == T_Q4_K ? 16 : 48;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t a = code_bytes(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]);
            const uint32_t b = code_bytes(c[16 + 4 * q], c[17 + 4 * q], c[18 + 4 * q], c[19 + 4 * q]);
            const uint32_t na = a & 0x0f0f0f0fu, nb4 = b & 0x0f0f0f0fu;
            const uint32_t pa = lane_xor(na, 1), pb = lane_xor(nb4, 1);
            reinterpret_cast<uint32_t*>(out + QS + 32 * (j >> 1))[(j & 1) * 4 + q] =
                (j & 1) ? pb | (nb4 << 4) : na | (pa << 4);
            if (TYPE == T_Q5_K) {   // bit j of byte l: sub-block j's fifth bit of value l
                uint32_t ha = ((a >> 4) & 0x01010101u) << j, hb = ((b >> 4) & 0x01010101u) << j;
#pragma unroll
                for (int m = 1; m < 8; m <<= 1) {
                    ha |= lane_xor(ha, m);
                    hb |= lane_xor(hb, m);
                }
                if (j < 2) reinterpret_cast<uint32_t*>(out + 16)[j * 4 + q] = j ? hb : ha;
            }
        }
    } else {
        float fit;
        bool tiny;
        const float scale = fit_scale_sym16(v, fit, tiny);
        // the first scale of largest magnitude among the 16 (a NaN never wins)
        const float mag = fabsf(scale);
        float max_abs = __builtin_fmaxf(mag, 0.f);
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) max_abs = __builtin_fmaxf(max_abs, __shfl_xor(max_abs, m, 64));
        const uint32_t hits = uint32_t(__ballot(mag == max_abs) >> (16 * slot)) & 0xffffu;
        const float max_scale = __shfl(scale, 16 * slot + (hits ? __builtin_ctz(hits) : 0), 64);
        const bool zero = max_abs < 1e-15f;
        const float iscale = -128.f / max_scale;
        const float hd = 1 / iscale;
        const int sv = round_even(iscale * scale);
        const int8_t sc = int8_t(sv < 127 ? sv : 127);
        const float ds = half_round(hd) * sc;
        uint32_t code[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float c[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // scale 0: the codes of the fit
                c[i] = ds == 0.f && tiny ? 0.f : code_sym(ds != 0.f ? v[4 * q + i] / ds : fit * v[4 * q + i]) + 32.f;
            }
            code[q] = zero ? 0u : code_bytes(c[0], c[1], c[2], c[3]);
        }
        // sub-block s = j % 8 of half h = j / 8: low nibbles of s < 4 pair
        // with s + 4's; the four s of equal parity share the high bits' bytes
        const int s = j & 7, h = j >> 3;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t lo = code[q] & 0x0f0f0f0fu;
            const uint32_t word = lo | (lane_xor(lo, 4) << 4);
            uint32_t hi = ((code[q] >> 4) & 0x03030303u) << (2 * (s >> 1));
            hi |= lane_xor(hi, 2);
            hi |= lane_xor(hi, 4);
            // (a 210-byte block is 2-byte aligned)
            uint16_t* ql = reinterpret_cast<uint16_t*>(out + 64 * h + 16 * s + 4 * q);
            uint16_t* qh = reinterpret_cast<uint16_t*>(out + 128 + 32 * h + 16 * s + 4 * q);
            if (s < 4) {
                ql[0] = uint16_t(word);
                ql[1] = uint16_t(word >> 16);
            }
            if (s < 2) {
                qh[0] = uint16_t(hi);
                qh[1] = uint16_t(hi >> 16);
            }
        }
        out[192 + j] = zero ? 0 : uint8_t(sc);
        if (j == 0) *reinterpret_cast<uint16_t*>(out + 208) = zero ? uint16_t(0) : float_to_half_bits(hd);
    }
    __syncthreads();
    const int bytes = int(min(int64_t(PER), total - first)) * BB;
    uint8_t* o = dst + first * BB;
    if (reinterpret_cast<uintptr_t>(o) % 4 == 0) {
        for (int i = 4 * lane; i + 4 <= bytes; i += 256)
            *reinterpret_cast<uint32_t*>(o + i) = *reinterpret_cast<const uint32_t*>(buf + i);
        if (lane < bytes % 4) o[bytes - bytes % 4 + lane] = buf[bytes - bytes % 4 + lane];
    } else {
        for (int i = lane; i < bytes; i += 64) o[i] = buf[i];
    }
}

}  // namespace

void launch_quantize_weights(int type, const float* x, int64_t x_stride, int rows, int K, void* dst,
                             hipStream_t stream) {
    const int per = type == T_Q6_K ? 4 : 8;   // super-blocks per wave
    const int64_t blocks = int64_t(rows) * (K / 256);
    const dim3 grid(unsigned((blocks + per - 1) / per)), block(64);
    uint8_t* d = static_cast<uint8_t*>(dst);
    switch (type) {
        case T_Q4_K: hipLaunchKernelGGL(quantize_weights_kernel<T_Q4_K>, grid, block, 0, stream, x, x_stride, rows, K, d); break;
        case T_Q5_K: hipLaunchKernelGGL(quantize_weights_kernel<T_Q5_K>, grid, block, 0, stream, x, x_stride, rows, K, d); break;
        case T_Q6_K: hipLaunchKernelGGL(quantize_weights_kernel<T_Q6_K>, grid, block, 0, stream, x, x_stride, rows, K, d); break;
        default: break;
    }
}

}  // namespace samhip
