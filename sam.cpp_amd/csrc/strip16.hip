// Exact int8 products of Q4_K and Q5_K weights below 256 activation rows and
// past one super-block of K (the text encoder's 32 tokens), in two launches:
// one packs the activation rows once, in the order in which the matrix cores
// read them, and the product's workgroups then take the whole K range each.
//
//   pack : 32 lanes of 8 values per row and 256 values, ggml's quantize_row
//          to Q8_K.  Codes in MFMA operand order [row tile of 16][32-value
//          step][lane][8 bytes], the blocks' scales and the code sums of the
//          weight's sub-blocks, 16 rows each.
//   strip: a workgroup of NW waves per 16 weight rows and 16 T activation
//          rows.  A wave takes runs of U pairs of 32-value steps of one
//          super-block; a pair shares its bytes (low and high nibbles), a run
//          the header, and no two waves read the same codes, so both operands
//          go from memory to registers without LDS.  A load of a wave touches
//          16 weight rows, 16 cache lines: runs are as long as the waves
//          allow (K = 4096: a super-block each; with a header per pair the
//          product took 10.1 us against 8.6).  Per step and tile of
//          activation rows one v_mfma_i32_16x16x32_i8, then
//            acc += d_x ((d sc_j) dot - (dmin m_j) sum(codes_j))
//          in F32, as in the strip kernel of one launch (skinny.hip).  The
//          waves' partial tiles are added in LDS in wave order.
//
// Bound by latency: two launches, a trip of the weight from HBM, the VALU
// steps per block.  The text encoder's 97 Q4_K products as a replayed graph:
// 882 -> 772 us (836 -> 690 back to back), against workgroups that each packed
// the activation slice (128 KB of F32 rows at K = 1024) and left K-split
// partial sums for a reduction.  Not kept: workgroups beside the packing that
// read the weight ahead into the same XCD's L2 (742 against 729 us at that
// point), 8 waves with longer runs at K = 1024 (level), 4 (+6 %).
#include <algorithm>

#include "internal.hpp"
#include "q8stage.hpp"

namespace samhip {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Byte offsets of the packed activations: codes, then block scales, then
// code sums (rows padded to a multiple of 32).
struct PackedRows {
    size_t scale_at, sum_at, bytes;
};
PackedRows packed_rows(int M, int K) {
    PackedRows p;
    const size_t rows = size_t(M + 31) / 32 * 32;
    p.scale_at = rows * size_t(K);
    p.sum_at = p.scale_at + rows * size_t(K / 256) * 4;
    p.bytes = p.sum_at + rows * size_t(K / 32) * 4;
    return p;
}

// 32-lane unit u: row u / nsb (rows past M pack as zeros), 256 values at
// 256 (u % nsb).
template <bool XVEC>
__global__ __launch_bounds__(256) void strip_pack_kernel(const float* __restrict__ X, int64_t ldx, int M, int nsb,
                                                         int units, int8_t* __restrict__ codes,
                                                         float* __restrict__ scales, float* __restrict__ sums) {
    const int lane = threadIdx.x & 63, li = lane & 31;
    const int unit = blockIdx.x * 8 + (threadIdx.x >> 5);
    const int u = min(unit, units - 1);
    const int m = u / nsb, b = u - m * nsb;
    floatx8 v{0, 0, 0, 0, 0, 0, 0, 0};
    if (m < M) {
        const float* xr = X + int64_t(m) * ldx + 256 * b + 8 * li;
        if (XVEC) {
            const floatx4 lo = load4f(xr), hi = load4f(xr + 4);
            v = floatx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = xr[i];
        }
    }
    float d;
    int c[8], sum = 0;
    quant8_icodes<T_Q8_K, false>(v, lane, d, c);
#pragma unroll
    for (int i = 0; i < 8; ++i) sum += c[i];
    sum = group_sum<4>(sum);
    uint32_t w[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        w[i] = __builtin_amdgcn_perm(
            __builtin_amdgcn_perm(uint32_t(c[4 * i + 3]), uint32_t(c[4 * i + 2]), 0x0c0c0400u),
            __builtin_amdgcn_perm(uint32_t(c[4 * i + 1]), uint32_t(c[4 * i]), 0x0c0c0400u), 0x05040100u);
    if (unit >= units) return;
    const int tile = m >> 4, r = m & 15, step = 8 * b + (li >> 2), kq = li & 3;
    *reinterpret_cast<u32x2*>(codes + ((int64_t(tile) * 8 * nsb + step) * 64 + r + 16 * kq) * 8) = u32x2{w[0], w[1]};
    if (li == 0) scales[(tile * nsb + b) * 16 + r] = d;
    if (kq == 0) sums[(int64_t(tile) * 8 * nsb + step) * 16 + r] = float(sum);
}

// What one lane needs of U pairs of 32-value steps of its weight row, all in
// one super-block: the header and bytes 8 kq .. 8 kq + 7 of every step's
// codes.  Rows and row stride are 16-byte aligned.
template <int WT, int U>
struct WeightRun {
    u32x4 hdr;
    u32x2 qs[U], qh;
    // pair p0 is a multiple of U
    __device__ __forceinline__ void load(const uint8_t* row, int p0, int kq) {
        const uint8_t* b = row + block_bytes(WT) * int64_t(p0 >> 2);
        hdr = *reinterpret_cast<const u32x4*>(b);
        if (WT == T_Q5_K) qh = *reinterpret_cast<const u32x2*>(b + 16 + 8 * kq);
#pragma unroll
        for (int u = 0; u < U; ++u)
            qs[u] = *reinterpret_cast<const u32x2*>(b + (WT == T_Q4_K ? 16 : 48) + 32 * ((p0 & 3) + u) + 8 * kq);
    }
    // sub-block j = 2 ((p0 & 3) + u) + e
    __device__ __forceinline__ u32x2 codes(int u, int e, int j) const {
        u32x2 q{(qs[u][0] >> (4 * e)) & 0x0f0f0f0fu, (qs[u][1] >> (4 * e)) & 0x0f0f0f0fu};
        if (WT == T_Q5_K) {
            q[0] |= ((qh[0] >> j) & 0x01010101u) << 4;
            q[1] |= ((qh[1] >> j) & 0x01010101u) << 4;
        }
        return q;
    }
    __device__ __forceinline__ void scales(int j, float& ws, float& wm) const {
        const uint32_t sc3[3] = {hdr[1], hdr[2], hdr[3]};
        int sc, mn;
        k4_scale_min(j, sc3, sc, mn);
        ws = half_bits_to_float(hdr[0] & 0xffffu) * float(sc);
        wm = half_bits_to_float(hdr[0] >> 16) * float(mn);
    }
};

template <int WT, int NW, int U, int T>
__global__ __launch_bounds__(64 * NW) void strip16_kernel(const int8_t* __restrict__ codes,
                                                          const float* __restrict__ scales,
                                                          const float* __restrict__ sums,
                                                          const uint8_t* __restrict__ W, int64_t w_stride,
                                                          float* __restrict__ Y, int64_t ldy, int M, int N, int nsb,
                                                          int RG) {
#pragma clang fp contract(off)
    constexpr int SL = (32 * U + 63) / 64;   // loads of a run's 32 U code sums
    // a run's 16 scales, then the 16 code sums of each of its 2 U steps
    __shared__ __attribute__((aligned(16))) float rowv[NW][T][1 + 2 * U][16];
    __shared__ __attribute__((aligned(16))) float red[NW][4 * T * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = blockIdx.x % RG, mb = blockIdx.x / RG, n0 = 16 * rg;
    const int col = lane & 15, kq = lane >> 4, pairs = 4 * nsb;
    const uint8_t* row = W + int64_t(min(n0 + col, N - 1)) * w_stride;
    codes += int64_t(mb) * T * nsb * 8 * 512;
    scales += int64_t(mb) * T * nsb * 16;
    sums += int64_t(mb) * T * nsb * 8 * 16;

    float acc[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][i] = 0.f;

    for (int p0 = wave * U; p0 < pairs; p0 += NW * U) {
        WeightRun<WT, U> w;
        u32x2 a[T][U][2];
        float dv[T], sv[T][SL];
        w.load(row, p0, kq);
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    a[t][u][e] = *reinterpret_cast<const u32x2*>(
                        codes + ((int64_t(t) * 8 * nsb + 2 * (p0 + u) + e) * 64 + lane) * 8);
            dv[t] = scales[(t * nsb + (p0 >> 2)) * 16 + col];
#pragma unroll
            for (int l = 0; l < SL; ++l)
                sv[t][l] = sums[(int64_t(t) * 8 * nsb + 2 * p0) * 16 + (64 * l + lane) % (32 * U)];
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if (lane < 16) rowv[wave][t][0][lane] = dv[t];
#pragma unroll
            for (int l = 0; l < SL; ++l)
                if (32 * U % 64 == 0 || lane < 32 * U) (&rowv[wave][t][1][0])[64 * l + lane] = sv[t][l];
        }
        wave_lds_handoff();   // the wave's own row vectors
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int j = U == 4 ? 2 * u + e : 2 * ((p0 & 3) + u) + e;
                const u32x2 q = w.codes(u, e, j);
                float ws, wm;
                w.scales(j, ws, wm);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    // element i: activation row 16 t + 4 kq + i, weight row col
                    const floatx4 dx = *reinterpret_cast<const floatx4*>(&rowv[wave][t][0][4 * kq]);
                    const floatx4 cs = *reinterpret_cast<const floatx4*>(&rowv[wave][t][1 + 2 * u + e][4 * kq]);
                    const i32x4 dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                        __builtin_bit_cast(long, a[t][u][e]), __builtin_bit_cast(long, q), i32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = __builtin_fmaf(-wm, cs[i], ws * float(dot[i]));
                        acc[t][i] = __builtin_fmaf(dx[i], v, acc[t][i]);
                    }
                }
            }
        wave_lds_handoff();   // read before the next run's are stored
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][(4 * t + i) * 64 + lane] = acc[t][i];
    __syncthreads();
    for (int o = threadIdx.x; o < 256 * T; o += 64 * NW) {
        const int m = o >> 4, n = o & 15;
        const int at = (4 * (m >> 4) + (m & 3)) * 64 + n + 16 * ((m >> 2) & 3);
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < NW; ++q) v += red[q][at];
        const int gm = 16 * T * mb + m;
        if (gm < M && n0 + n < N) Y[int64_t(gm) * ldy + n0 + n] = v;
    }
}

}  // namespace

size_t strip16_bytes(int M, int K) { return packed_rows(M, K).bytes; }

bool strip16_supported(int wtype, int M, int K, const void* w, int64_t w_stride) {
    return (wtype == T_Q4_K || wtype == T_Q5_K) && K > 256 && K % 256 == 0 && strip16_bytes(M, K) <= kStrip16Bytes &&
           reinterpret_cast<uintptr_t>(w) % 16 == 0 && w_stride % 16 == 0;
}

const char* strip16_variant(int wtype) { return wtype == T_Q4_K ? "skinny_i8mfma16_q4_k" : "skinny_i8mfma16_q5_k"; }

void launch_strip16_pack(const float* x, int64_t ldx, void* scratch, int M, int K, hipStream_t stream) {
    const PackedRows pr = packed_rows(M, K);
    int8_t* codes = static_cast<int8_t*>(scratch);
    float* scales = reinterpret_cast<float*>(codes + pr.scale_at);
    float* sums = reinterpret_cast<float*>(codes + pr.sum_at);
    const int nsb = K / 256, units = (M + 31) / 32 * 32 * nsb;
    const dim3 grid(unsigned((units + 7) / 8)), block(256);
    if (reinterpret_cast<uintptr_t>(x) % 16 == 0 && ldx % 4 == 0)
        hipLaunchKernelGGL(strip_pack_kernel<true>, grid, block, 0, stream, x, ldx, M, nsb, units, codes, scales, sums);
    else
        hipLaunchKernelGGL(strip_pack_kernel<false>, grid, block, 0, stream, x, ldx, M, nsb, units, codes, scales, sums);
}

void launch_strip16(int wtype, const void* scratch, const void* w, int64_t w_stride, float* y, int64_t ldy, int M, int N,
                    int K, int cus, hipStream_t stream) {
    const PackedRows pr = packed_rows(M, K);
    const int8_t* codes = static_cast<const int8_t*>(scratch);
    const float* scales = reinterpret_cast<const float*>(codes + pr.scale_at);
    const float* sums = reinterpret_cast<const float*>(codes + pr.sum_at);
    const uint8_t* wb = static_cast<const uint8_t*>(w);
    const int nsb = K / 256, RG = (N + 15) / 16;
    // two row tiles per workgroup share its weight; one while that still
    // leaves every workgroup a CU (and for 16 rows and fewer)
    const int tiles = (M + 15) / 16, pairs = 4 * nsb;
    const bool one = tiles == 1 || RG * tiles <= cus;
    const dim3 grid(unsigned(RG * (one ? tiles : (tiles + 1) / 2)));
#define SAMHIP_STRIP16(WT, NW, U, T)                                                                               \
    hipLaunchKernelGGL((strip16_kernel<WT, NW, U, T>), grid, dim3(64 * NW), 0, stream, codes, scales, sums, wb, w_stride, \
                       y, ldy, M, N, nsb, RG)
#define SAMHIP_STRIP16_U(WT, T)                           \
    do {                                                  \
        if (pairs <= 8) SAMHIP_STRIP16(WT, 8, 1, T);      \
        else if (pairs <= 16) SAMHIP_STRIP16(WT, 16, 1, T); \
        else if (pairs <= 32) SAMHIP_STRIP16(WT, 16, 2, T); \
        else SAMHIP_STRIP16(WT, 16, 4, T);                \
    } while (0)
    if (wtype == T_Q4_K) {
        if (one) SAMHIP_STRIP16_U(T_Q4_K, 1);
        else SAMHIP_STRIP16_U(T_Q4_K, 2);
    } else {
        if (one) SAMHIP_STRIP16_U(T_Q5_K, 1);
        else SAMHIP_STRIP16_U(T_Q5_K, 2);
    }
#undef SAMHIP_STRIP16_U
#undef SAMHIP_STRIP16
}

}  // namespace samhip
