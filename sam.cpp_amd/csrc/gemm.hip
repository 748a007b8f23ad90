// Quantized-weight GEMM for gfx950: Y[m][n] = rs[m] * sum_k A[m][k] * Wq[n][k]
//   A  : staged fp16 activations [M][K] (row scale rs[m] = 2^e)
//   Wq : GGUF-packed weight rows (Q8_0 / Q4_K / Q5_K / Q6_K), any row stride
//   Y  : F32 [M][N] with row stride ldy
// Weights are dequantized to fp16(ggml to_float(W)) while they travel from
// HBM to LDS; the product runs on v_mfma_f32_32x32x16_f16 with F32
// accumulation.  This replaces ggml's MUL_MAT kernels for packed weights
// (CPU vec_dot_* / CUDA MMQ, tests/runtime/ggml/test_quantization.cpp:604-614).
#include "internal.hpp"

namespace samhip {

namespace {

constexpr int BM = 128, BN = 128, BK = 32;
constexpr int LDS_STRIDE = BK + 8;   // halves; 80-byte rows keep 16-byte reads conflict-free
constexpr int GROUP_M = 8;
// The 16 weights of one thread and K step between their load and their
// decoding.  WeightPiece aligns the bytes as part of the load, which waits
// for them; Q8_0 rows (the ones this kernel gets by default) keep the dwords
// as they were read, so that DEPTH steps of loads can be in flight.
template <int WT> struct StepPiece : WeightPiece<WT> {
    __device__ __forceinline__ void load_step(const uint8_t* row, int step, int h) { this->load(row, step, h); }
    __device__ __forceinline__ void decode(const uint8_t*, int step, int h, _Float16* out) const {
        this->dequant(step, h, out);
    }
};
template <> struct StepPiece<T_Q8_0> {
    uint32_t w[5], d;
    // byte (0 or 2) at which the step's block starts in its first dword
    static __device__ __forceinline__ uint32_t shift(const uint8_t* row, int step) {
        return uint32_t(reinterpret_cast<uintptr_t>(row) + 34 * step) & 2;
    }
    __device__ __forceinline__ void load_step(const uint8_t* row, int step, int h) {
        const uint32_t sd = shift(row, step), sc = sd ^ 2;   // the codes start two bytes on
        const uint8_t* blk = row + 34 * step;
        d = *reinterpret_cast<const uint32_t*>(blk - sd);
        const uint32_t* q = reinterpret_cast<const uint32_t*>(blk + 2 + 16 * h - sc);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = q[i];
        w[4] = q[sc ? 4 : 3];   // no dword without one of the 16 bytes is touched
    }
    __device__ __forceinline__ void decode(const uint8_t* row, int step, int, _Float16* out) const {
        const uint32_t sd = shift(row, step), sc = sd ^ 2;
        const _Float16 dh = __builtin_bit_cast(_Float16, uint16_t(sd ? d >> 16 : d));
#pragma unroll
        for (int i = 0; i < 4; ++i) mul_i8x4_to_half(funnel_bytes(w[i + 1], w[i], sc), dh, out + 4 * i);
    }
};

// K steps in flight per thread, in registers, where every tile has a CU to
// itself: one step's products (8 MFMAs a wave) are far shorter than the
// latency of its scattered packed-weight loads.  M = 300, N = 259, K = 1024 (9
// tiles) with its staging Q8_0 44 -> 31 us, Q4_K 58 -> 45, M = 4096, N = 1024
// (256 tiles) 55 -> 41 and 69 -> 55.
template <int WT>
constexpr int kDepth = WT == T_Q8_0 ? 4 : 2;
// More tiles than CUs hide one another's loads instead: one step in flight,
// in at most 128 registers, so that four workgroups fit a CU.  Against the
// rings (145 .. 172 registers, three): M = 5184, N = 3072, K = 1024 Q8_0 92 ->
// 82 us, Q5_K 131 -> 118, M = 10000, N = 4736 Q4_K 314 -> 285, Q5_K 366 -> 309,
// M = 3000, N = 1500, K = 2048 (288 tiles) Q8_0 88 -> 77, Q6_K level at 93.

// Tile order: blocks are dispatched round-robin over the 8 XCDs, so give each
// XCD a contiguous range of tiles, and walk that range in groups of GROUP_M
// row-tiles so that concurrently resident tiles share A rows and W rows in
// the XCD's L2.
__device__ __forceinline__ void tile_of(int bid, int nblocks, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int per = nblocks / 8, rem = nblocks % 8;
    const int xcd = bid % 8, idx = bid / 8;
    const int t = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
    const int span = GROUP_M * tiles_n;
    const int group = t / span, first = group * GROUP_M;
    const int gm = min(tiles_m - first, GROUP_M);
    const int within = t % span;
    tm = first + within % gm;
    tn = within / gm;
}

template <int WT, int DEPTH>
__global__ __launch_bounds__(256, 2) void gemm_kernel(const _Float16* __restrict__ A, int64_t lda,
                                                      const float* __restrict__ row_scale,
                                                      const uint8_t* __restrict__ W, int64_t w_stride,
                                                      float* __restrict__ Y, int64_t ldy, int M, int N, int K,
                                                      int tiles_m, int tiles_n) {
    static_assert(DEPTH == 1 || DEPTH % 2 == 0, "the LDS buffer alternates per step");
    __shared__ _Float16 As[2][BM * LDS_STRIDE];
    __shared__ _Float16 Bs[2][BN * LDS_STRIDE];

    int tm, tn;
    tile_of(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    // loader role: row lr of the tile, 16-element half lh of the K step
    const int lr = tid >> 1, lh = tid & 1;
    // rows past M or N repeat the last one; their products are not stored
    const _Float16* a_src = A + int64_t(min(m0 + lr, M - 1)) * lda + 16 * lh;
    const uint8_t* w_row = W + int64_t(min(n0 + lr, N - 1)) * w_stride;

    floatx16 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    u32x4 a_reg[DEPTH][2];
    StepPiece<WT> b_reg[DEPTH];

    const int nsteps = K / BK;
    auto global_load = [&](int slot, int step) {
        // past the range: a repeat of the last step, which may reach the LDS
        // buffer that no later step reads, and no product
        const int st = min(step, nsteps - 1);
        const u32x4* p = reinterpret_cast<const u32x4*>(a_src + BK * st);
        a_reg[slot][0] = p[0];
        a_reg[slot][1] = p[1];
        b_reg[slot].load_step(w_row, st, lh);
    };
    auto lds_store = [&](int buf, int slot, int step) {
        u32x4* ad = reinterpret_cast<u32x4*>(&As[buf][lr * LDS_STRIDE + 16 * lh]);
        ad[0] = a_reg[slot][0];
        ad[1] = a_reg[slot][1];
        _Float16 w[16];
        b_reg[slot].decode(w_row, step, lh, w);
        half8* bd = reinterpret_cast<half8*>(&Bs[buf][lr * LDS_STRIDE + 16 * lh]);
        bd[0] = half8{w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7]};
        bd[1] = half8{w[8], w[9], w[10], w[11], w[12], w[13], w[14], w[15]};
    };

    const int frag_row = lane & 31, frag_k = 8 * (lane >> 5);
    auto products = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < BK; ks += 16) {
            half8 af[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                af[i] = *reinterpret_cast<const half8*>(&As[buf][(wm * 64 + i * 32 + frag_row) * LDS_STRIDE + ks + frag_k]);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                bf[j] = *reinterpret_cast<const half8*>(&Bs[buf][(wn * 64 + j * 32 + frag_row) * LDS_STRIDE + ks + frag_k]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    };
    if constexpr (DEPTH == 1) {
        global_load(0, 0);
        lds_store(0, 0, 0);
        __syncthreads();
        for (int s = 0; s < nsteps; ++s) {
            if (s + 1 < nsteps) global_load(0, s + 1);
            products(s & 1);
            if (s + 1 < nsteps) lds_store((s & 1) ^ 1, 0, s + 1);
            __syncthreads();
        }
    } else {
        // slot i of the register ring holds a step s with s % DEPTH == i
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) global_load(i, i);
        lds_store(0, 0, 0);
        global_load(0, DEPTH);
        __syncthreads();
        // whole turns of the ring without a branch, so that each wait counts
        // exactly the loads issued since; then the up to DEPTH - 1 steps left
        int s0 = 0;
        for (; s0 + DEPTH <= nsteps; s0 += DEPTH) {
#pragma unroll
            for (int u = 0; u < DEPTH; ++u) {
                const int next = (u + 1) % DEPTH;
                products(u & 1);
                lds_store((u & 1) ^ 1, next, min(s0 + u + 1, nsteps - 1));
                global_load(next, s0 + u + 1 + DEPTH);
                __syncthreads();
            }
        }
#pragma unroll
        for (int u = 0; u < DEPTH - 1; ++u) {
            if (s0 + u >= nsteps) break;
            products(u & 1);
            if (s0 + u + 1 < nsteps) lds_store((u & 1) ^ 1, u + 1, s0 + u + 1);
            __syncthreads();
        }
    }

    // 32x32 accumulator layout: lane l holds column l%32, rows 8*(r/4) + 4*(l/32) + r%4.
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (m >= M) continue;
            const float rs = row_scale[m];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int n = n0 + wn * 64 + j * 32 + (lane & 31);
                if (n < N) Y[int64_t(m) * ldy + n] = acc[i][j][r] * rs;
            }
        }
    }
}

}  // namespace

const char* gemm_variant(int wtype) {
    switch (wtype) {
        case T_Q8_0: return "gemm_f16mfma_128x128x32_q8_0";
        case T_Q4_K: return "gemm_f16mfma_128x128x32_q4_k";
        case T_Q5_K: return "gemm_f16mfma_128x128x32_q5_k";
        case T_Q6_K: return "gemm_f16mfma_128x128x32_q6_k";
        default: return nullptr;
    }
}

const char* launch_gemm(int wtype, const _Float16* a, int64_t lda, const float* row_scale, const void* w,
                        int64_t w_stride, float* y, int64_t ldy, int M, int N, int K, int cus, hipStream_t stream) {
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const dim3 grid(unsigned(tiles_m * tiles_n)), block(256);
    const uint8_t* wb = static_cast<const uint8_t*>(w);
#define SAMHIP_GEMM(T)                                                                                              \
    do {                                                                                                            \
        if (tiles_m * tiles_n <= cus)                                                                               \
            hipLaunchKernelGGL((gemm_kernel<T, kDepth<T>>), grid, block, 0, stream, a, lda, row_scale, wb, w_stride, \
                               y, ldy, M, N, K, tiles_m, tiles_n);                                                  \
        else                                                                                                        \
            hipLaunchKernelGGL((gemm_kernel<T, 1>), grid, block, 0, stream, a, lda, row_scale, wb, w_stride, y, ldy, \
                               M, N, K, tiles_m, tiles_n);                                                          \
    } while (0)
    switch (wtype) {
        case T_Q8_0: SAMHIP_GEMM(T_Q8_0); break;
        case T_Q4_K: SAMHIP_GEMM(T_Q4_K); break;
        case T_Q5_K: SAMHIP_GEMM(T_Q5_K); break;
        case T_Q6_K: SAMHIP_GEMM(T_Q6_K); break;
        default: return nullptr;
    }
#undef SAMHIP_GEMM
    return gemm_variant(wtype);
}

}  // namespace samhip
