// gemm_bf16.hip — the BF16-mode linear layer for gfx950 (the layers a
// quantized checkpoint keeps unquantized: img_in, txt_in, norm_out and
// proj_out, transformer.cu:396-419, 874-895):
//   out[m,n] = sum_k bf16(x[m,k]) * w[n,k] + bias[n]   (then GELU-tanh)
// with x fp32 (rounded to bf16, round to nearest even, as the reference's
// fp32_to_bf16 pass) or bf16, w bf16 [N, K], fp32 accumulation and an fp32
// output. Replaces linear_forward_bf16 / linear_forward_bf16_bf16in
// (cuda_kernels.cu:4534-4596: fp32_to_bf16, cublasGemmEx bf16 x bf16 -> fp32,
// bias_add_fp32, gelu_fp32) with one kernel: the fp32 -> bf16 rounding
// happens on the operand registers and the bias / GELU on the accumulators.
// With `accumulate`, the product is added to the fp32 values already in out
// before the bias (the INT4 linear's residual GEMM onto its low-rank term,
// cublasGemmEx with beta = 1, cuda_kernels.cu:4488-4497).
//
// Shapes (M = tokens): img_in 3072 x 64, txt_in 3072 x 3584, norm_out
// 6144 x 3072 at M = 1 (or 2), proj_out 64 x 3072. They are bound by reading
// the weights (norm_out, txt_in) or the activations (proj_out) or by writing
// the output (img_in). Short K (img_in) takes gemm_bf16_shortk_kernel, K of
// whole 128-element stages gemm_bf16_dma_kernel, other multiples of 32
// gemm_bf16_kernel, built like the small-M quantized linear: a workgroup owns
// a 32x32 or 64x64 output tile, its four waves split K in 32-element blocks
// dealt round-robin (every operand byte is read by one wave), and the partial
// tiles are summed through LDS in wave order. Operands go straight from global
// memory into MFMA fragment registers with buffer loads (rows past M or N and
// blocks past K read as zero), DEPTH blocks in flight per wave.
// v_mfma_f32_32x32x16_bf16: lane (row r = lane%32, half h = lane/32) of a
// 32-row block holds, for k-step s of K block kb, the 8 elements
// kb*32 + 16h + 8s .. +7; both operands use the same assignment, so each dot
// product covers every k once.
#include <utility>

#include "qimg_device.h"
#include "qimg_internal.h"

namespace qimg {

namespace {

constexpr int BF_THR = 256;  // four waves, one K quarter each
constexpr int BF_KB = 32;    // elements of K per block
constexpr int SK_M = 64, SK_N = 128;  // tile of the short-K kernel
constexpr int SK_XP = 72;  // bf16 per LDS row of 64 x values (16 rows fall on 16 bank groups)
constexpr int kShortKMaxN = 1 << 22;  // its tile's output rows stay below 2^31 bytes (kOob out of range)
constexpr int kRsrcWord3 = 0x00020000;  // raw unswizzled buffer (gfx9 family)
constexpr uint32_t kOob = 0x80000000u;  // offset >= num_records: reads zero

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

template <int TMW, int TNW>
struct BfEpi {
    float b[TMW * TNW][4];
};

// 16 fp32 -> 8 + 8 bf16 (round to nearest even, the reference's
// __float2bfloat16) as two MFMA fragments.
__device__ __forceinline__ void f32x16_to_frags(const v4f (&x)[4], v8bf& lo, v8bf& hi) {
    uint32_t p[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        p[2 * i] = pack_bf16x2(x[i][0], x[i][1]);
        p[2 * i + 1] = pack_bf16x2(x[i][2], x[i][3]);
    }
    lo = __builtin_bit_cast(v8bf, (v4i){static_cast<int>(p[0]), static_cast<int>(p[1]), static_cast<int>(p[2]),
                                        static_cast<int>(p[3])});
    hi = __builtin_bit_cast(v8bf, (v4i){static_cast<int>(p[4]), static_cast<int>(p[5]), static_cast<int>(p[6]),
                                        static_cast<int>(p[7])});
}

template <bool XF32, int TMW, int TNW, int DEPTH, bool GELU>
__global__ __launch_bounds__(BF_THR) void gemm_bf16_kernel(const void* __restrict__ X,
                                                           const uint16_t* __restrict__ Wt,
                                                           const uint16_t* __restrict__ bias,
                                                           float* out, int M, int N, int K, int accumulate) {
    constexpr int MB = 32 * TMW;
    constexpr int NB = 32 * TNW;
    constexpr int NBLK = TMW * TNW;
    constexpr int NW = BF_THR / 64;
    constexpr int XE = XF32 ? 4 : 2;  // bytes per x element
    // partial tiles [wave][block][run g][lane], 16 bytes each
    __shared__ v4f red[NW * NBLK * 4 * 64];

    const int tiles_m = (M + MB - 1) / MB;
    const int tiles_n = (N + NB - 1) / NB;
    const int logical = xcd_remap(blockIdx.x, tiles_m * tiles_n);
    const int m0 = (logical % tiles_m) * MB;
    const int n0 = (logical / tiles_m) * NB;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31;
    const int h = lane >> 5;

    // bias of the (row, 4-column run) groups this thread stores (the
    // mapping of the epilogue below), loaded now
    BfEpi<TMW, TNW> epi;
#pragma unroll
    for (int q = 0; q < NBLK; ++q) {
        const int idx = threadIdx.x + BF_THR * q;
        const int blk = idx >> 8;
        const int nb = n0 + 32 * (blk % TNW) + 8 * ((idx >> 6) & 3) + 4 * ((idx >> 5) & 1);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            epi.b[q][c] = bias != nullptr ? bf16_to_f32(bias[nb + c < N ? nb + c : N - 1]) : 0.0f;
    }

    const int nkb = K / BF_KB;
    const int T = (nkb + NW - 1) / NW;
    const int Tp = ((T + DEPTH - 1) / DEPTH) * DEPTH;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(X), 0, static_cast<int>(static_cast<int64_t>(M) * K * XE), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(Wt), 0, static_cast<int>(static_cast<int64_t>(N) * K * 2), kRsrcWord3);
    uint32_t ox[TMW], ow[TNW];
#pragma unroll
    for (int i = 0; i < TMW; ++i) {
        const int gm = m0 + 32 * i + r;
        ox[i] = (static_cast<uint32_t>(gm) * K + 16 * h) * XE | (gm < M ? 0u : kOob);
    }
#pragma unroll
    for (int j = 0; j < TNW; ++j) {
        const int gn = n0 + 32 * j + r;
        ow[j] = (static_cast<uint32_t>(gn) * K + 16 * h) * 2 | (gn < N ? 0u : kOob);
    }

    v16f acc[TMW][TNW];
#pragma unroll
    for (int i = 0; i < TMW; ++i)
#pragma unroll
        for (int j = 0; j < TNW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // one K block's operands of this lane: x 16 elements per row block,
    // w 16 elements per column block
    v4f bx[DEPTH][TMW][XF32 ? 4 : 1];
    v4i bxh[DEPTH][TMW][2];
    v4i bw[DEPTH][TNW][2];
    auto load = [&](int d, int t) {
        const int kb = NW * t + wave;
        const uint32_t kbad = kb < nkb ? 0u : kOob;
#pragma unroll
        for (int i = 0; i < TMW; ++i) {
            const uint32_t o = (ox[i] + static_cast<uint32_t>(kb) * BF_KB * XE) | (ox[i] & kOob) | kbad;
            if constexpr (XF32) {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    bx[d][i][s] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rx, o + 16 * s, 0, 0));
            } else {
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    bxh[d][i][s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rx, o + 16 * s, 0, 0));
            }
        }
#pragma unroll
        for (int j = 0; j < TNW; ++j) {
            const uint32_t o = (ow[j] + static_cast<uint32_t>(kb) * BF_KB * 2) | (ow[j] & kOob) | kbad;
#pragma unroll
            for (int s = 0; s < 2; ++s)
                bw[d][j][s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, o + 16 * s, 0, 0));
        }
    };
    auto compute = [&](int d) {
        v8bf fx[TMW][2];
#pragma unroll
        for (int i = 0; i < TMW; ++i) {
            if constexpr (XF32) {
                f32x16_to_frags(bx[d][i], fx[i][0], fx[i][1]);
            } else {
                fx[i][0] = __builtin_bit_cast(v8bf, bxh[d][i][0]);
                fx[i][1] = __builtin_bit_cast(v8bf, bxh[d][i][1]);
            }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < TMW; ++i)
#pragma unroll
                for (int j = 0; j < TNW; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, bw[d][j][s]),
                                                                        fx[i][s], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        load(d, d);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int t0 = 0; t0 < Tp; t0 += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            compute(d);
            load(d, t0 + d + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // partial tiles -> LDS; the first wave's lanes own whole runs below
#pragma unroll
    for (int i = 0; i < TMW; ++i)
#pragma unroll
        for (int j = 0; j < TNW; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                red[((wave * NBLK + i * TNW + j) * 4 + g) * 64 + lane] =
                    (v4f){acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    __syncthreads();

    // Epilogue: thread idx owns (block, run g, lane) groups of 4 columns:
    // row m = 32 i + lane%32, columns 8 g + 4 (lane/32) + c (the MFMA D
    // layout, D = W x X^T indexed [n][m]). Partials are added in wave order,
    // then the bias (bias_add_fp32), then GELU (gelu_fp32).
    const bool vec_ok = (N & 3) == 0;
#pragma unroll
    for (int q = 0; q < NBLK; ++q) {
        const int idx = threadIdx.x + BF_THR * q;
        const int blk = idx >> 8;
        const int g = (idx >> 6) & 3;
        const int ln = idx & 63;
        const int i = blk / TNW;
        const int j = blk % TNW;
        const int m = m0 + 32 * i + (ln & 31);
        const int nb = n0 + 32 * j + 8 * g + 4 * (ln >> 5);
        if (m >= M || nb >= N) continue;
        v4f sum = red[(blk * 4 + g) * 64 + ln];
#pragma unroll
        for (int w = 1; w < NW; ++w) sum += red[((w * NBLK + blk) * 4 + g) * 64 + ln];
        float* o = out + static_cast<int64_t>(m) * N + nb;
        float prev[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (accumulate) {
            if (vec_ok) {
                const v4f p4 = *reinterpret_cast<const v4f*>(o);
                prev[0] = p4[0]; prev[1] = p4[1]; prev[2] = p4[2]; prev[3] = p4[3];
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (nb + c < N) prev[c] = o[c];
            }
        }
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float t = sum[c];
            if (accumulate) t = t + prev[c];
            if (bias != nullptr) t = t + epi.b[q][c];
            if (GELU) t = gelu_tanh(t);
            v[c] = t;
        }
        if (vec_ok) {
            *reinterpret_cast<v4f*>(o) = (v4f){v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (nb + c < N) o[c] = v[c];
        }
    }
}

// Short K (img_in: K = 64): bound by writing the output. A workgroup owns 64
// rows x 128 columns, each wave 64 x 32 (two 32x32 blocks), and runs the
// whole of K, so no partial tiles are reduced; the fragments are those of
// gemm_bf16_kernel with x as the A operand, the products summed in K-block
// order. 64 k of the tile's x rows at a time come in whole lines, are rounded
// to bf16 once and shared through LDS (every wave loading its own fp32
// fragments, 32 lines an instruction, cost 7 us of 21); w goes straight to
// fragments. The tile then goes through LDS, so that a store instruction
// writes 512 contiguous bytes of two rows. Tiles are numbered n first, so that
// workgroups in flight together write whole output rows. 4096x3072x64: 29.9
// us with fragments and 16-byte stores of 32 rows per instruction, 21 with the
// output through LDS, 11.8 with x through LDS too (51 MB: 4.3 TB/s; a fill of
// the output alone takes 9.4 us); 6889 rows 16.8, K = 256 58 -> 22.5.
template <bool XF32, bool GELU>
__global__ __launch_bounds__(BF_THR) void gemm_bf16_shortk_kernel(const void* __restrict__ X,
                                                                  const uint16_t* __restrict__ Wt,
                                                                  const uint16_t* __restrict__ bias,
                                                                  float* out, int M, int N, int K, int accumulate) {
    constexpr int XE = XF32 ? 4 : 2;
    constexpr int PITCH = SK_N + 4;
    __shared__ __attribute__((aligned(16))) float stage[SK_M * PITCH];
    const int tiles_m = (M + SK_M - 1) / SK_M;
    const int tiles_n = (N + SK_N - 1) / SK_N;
    const int logical = xcd_remap(blockIdx.x, tiles_m * tiles_n);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = (logical / tiles_n) * SK_M;
    const int n0 = (logical % tiles_n) * SK_N;
    const int r = lane & 31;
    const int h = lane >> 5;
    const int n = n0 + 32 * wave + r;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(X), 0, static_cast<int>(static_cast<int64_t>(M) * K * XE), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(Wt), 0, static_cast<int>(static_cast<int64_t>(N) * K * 2), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(bias), 0, bias != nullptr ? N * 2 : 0, kRsrcWord3);
    // the tile's rows of out, those past M out of range
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        out + static_cast<int64_t>(m0) * N, 0, (M - m0 < SK_M ? M - m0 : SK_M) * N * 4, kRsrcWord3);
    const uint32_t ow = n < N ? (static_cast<uint32_t>(n) * K + 16 * h) * 2 : kOob;
    const float bv = bf16_to_f32(
        static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(rb, static_cast<uint32_t>(n) * 2, 0, 0)));
    v16f acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
    const int nkb = K / BF_KB;
    uint16_t* xs = reinterpret_cast<uint16_t*>(stage);
    for (int k2 = 0; k2 < nkb; k2 += 2) {
        // x rows, 64 k: thread t takes 16-byte pieces t, t + 256, ..
        constexpr int PER_ROW = XF32 ? 16 : 8, PIECES = SK_M * PER_ROW / BF_THR;
        v4i xr[PIECES], wr[2][2];
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
            const int row = m0 + (static_cast<int>(threadIdx.x) + BF_THR * q) / PER_ROW;
            const int k = k2 * BF_KB + (static_cast<int>(threadIdx.x) % PER_ROW) * (16 / XE);
            xr[q] = __builtin_bit_cast(
                v4i, __builtin_amdgcn_raw_buffer_load_b128(
                         rx, row < M && k < K ? (static_cast<uint32_t>(row) * K + k) * XE : kOob, 0, 0));
        }
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const uint32_t bad = k2 + d < nkb ? 0u : kOob;  // past K: zeros
#pragma unroll
            for (int q = 0; q < 2; ++q)
                wr[d][q] = __builtin_bit_cast(
                    v4i, __builtin_amdgcn_raw_buffer_load_b128(
                             rw, ((ow + static_cast<uint32_t>(k2 + d) * BF_KB * 2 + 16 * q) | (ow & kOob) | bad), 0, 0));
        }
        if (k2 > 0) __syncthreads();  // every wave has read the previous rows
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
            const int idx = static_cast<int>(threadIdx.x) + BF_THR * q;
            uint16_t* o = xs + idx / PER_ROW * SK_XP + idx % PER_ROW * (16 / XE);
            if constexpr (XF32) {
                const v4f f = __builtin_bit_cast(v4f, xr[q]);
                *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]));
            } else {
                *reinterpret_cast<v4i*>(o) = xr[q];
            }
        }
        __syncthreads();
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        *reinterpret_cast<const v8bf*>(xs + (32 * i + r) * SK_XP + 32 * d + 16 * h + 8 * q),
                        __builtin_bit_cast(v8bf, wr[d][q]), acc[i], 0, 0, 0);
    }
    __syncthreads();  // the output tile takes x's place
    const bool vec_ok = (N & 3) == 0;
    const int sc = 4 * (threadIdx.x & 31);  // columns this thread stores
    const int sr = threadIdx.x >> 5;        // and its first row
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        // element e: row 32 i + 8 (e / 4) + 4 h + e % 4, column n
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = acc[i][e];
        if (accumulate) {
            float prev[16];
#pragma unroll
            for (int e = 0; e < 16; ++e)
                prev[e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(
                               ro, n < N ? (static_cast<uint32_t>(32 * i + 8 * (e >> 2) + 4 * h + (e & 3)) * N + n) * 4 : kOob, 0, 0));
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = v[e] + prev[e];
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            if (bias != nullptr) v[e] = v[e] + bv;
            if (GELU) v[e] = gelu_tanh(v[e]);
            stage[(32 * i + 8 * (e >> 2) + 4 * h + (e & 3)) * PITCH + 32 * wave + r] = v[e];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SK_M / 8; ++q) {
        const int row = sr + 8 * q;
        const v4f t = *reinterpret_cast<const v4f*>(stage + row * PITCH + sc);
        const uint32_t o = (static_cast<uint32_t>(row) * N + n0 + sc) * 4;
        if (vec_ok) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, t), ro, n0 + sc < N ? o : kOob, 0, 0);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float tc = t[c];
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(tc), ro, n0 + sc + c < N ? o + 4 * c : kOob,
                                                      0, 0);
            }
        }
    }
}

// Long K (txt_in, norm_out, proj_out, the INT4 linears' down factor): tiles
// of TM rows x TN columns whose operands stream through LDS. A stage is 128
// elements of K of the tile's x and w rows, filled by direct global->LDS DMA
// of whole lines (1 KB per instruction; the direct fragment loads of
// gemm_bf16_kernel touch 16 to 64 bytes of each of 32 lines) into a ring of
// NS stages, NS - 1 in flight. Four waves take 32 elements of K each and compute
// the whole tile (v_mfma_f32_16x16x32_bf16, w as the A operand), so each operand
// byte leaves LDS once; tiles of 32 and 64 rows have eight waves, four for each
// half of the rows (w leaves LDS twice, and a SIMD has a second wave to run
// while one waits for its fragments). x is rounded to bf16 on the fragments.
// The partial tiles are summed through LDS in wave order, and the stores run
// along n. One barrier per stage: stage s has landed in every wave, and every
// wave is done with stage s - 1, whose slot is refilled right after.
// LDS chunk c of row r sits at c ^ (r & 15): the 16 rows of a fragment read
// fall on 16 different bank groups.
// Rows past M and N re-read the last row and are not stored. With out16 the
// result is rounded to bf16 there, rows of ldo (out is not touched). x has rows
// of ldx.
// Measured against gemm_bf16_kernel (us, fp32 x): txt_in 256x3072x3584 48 ->
// 18.4 (23.3 with four waves; 512 rows 44.2 -> 35.8), proj_out 4096x64x3072 25
// -> 10.9 (50 MB of x: 4.6 TB/s), norm_out 1x6144x3072 11 -> 7.9 (38 MB of w:
// 4.8 TB/s); the INT4 down factor 4096x32x3072 (bf16 x) 15.7 -> 6.7. txt_in
// has 192 workgroups that each take 1.4 MB through their CU's port with 96 KB
// in flight. It is the faster one for every K of whole 128 timed (1 to 8192 rows,
// N 64 to 6144, K 128 to 12288): 1024x3072x3072 111 -> 55 us, 8192x3072x3072 907
// -> 422, 2048x6144x3072 456 -> 328, bf16 x 1024x3072x384 18.8 -> 12.4.
template <bool XF32, int TM, int TN>
struct BfDma {
    static constexpr int KS = 128;                        // K elements per stage
    static constexpr int XE = XF32 ? 4 : 2;
    static constexpr int XROW = KS * XE, WROW = KS * 2;   // bytes per row of a stage
    static constexpr int XB = TM * XROW, WB = TN * WROW;
    static constexpr int STAGE = XB + WB;
    static constexpr int NS = 144 * 1024 / STAGE < 8 ? 144 * 1024 / STAGE : 8;
    static constexpr int MH = TM >= 32 ? 2 : 1;           // waves along the tile's rows
    static constexpr int NW = 4 * MH, THR = 64 * NW;
    static constexpr int XI = XB / (1024 * NW), WI = WB / (1024 * NW);  // DMA instructions per wave and stage
    static constexpr int PER = XI + WI;
    static_assert(XB % (1024 * NW) == 0 && WB % (1024 * NW) == 0 && NS >= 3 && (NS - 1) * PER <= 63,
                  "stage split over the waves");
    static_assert(NS * STAGE >= 4 * TM * (TN + 4) * 4, "the partial tiles reuse the ring");
};

template <bool XF32, int TM, int TN, bool GELU>
__global__ __launch_bounds__((BfDma<XF32, TM, TN>::THR)) void gemm_bf16_dma_kernel(const void* __restrict__ X,
                                                               const uint16_t* __restrict__ Wt,
                                                               const uint16_t* __restrict__ bias, float* out,
                                                               uint16_t* out16, int64_t ldx, int64_t ldo, int M,
                                                               int N, int K, int accumulate) {
    using G = BfDma<XF32, TM, TN>;
    constexpr int NS = G::NS, PER = G::PER, XI = G::XI, NW = G::NW;
    constexpr int WM = TM / G::MH;  // rows of a wave
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * G::STAGE];

    const int tiles_m = (M + TM - 1) / TM;
    const int tiles_n = (N + TN - 1) / TN;
    const int logical = xcd_remap(blockIdx.x, tiles_m * tiles_n);
    // tiles that share rows of the larger operand are numbered in a row: one
    // XCD's L2 reads them once (proj_out's x, txt_in's w)
    const bool x_larger = static_cast<int64_t>(M) * G::XE > static_cast<int64_t>(N) * 2;
    const int m0 = (x_larger ? logical / tiles_n : logical % tiles_m) * TM;
    const int n0 = (x_larger ? logical % tiles_n : logical / tiles_m) * TN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ks = wave & 3;           // this wave's 32 elements of a stage's K
    const int mw = (wave >> 2) * WM;   // and its rows of the tile

    // bias of the four columns this thread stores in every row it stores
    const int col = n0 + 4 * (static_cast<int>(threadIdx.x) % (TN / 4));
    float bv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) bv[c] = bias != nullptr ? bf16_to_f32(bias[col + c < N ? col + c : N - 1]) : 0.0f;

    // DMA instruction j of this wave fills KB NW j + wave of the stage (x
    // rows, then w rows)
    const uint8_t* src[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const bool is_x = j < XI;
        const int rb = is_x ? G::XROW : G::WROW;  // bytes per row
        const int off = (NW * (is_x ? j : j - XI) + wave) * 1024 + lane * 16;
        const int row = off / rb;
        const int c = ((off % rb) >> 4) ^ (row & 15);
        if (is_x) {
            const int gm = m0 + row < M ? m0 + row : M - 1;
            src[j] = static_cast<const uint8_t*>(X) + gm * ldx * G::XE + c * 16;
        } else {
            const int gn = n0 + row < N ? n0 + row : N - 1;
            src[j] = reinterpret_cast<const uint8_t*>(Wt) + static_cast<int64_t>(gn) * K * 2 + c * 16;
        }
    }
    auto issue = [&](int s, int slot) {
        uint8_t* dst = lds + slot * G::STAGE + wave * 1024;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(src[j] + static_cast<int64_t>(s) * (j < XI ? G::XROW : G::WROW)),
                                             (lds_ptr_t)(dst + j * (NW * 1024)), 16, 0, 1);
    };

    const int r = lane & 15;
    const int kq = lane >> 4;
    v4f acc[WM / 16][TN / 16];
#pragma unroll
    for (int i = 0; i < WM / 16; ++i)
#pragma unroll
        for (int j = 0; j < TN / 16; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    // lane (row r, kq) of a fragment holds elements 32 ks + 8 kq .. +7
    auto compute = [&](int slot) {
        const uint8_t* xs = lds + slot * G::STAGE;
        const uint8_t* ws = xs + G::XB;
        v8bf fx[WM / 16], fw[TN / 16];
#pragma unroll
        for (int j = 0; j < TN / 16; ++j)
            fw[j] = *reinterpret_cast<const v8bf*>(ws + (16 * j + r) * G::WROW + (((4 * ks + kq) ^ r) << 4));
#pragma unroll
        for (int i = 0; i < WM / 16; ++i) {
            const uint8_t* row = xs + (mw + 16 * i + r) * G::XROW;
            if constexpr (XF32) {
                const v4f lo = *reinterpret_cast<const v4f*>(row + (((8 * ks + 2 * kq) ^ r) << 4));
                const v4f hi = *reinterpret_cast<const v4f*>(row + (((8 * ks + 2 * kq + 1) ^ r) << 4));
                fx[i] = __builtin_bit_cast(v8bf, (v4i){static_cast<int>(pack_bf16x2(lo[0], lo[1])),
                                                       static_cast<int>(pack_bf16x2(lo[2], lo[3])),
                                                       static_cast<int>(pack_bf16x2(hi[0], hi[1])),
                                                       static_cast<int>(pack_bf16x2(hi[2], hi[3]))});
            } else {
                fx[i] = *reinterpret_cast<const v8bf*>(row + (((4 * ks + kq) ^ r) << 4));
            }
        }
#pragma unroll
        for (int i = 0; i < WM / 16; ++i)
#pragma unroll
            for (int j = 0; j < TN / 16; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[j], fx[i], acc[i][j], 0, 0, 0);
    };

    const int T = K / G::KS;
#pragma unroll
    for (int d = 0; d < NS - 1; ++d)
        if (d < T) issue(d, d);
    int s = 0, slot = 0;
    for (; s + NS - 1 < T; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<(NS - 2) * PER>();
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(s + NS - 1, slot == 0 ? NS - 1 : slot - 1);
        compute(slot);
        slot = slot + 1 == NS ? 0 : slot + 1;
    }
    // the last NS - 1 stages: nothing left to refill
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<0>();
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    for (; s < T; ++s) {
        compute(slot);
        slot = slot + 1 == NS ? 0 : slot + 1;
    }
    __syncthreads();  // every wave is done with the ring: the partial tiles take its place

    constexpr int PITCH = TN + 4;
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < WM / 16; ++i)
#pragma unroll
        for (int j = 0; j < TN / 16; ++j)
            *reinterpret_cast<v4f*>(red + (ks * TM + mw + 16 * i + r) * PITCH + 16 * j + 4 * kq) = acc[i][j];
    __syncthreads();
    const bool vec_ok = (N & 3) == 0;
#pragma unroll
    for (int q = 0; q < (TM * TN / 4 + G::THR - 1) / G::THR; ++q) {
        const int idx = static_cast<int>(threadIdx.x) + G::THR * q;
        const int row = idx / (TN / 4);
        const int m = m0 + row;
        if (row >= TM || m >= M || col >= N) continue;
        const float* p = red + row * PITCH + (col - n0);
        v4f sum = *reinterpret_cast<const v4f*>(p);
#pragma unroll
        for (int w = 1; w < 4; ++w) sum += *reinterpret_cast<const v4f*>(p + w * TM * PITCH);
        float* o = out + static_cast<int64_t>(m) * N + col;
        v4f prev = {0.0f, 0.0f, 0.0f, 0.0f};
        if (accumulate) {
            if (vec_ok) {
                prev = *reinterpret_cast<const v4f*>(o);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (col + c < N) prev[c] = o[c];
            }
        }
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float t = sum[c];
            if (accumulate) t = t + prev[c];
            if (bias != nullptr) t = t + bv[c];
            if (GELU) t = gelu_tanh(t);
            v[c] = t;
        }
        if (out16 != nullptr) {
            uint16_t* o16 = out16 + m * ldo + col;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (col + c < N) o16[c] = f32_to_bf16(v[c]);
        } else if (vec_ok) {
            *reinterpret_cast<v4f*>(o) = (v4f){v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (col + c < N) o[c] = v[c];
        }
    }
}

// Shapes the tiled kernel does not take (K not a multiple of 32, or byte
// sizes past the 32-bit buffer range): one thread per output, products
// summed in k order.
template <bool XF32>
__global__ __launch_bounds__(256) void gemm_bf16_simple_kernel(const void* __restrict__ X,
                                                               const uint16_t* __restrict__ Wt,
                                                               const uint16_t* __restrict__ bias,
                                                               float* out, int M, int N, int K, int gelu,
                                                               int accumulate) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<int64_t>(M) * N) return;
    const int m = static_cast<int>(idx / N);
    const int n = static_cast<int>(idx % N);
    const uint16_t* w = Wt + static_cast<int64_t>(n) * K;
    float s = 0.0f;
    for (int k = 0; k < K; ++k) {
        float xv;
        if constexpr (XF32)
            xv = bf16_to_f32(f32_to_bf16(static_cast<const float*>(X)[static_cast<int64_t>(m) * K + k]));
        else
            xv = bf16_to_f32(static_cast<const uint16_t*>(X)[static_cast<int64_t>(m) * K + k]);
        s = __builtin_fmaf(xv, bf16_to_f32(w[k]), s);
    }
    if (accumulate) s = s + out[idx];
    if (bias != nullptr) s = s + bf16_to_f32(bias[n]);
    if (gelu) s = gelu_tanh(s);
    out[idx] = s;
}

template <bool XF32, int TMW, int TNW>
hipError_t launch_tiled_bf16(const void* x, int M, int K, const uint16_t* w, int N, const uint16_t* bias, float* out,
                             int gelu, int accumulate, hipStream_t stream) {
    constexpr int DEPTH = 4;
    const int tiles = ((M + 32 * TMW - 1) / (32 * TMW)) * ((N + 32 * TNW - 1) / (32 * TNW));
    if (gelu)
        hipLaunchKernelGGL((gemm_bf16_kernel<XF32, TMW, TNW, DEPTH, true>), dim3(tiles), dim3(BF_THR), 0, stream, x,
                           w, bias, out, M, N, K, accumulate);
    else
        hipLaunchKernelGGL((gemm_bf16_kernel<XF32, TMW, TNW, DEPTH, false>), dim3(tiles), dim3(BF_THR), 0, stream, x,
                           w, bias, out, M, N, K, accumulate);
    return hipGetLastError();
}

template <bool XF32, int TM, int TN>
hipError_t launch_dma_bf16(const void* x, int M, int K, const uint16_t* w, int N, const uint16_t* bias, float* out,
                           uint16_t* out16, int64_t ldx, int64_t ldo, int gelu, int accumulate, hipStream_t stream) {
    constexpr int THR = BfDma<XF32, TM, TN>::THR;
    const int tiles = ((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    if (gelu)
        hipLaunchKernelGGL((gemm_bf16_dma_kernel<XF32, TM, TN, true>), dim3(tiles), dim3(THR), 0, stream, x, w, bias,
                           out, out16, ldx, ldo, M, N, K, accumulate);
    else
        hipLaunchKernelGGL((gemm_bf16_dma_kernel<XF32, TM, TN, false>), dim3(tiles), dim3(THR), 0, stream, x, w, bias,
                           out, out16, ldx, ldo, M, N, K, accumulate);
    return hipGetLastError();
}

// The tile of gemm_bf16_dma_kernel: one workgroup per CU streams its rows
// through the CU's L2 port, so the launch takes about the rounds of 256
// workgroups times the bytes of a tile's rows.
template <bool XF32>
hipError_t launch_best_dma_bf16(const void* x, int M, int K, const uint16_t* w, int N, const uint16_t* bias,
                                float* out, uint16_t* out16, int64_t ldx, int64_t ldo, int gelu, int accumulate,
                                hipStream_t stream) {
    constexpr int tm[] = {64, 64, 32, 32, 16, 16}, tn[] = {64, 32, 64, 32, 64, 32};
    int best = 0;
    int64_t best_cost = INT64_MAX;
    for (int i = 0; i < 6; ++i) {
        const int64_t tiles = static_cast<int64_t>((M + tm[i] - 1) / tm[i]) * ((N + tn[i] - 1) / tn[i]);
        const int64_t cost = (tiles + 255) / 256 * (tm[i] * (XF32 ? 4 : 2) + tn[i] * 2);
        if (cost < best_cost) {
            best_cost = cost;
            best = i;
        }
    }
    switch (best) {
    case 0: return launch_dma_bf16<XF32, 64, 64>(x, M, K, w, N, bias, out, out16, ldx, ldo, gelu, accumulate, stream);
    case 1: return launch_dma_bf16<XF32, 64, 32>(x, M, K, w, N, bias, out, out16, ldx, ldo, gelu, accumulate, stream);
    case 2: return launch_dma_bf16<XF32, 32, 64>(x, M, K, w, N, bias, out, out16, ldx, ldo, gelu, accumulate, stream);
    case 3: return launch_dma_bf16<XF32, 32, 32>(x, M, K, w, N, bias, out, out16, ldx, ldo, gelu, accumulate, stream);
    case 4: return launch_dma_bf16<XF32, 16, 64>(x, M, K, w, N, bias, out, out16, ldx, ldo, gelu, accumulate, stream);
    default: return launch_dma_bf16<XF32, 16, 32>(x, M, K, w, N, bias, out, out16, ldx, ldo, gelu, accumulate, stream);
    }
}

}  // namespace

bool linear_bf16_large(int M, int K, int N) {
    return K % 64 == 0 && static_cast<int64_t>((M + 255) / 256) * ((N + 255) / 256) >= 128;
}

hipError_t launch_linear_bf16(const void* x, int x_dtype, int M, int K, const uint16_t* w, int N,
                              const uint16_t* bias, float* out, int gelu, hipStream_t stream, int accumulate) {
    if (M == 0 || N == 0) return hipSuccess;
    const bool xf32 = x_dtype == QIMG_FP32;
    const int64_t xbytes = static_cast<int64_t>(M) * K * (xf32 ? 4 : 2);
    const int64_t wbytes = static_cast<int64_t>(N) * K * 2;
    // Large problems with bf16 x (the INT4 linear's residual GEMM at 4096
    // tokens): the quantized linear's 256x256 tiles with bf16 MFMA.
    if (!xf32 && linear_bf16_large(M, K, N))
        return launch_gemm_bf16_large(static_cast<const uint16_t*>(x), M, K, w, N, bias, out, gelu, accumulate,
                                      stream);
    const bool tiled = (K % BF_KB) == 0 && xbytes < (int64_t{1} << 31) && wbytes < (int64_t{1} << 31);
    if (!tiled) {
        const int64_t total = static_cast<int64_t>(M) * N;
        const int blocks = static_cast<int>((total + 255) / 256);
        if (xf32)
            hipLaunchKernelGGL(gemm_bf16_simple_kernel<true>, dim3(blocks), dim3(256), 0, stream, x, w, bias, out, M,
                               N, K, gelu, accumulate);
        else
            hipLaunchKernelGGL(gemm_bf16_simple_kernel<false>, dim3(blocks), dim3(256), 0, stream, x, w, bias, out, M,
                               N, K, gelu, accumulate);
        return hipGetLastError();
    }
    const int64_t big = static_cast<int64_t>((M + 63) / 64) * ((N + 63) / 64);
    // K of at most 256 (img_in) and 256 or more tiles of 64x64 (its own 64x128
    // tiles are half as many): no split of K over the waves. Against the DMA
    // kernel's K of whole 128 the line is more than 256, its one round of
    // workgroups (us, fp32 x, DMA / short-K: 300x3072x128 4.4 / 4.4, 342 rows 6.9
    // / 4.6; 1024x1024x256 5.1 / 5.9, 342x3072x256 7.9 / 6.0, 16384x64x256 5.1 /
    // 5.5, 32768x64x256 11.5 / 8.3). Against gemm_bf16_kernel it is the faster
    // form from 64 rows of 3072 on (K = 64: 3.9 / 3.3, 300 rows 9.5 / 3.7, 512
    // 13.6 / 4.1); below 256 tiles that kernel is kept.
    if (K <= 256 && big >= (K % 128 == 0 ? 257 : 256) && N <= kShortKMaxN) {
        const int tiles = ((M + SK_M - 1) / SK_M) * ((N + SK_N - 1) / SK_N);
#define QIMG_SHORTK(XF, GL)                                                                                    \
    hipLaunchKernelGGL((gemm_bf16_shortk_kernel<XF, GL>), dim3(tiles), dim3(BF_THR), 0, stream, x, w, bias, out, M, \
                       N, K, accumulate)
        if (xf32) {
            if (gelu)
                QIMG_SHORTK(true, true);
            else
                QIMG_SHORTK(true, false);
        } else {
            if (gelu)
                QIMG_SHORTK(false, true);
            else
                QIMG_SHORTK(false, false);
        }
#undef QIMG_SHORTK
        return hipGetLastError();
    }
    if (K % 128 == 0)
        return xf32 ? launch_best_dma_bf16<true>(x, M, K, w, N, bias, out, nullptr, K, N, gelu, accumulate, stream)
                    : launch_best_dma_bf16<false>(x, M, K, w, N, bias, out, nullptr, K, N, gelu, accumulate, stream);
    // other K: direct fragment loads, 64x64 tiles when they give at least
    // 256 workgroups, otherwise 32x32
    if (M > 32 && big >= 256)
        return xf32 ? launch_tiled_bf16<true, 2, 2>(x, M, K, w, N, bias, out, gelu, accumulate, stream)
                    : launch_tiled_bf16<false, 2, 2>(x, M, K, w, N, bias, out, gelu, accumulate, stream);
    return xf32 ? launch_tiled_bf16<true, 1, 1>(x, M, K, w, N, bias, out, gelu, accumulate, stream)
                : launch_tiled_bf16<false, 1, 1>(x, M, K, w, N, bias, out, gelu, accumulate, stream);
}

hipError_t launch_linear_bf16_out16(const uint16_t* x, int M, int K, const uint16_t* w, int N, uint16_t* out,
                                    float* tmp, hipStream_t stream) {
    if (M == 0 || N == 0) return hipSuccess;
    if (linear_bf16_out16_direct(K, N)) return launch_linear_bf16_out16_ld(x, K, M, K, w, N, out, N, stream);
    const hipError_t e = launch_linear_bf16(x, QIMG_BF16, M, K, w, N, nullptr, tmp, 0, stream);
    return e == hipSuccess ? launch_f32_to_bf16(tmp, out, static_cast<int64_t>(M) * N, stream) : e;
}

// (wider products may suit the 256x256 tiles)
bool linear_bf16_out16_direct(int K, int N) { return K > 0 && K % 128 == 0 && N <= 256; }

hipError_t launch_linear_bf16_out16_ld(const uint16_t* x, int64_t ldx, int M, int K, const uint16_t* w, int N,
                                       uint16_t* out, int64_t ldo, hipStream_t stream) {
    if (M == 0 || N == 0) return hipSuccess;
    if (!linear_bf16_out16_direct(K, N)) return hipErrorInvalidValue;
    return launch_best_dma_bf16<false>(x, M, K, w, N, nullptr, nullptr, out, ldx, ldo, 0, 0, stream);
}

}  // namespace qimg
