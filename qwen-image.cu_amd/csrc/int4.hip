// int4.hip — the INT4 weight paths of qwen-image.cu (cuda_kernels.cu:
// 2864-4532) for gfx950: INT4 dequantization (NF4 grid, offset-8 linear and
// two's complement nibbles), the INT4 weight and activation quantizers, the
// W4A4 GEMM, the AWQ GEMV with its repacking, and the nunchaku layout
// conversions. Packed nibbles hold the even column in the low nibble.
//
// W4A4 GEMM. gfx950 has no 4-bit integer MFMA, so INT4 x INT4 runs on
// v_mfma_i32_32x32x32_i8: a 32-bit word of eight nibbles becomes two words of
// int8 lanes with one AND each, (w << 4) & 0xF0F0F0F0 and w & 0xF0F0F0F0: each
// byte is 16 x the signed nibble (two's complement in the high half of the
// byte), so the MFMA returns 256 x the exact dot product, and the 2^-8 goes
// into the activation scale. The element order inside a fragment is a
// permutation of k that is the same for both operands, so every dot product
// is the exact int32 sum of the reference's group. Each group's sum is then
// rescaled and accumulated in fp32 in the reference's operation order,
// acc = acc + ((float)d * as[g,m]) * ws[g,n] (w4a4_gemm_regdirect_kernel,
// cuda_kernels.cu:4206-4212), so the result is the same for every tiling.
#include <algorithm>

#include "qimg_device.h"
#include "qimg_internal.h"

namespace qimg {

namespace {

__constant__ float kNf4Grid[16] = {-1.0f,   -0.6962f, -0.5251f, -0.3949f, -0.2844f, -0.1848f,
                                   -0.0911f, 0.0f,    0.0796f,  0.1609f,  0.2461f,  0.3379f,
                                   0.4407f,  0.5626f, 0.7230f,  1.0f};

__device__ __forceinline__ int nib_signed(int n) { return n >= 8 ? n - 16 : n; }

// Value of code n before its scale.
__device__ __forceinline__ float int4_code(int n, int nf4, int signed_int4) {
    if (nf4) return kNf4Grid[n];
    return static_cast<float>(signed_int4 ? nib_signed(n) : n - 8);
}

// The row passes below take `per` threads a row. Short rows share a workgroup
// of SHORT_THR threads, rpw of them side by side; others are nb parts of THR
// threads. Workgroups stride over the rows. (One kernel for both, and a grid of
// parts by rows, cost the long rows 0.2 us.)
constexpr int ROW_THR = 128, SHORT_THR = 256;
struct RowThread {
    int row, sub;   // the thread's first row, and which of the workgroup's rows that is
    int col, step;  // its place in the row, and rows to the next one
    bool live;      // false: past the last of the rpw rows
};
template <bool SHORT, int THR>
__device__ __forceinline__ RowThread row_thread(int per, int nb) {
    const int tid = static_cast<int>(threadIdx.x);
    if constexpr (SHORT) {
        // quotients of numbers up to 256, at least 1/512 from the next integer
        const float inv = __builtin_amdgcn_rcpf(static_cast<float>(per));
        const int rpw = static_cast<int>((SHORT_THR + 0.5f) * inv);
        const int sub = static_cast<int>((static_cast<float>(tid) + 0.5f) * inv);
        return {static_cast<int>(blockIdx.x) * rpw + sub, sub, tid - sub * per, static_cast<int>(gridDim.x) * rpw,
                sub < rpw};
    }
    return {static_cast<int>(blockIdx.x / nb), 0, static_cast<int>(blockIdx.x % nb) * THR + tid,
            static_cast<int>(gridDim.x / nb), true};
}

// dequantize_int4_to_bf16_kernel (cuda_kernels.cu:2876-2917): one thread per
// 4 packed bytes (8 columns, one 16-byte bf16 store), K % 8 == 0. Bound by
// writing the output; the next row's words are loaded before this one's are
// used. With pad > 0 a row of out is K + pad long, columns K .. K + r taken
// from up [N, r] and the rest zero. A byte's two code values come from an LDS
// table (grid lookups from constant memory and 64-bit divisions per thread had
// made it 13.5 us at 3072 x 3072, 1.7 TB/s; now 9.4 us).
template <bool SHORT>
__global__ __launch_bounds__(SHORT ? SHORT_THR : ROW_THR) void dequant_int4_bf16_kernel(const uint8_t* __restrict__ qw,
                                                                const float* __restrict__ scales,
                                                                uint16_t* __restrict__ out, int N, int K, int gs,
                                                                int nf4, int scales_gn, int signed_int4,
                                                                const uint16_t* __restrict__ up, int r, int pad,
                                                                int nb) {
    __shared__ float2 table[256];
    for (int i = threadIdx.x; i < 256; i += SHORT ? SHORT_THR : ROW_THR)
        table[i] = make_float2(int4_code(i & 15, nf4, signed_int4), int4_code(i >> 4, nf4, signed_int4));
    __syncthreads();
    const int G = K / gs;
    const int64_t ldo = K + pad;
    const RowThread t = row_thread<SHORT, ROW_THR>((K + pad) / 8, nb);
    if (!t.live) return;
    const int word = t.col;
    const int c0 = word * 8;
    const int stride = t.step;
    int row = t.row;
    if (c0 >= K) {
        if (c0 >= ldo) return;
        for (; row < N; row += stride) {
            u32x4 o;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int j = c0 - K + 2 * p;
                const uint16_t* u = up + static_cast<int64_t>(row) * r + j;
                o[p] = (j < r ? u[0] : 0u) | ((j + 1 < r ? static_cast<uint32_t>(u[1]) : 0u) << 16);
            }
            reinterpret_cast<u32x4*>(out + row * ldo)[word] = o;
        }
        return;
    }
    const int g0 = c0 / gs;
    const bool one = (c0 + 7) / gs == g0;  // one group for the 8 columns
    auto code = [&](int n) {
        return reinterpret_cast<const uint32_t*>(qw + static_cast<int64_t>(n) * (K / 2))[word];
    };
    auto scale = [&](int n, int g) {
        return scales_gn ? scales[static_cast<int64_t>(g) * N + n] : scales[static_cast<int64_t>(n) * G + g];
    };
    uint32_t wn = row < N ? code(row) : 0u;
    float sn = row < N ? scale(row, g0) : 0.0f;
    for (; row < N; row += stride) {
        const uint32_t w = wn;
        const float s = sn;
        if (row + stride < N) {
            wn = code(row + stride);
            sn = scale(row + stride, g0);
        }
        u32x4 o;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float2 v = table[(w >> (8 * p)) & 0xff];
            const float s0 = one ? s : scale(row, (c0 + 2 * p) / gs);
            const float s1 = one ? s : scale(row, (c0 + 2 * p + 1) / gs);
            o[p] = pack_bf16x2(v.x * s0, v.y * s1);
        }
        reinterpret_cast<u32x4*>(out + row * ldo)[word] = o;
    }
}

// INT4 weight quantizers, one wave per (row, group): the linear form
// (quantize_linear_int4_per_group_kernel, cuda_kernels.cu:3226-3288) and NF4
// (quantize_int4_per_group_kernel, :3290-3357).
template <bool NF4>
__global__ __launch_bounds__(256) void quant_int4_weight_kernel(const float* __restrict__ r,
                                                                uint8_t* __restrict__ qw,
                                                                float* __restrict__ scales, int N, int K, int gs) {
    const int G = K / gs;
    const int64_t task = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (task >= static_cast<int64_t>(N) * G) return;
    const int lane = threadIdx.x & 63;
    const int64_t row = task / G;
    const int g = static_cast<int>(task % G);
    const float* p = r + row * K + static_cast<int64_t>(g) * gs;
    float amax = 0.0f;
    for (int i = lane; i < gs; i += 64) amax = fmaxf(amax, fabsf(p[i]));
    amax = wave_max(amax);
    const float scale = NF4 ? amax : amax / 7.0f;
    if (lane == 0) scales[row * G + g] = scale;
    const float inv = NF4 ? (scale > 0.0f ? 1.0f / scale : 0.0f) : (amax > 0.0f ? 7.0f / amax : 0.0f);
    for (int i = lane; i < gs / 2; i += 64) {
        int q[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float v = p[2 * i + e] * inv;
            if (NF4) {
                int best_j = 0;
                float best = 1e9f;
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const float d = fabsf(v - kNf4Grid[j]);
                    if (d < best) {
                        best = d;
                        best_j = j;
                    }
                }
                q[e] = best_j;
            } else {
                const int t = static_cast<int>(roundf(v));
                q[e] = (t < -7 ? -7 : (t > 7 ? 7 : t)) + 8;
            }
        }
        qw[row * (K / 2) + (static_cast<int64_t>(g) * gs) / 2 + i] = static_cast<uint8_t>(q[0] | (q[1] << 4));
    }
}

// Activation INT4 quant (quantize_activation_int4_kernel, cuda_kernels.cu:
// 3575-3636; with a smooth divide and a bf16 copy, fused_smooth_bf16_quant_
// kernel, :3650-3705). A thread owns V columns of a row; a group of gs
// columns is gs/V consecutive lanes of one wave (gs = 32, 64 or 128), reduced
// with lane exchanges. scales [G, M]. Bound by HBM, the IEEE divisions next:
// 8 columns (32 bytes in, 16 and 4 out) took 4352 x 3072 from 33.9 us (2.5
// TB/s; 2 columns, a 64-bit division per thread and 1-byte stores) to 20.2 us
// (4.3 TB/s). A few rows do not fill the chip, and a thread's chain of 8 is
// what counts: they have 2 columns a thread (16 x 3072 2.37 -> 2.19 us).
template <int GS, int V, bool SHORT>
__global__ __launch_bounds__(SHORT || V == 2 ? 256 : ROW_THR) void quant_act_int4_kernel(const float* __restrict__ x,
                                                                 const float* __restrict__ smooth,
                                                                 uint16_t* __restrict__ bf16_out,
                                                                 uint8_t* __restrict__ packed,
                                                                 float* __restrict__ scales, int M, int K, int nb) {
    typedef float vec __attribute__((ext_vector_type(V < 4 ? V : 4)));
    constexpr int E = V < 4 ? V : 4, H = V / E;  // elements per load, loads
    const RowThread t = row_thread<SHORT, V == 2 ? 256 : ROW_THR>(K / V, nb);
    const int c = t.col * V;
    // every lane takes part in the exchanges; lanes past the row or the last
    // row hold zeros
    const bool in_row = c < K && t.live;
    float sm[V];
    if (smooth != nullptr && in_row) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const vec u = reinterpret_cast<const vec*>(smooth + c)[h];
#pragma unroll
            for (int e = 0; e < E; ++e) sm[E * h + e] = u[e];
        }
    }
    // (m0: the workgroup's first row, for whole waves)
    for (int m0 = SHORT ? blockIdx.x * (t.step / gridDim.x) : t.row; m0 < M; m0 += t.step) {
        const int m = SHORT ? m0 + t.sub : m0;
        const bool live = SHORT ? in_row && m < M : in_row;
        float v[V] = {};
        if (live) {
#pragma unroll
            for (int h = 0; h < H; ++h) {
                const vec u = reinterpret_cast<const vec*>(x + static_cast<int64_t>(m) * K + c)[h];
#pragma unroll
                for (int e = 0; e < E; ++e) v[E * h + e] = u[e];
            }
            if (smooth != nullptr) {
#pragma unroll
                for (int e = 0; e < V; ++e) v[e] = v[e] / sm[e];
            }
            if (bf16_out != nullptr) {
                uint16_t* o = bf16_out + static_cast<int64_t>(m) * K + c;
                uint32_t w[V / 2];
#pragma unroll
                for (int e = 0; e < V / 2; ++e) w[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
                if constexpr (V == 8)
                    *reinterpret_cast<u32x4*>(o) = (u32x4){w[0], w[1], w[2], w[3]};
                else
                    *reinterpret_cast<uint32_t*>(o) = w[0];
            }
        }
        float amax = 0.0f;
#pragma unroll
        for (int e = 0; e < V; ++e) amax = fmaxf(amax, fabsf(v[e]));
#pragma unroll
        for (int off = 1; off < GS / V; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, kWave));
        if (!live) continue;
        if ((c % GS) == 0) scales[static_cast<int64_t>(c / GS) * M + m] = amax / 7.0f;
        const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            int q = static_cast<int>(roundf(v[e] * inv));
            q = q < -7 ? -7 : (q > 7 ? 7 : q);
            w |= static_cast<uint32_t>(q & 0xF) << (4 * e);
        }
        uint8_t* o = packed + static_cast<int64_t>(m) * (K / 2) + c / 2;
        if constexpr (V == 8)
            *reinterpret_cast<uint32_t*>(o) = w;
        else
            *o = static_cast<uint8_t>(w);
    }
}

// ---- W4A4 GEMM ---------------------------------------------------------
// The kernel is bound by the vector ALU: each group of 64 columns costs a
// 32 x 32 block two MFMAs (64 cycles of the matrix core) and 16 x 4 vector
// operations (a conversion, two products and a sum per accumulator in the
// reference's rounding order, 256 cycles), to which the compiled code of groups
// of 64 and 128 adds a copy of each MFMA result out of the accumulation
// registers (16 operations) and about 23 of unpacking and addressing: 415 in the
// loop of a stage of 2 x 2 groups and blocks, 106 us at 4352 x 3072 x 3072, group
// 64, and 2.4 GHz (the 16 x 4 alone: 65). So everything else is kept off the
// vector pipe's critical path: packed operands come by DMA into a two-slot LDS
// ring of 128 columns (one barrier a stage), and the outputs are laid out with n
// across the lanes, so a store writes 128 consecutive bytes of two rows and the
// activation scales are LDS broadcasts. A wave owns 32 x 64 outputs (four waves
// per SIMD; three for groups of 128, which hold 140 registers); 64 x 64 (two per
// SIMD, fewer unpacks per product) measured 134 against 112 us at 4352 x 3072 x
// 3072, group 64, and 48 against 30 us at 256 rows. Before, lanes ran across m
// (each 4-byte access touched 64 lines) and fragments were loaded straight from
// global memory: 254 us, and 19 us more for the low-rank product that is now
// multiplied here. 112 us is 0.73 POP/s.
constexpr int W4_THR = 256;   // four waves, 2 x 2
constexpr int W4_BM = 64;
constexpr int W4_BN = 128;
constexpr int W4_STG = 64;    // packed bytes of a row per stage (128 columns)

// Eight packed bytes (16 nibbles) -> one i8 MFMA fragment of 16 bytes, each
// 16 x its signed nibble.
__device__ __forceinline__ v4i unpack16(uint32_t x, uint32_t y) {
    return (v4i){static_cast<int>((x << 4) & 0xF0F0F0F0u), static_cast<int>(x & 0xF0F0F0F0u),
                 static_cast<int>((y << 4) & 0xF0F0F0F0u), static_cast<int>(y & 0xF0F0F0F0u)};
}

// out[m,n] = sum_g ((float)d_g * as[g,m]) * ws[g,n] + bias[n], onto the
// low-rank product lr[m,:] . up[n,:] (bf16 factors of rank r, r % 16 == 0,
// fp32 sums; the reference adds the residual to it, cuda_kernels.cu:4521) or,
// with `accumulate`, onto out's own values; then GELU (gelu_fp32,
// :4529-4531). CH: 64-column chunks of a group (0: any number, four waves per
// SIMD demanded, so that the sums carried from chunk to chunk stay in vector
// registers; copied from and to accumulation registers, with a select of zero
// at each chunk, 16 x 3072 x 3072 of group 192 took 33.4 us, now 26.6). The MFMA
// is issued as D = A x W^T: lane l holds column n = l % 32 and rows m = 8 (r/4)
// + 4 (l/32) + r%4 of each 32 x 32 block.
template <int CH, bool GELU>
__global__ __launch_bounds__(W4_THR, CH == 0 ? 4 : 1) void w4a4_gemm_kernel(const uint8_t* act,
                                                              const uint8_t* wgt,
                                                              const float* as,
                                                              const float* ws, float* out, int M, int N,
                                                              int K, int chunks, int accumulate,
                                                              const uint16_t* bias,
                                                              const uint16_t* lr,
                                                              const uint16_t* up, int r) {
    constexpr int NDMA = (W4_BM + W4_BN) / 16 / (W4_THR / 64);  // DMA instructions per wave and stage
    // One LDS object: with a second one, or with restrict arguments, the
    // compiler holds every LDS read until the DMA in flight has landed.
    constexpr int OPB = (W4_BM + W4_BN) * W4_STG;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * OPB + 4 * (W4_BM + W4_BN) * 4];
    float (*s_sc)[2][W4_BM + W4_BN] = reinterpret_cast<float (*)[2][W4_BM + W4_BN]>(lds + 2 * OPB);
    const int tiles_m = (M + W4_BM - 1) / W4_BM;
    const int tiles_n = (N + W4_BN - 1) / W4_BN;
    const int logical = xcd_remap(blockIdx.x, tiles_m * tiles_n);
    // M-tile fastest: consecutive workgroups share a weight slice
    const int m0 = (logical % tiles_m) * W4_BM;
    const int n0 = (logical / tiles_m) * W4_BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int h = lane >> 5;
    const int KB = K / 2;
    const int nch = K / 64;
    const int nst = (nch + 1) / 2;

    // A DMA instruction fills 16 rows x 64 bytes. Chunk c (16 bytes) of row t
    // sits at position c ^ ((t >> 2) & 3), so the 16 rows of a fragment read
    // cover all banks. Rows past the end repeat the last one (computed,
    // never stored); the half stage past an odd number of chunks repeats
    // the row's start (never used).
    const uint8_t* src[NDMA];
    int col[NDMA];
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
        const int t = (wave * NDMA + i) * 16 + (lane >> 2);
        col[i] = 16 * ((lane & 3) ^ ((t >> 2) & 3));
        const bool is_a = t < W4_BM;
        const int row = is_a ? m0 + t : n0 + t - W4_BM;
        const int last = (is_a ? M : N) - 1;
        src[i] = (is_a ? act : wgt) + static_cast<int64_t>(row < last ? row : last) * KB;
    }
    auto issue = [&](int st, int slot) {
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            const int c = st * W4_STG + col[i];
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(src[i] + (c < KB ? c : 0)),
                                             (lds_ptr_t)(lds + slot * OPB + (wave * NDMA + i) * 1024), 16, 0, 1);
        }
    };
    // The scales of a stage's two chunks: thread t carries row t's (as, times
    // the 2^-8 of the unpacking) or column t - W4_BM's.
    const bool sc_a = tid < W4_BM;
    const bool sc_live = tid < W4_BM + W4_BN;
    const int sc_i = sc_a ? (m0 + tid < M ? m0 + tid : M - 1) : (n0 + tid - W4_BM < N ? n0 + tid - W4_BM : N - 1);
    const int sc_stride = sc_a ? M : N;
    const float* sc_p = (sc_a ? as : ws) + sc_i;
    const float sc_mul = sc_a ? 0.00390625f : 1.0f;
    float sc[2] = {0.0f, 0.0f};
    auto load_sc = [&](int st) {
        if (!sc_live) return;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = 2 * st + u < nch ? 2 * st + u : nch - 1;
            sc[u] = sc_p[static_cast<int64_t>(CH == 1 ? c : c / (CH ? CH : chunks)) * sc_stride];
        }
    };
    auto store_sc = [&](int slot) {
        if (!sc_live) return;
#pragma unroll
        for (int u = 0; u < 2; ++u) s_sc[slot][u][tid] = sc[u] * sc_mul;
    };

    float acc[2][16];
    v16i d[CH == 0 ? 2 : 1];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;

    auto mfma2 = [&](const u32x4& a, const u32x4& w, v16i c) {
        c = __builtin_amdgcn_mfma_i32_32x32x32_i8(unpack16(a.x, a.y), unpack16(w.x, w.y), c, 0, 0, 0);
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(unpack16(a.z, a.w), unpack16(w.z, w.w), c, 0, 0, 0);
    };
    // (float)(d >> 8) * sa == (float)d * (sa * 2^-8): d = 256 x an exact sum
    // below 2^24 in magnitude, and the power-of-two scaling is exact, so the
    // product rounds identically.
    auto rescale = [&](const v16i& dd, float (&o)[16], const float* s_a, float sw) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4f sa = *reinterpret_cast<const v4f*>(s_a + 8 * q);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
#pragma clang fp contract(off)
                const float t = static_cast<float>(dd[4 * q + c]) * sa[c];
                o[4 * q + c] = o[4 * q + c] + t * sw;
            }
        }
    };
    const int arow = wm * 32 + (lane & 31);
    const int wrow = wn * 64 + (lane & 31);
    const int sw8 = ((lane & 31) >> 2) & 3;  // rows 32 apart share it

    issue(0, 0);
    load_sc(0);
    store_sc(0);
    int cg = 0;
    for (int st = 0; st < nst; ++st) {
        const int slot = st & 1;
        wait_vmcnt<0>();  // this wave's part of the stage, issued a stage ago
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (st + 1 < nst) {
            issue(st + 1, slot ^ 1);
            load_sc(st + 1);
        }
        const uint8_t* ob = lds + slot * OPB;
        if constexpr (CH == 2) {
            u32x4 a[2], w[2][2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int off = 16 * ((2 * u + h) ^ sw8);
                a[u] = *reinterpret_cast<const u32x4*>(ob + arow * W4_STG + off);
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    w[j][u] = *reinterpret_cast<const u32x4*>(ob + (W4_BM + wrow + 32 * j) * W4_STG + off);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const v16i zero = {};
                const v16i dd = mfma2(a[1], w[j][1], mfma2(a[0], w[j][0], zero));
                rescale(dd, acc[j], &s_sc[slot][0][wm * 32 + 4 * h], s_sc[slot][0][W4_BM + wrow + 32 * j]);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (2 * st + u >= nch) break;
                const int off = 16 * ((2 * u + h) ^ sw8);
                const u32x4 a = *reinterpret_cast<const u32x4*>(ob + arow * W4_STG + off);
                u32x4 w[2];
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    w[j] = *reinterpret_cast<const u32x4*>(ob + (W4_BM + wrow + 32 * j) * W4_STG + off);
                const bool first = CH == 1 || cg == 0;
                const bool last = CH == 1 || cg + 1 == chunks;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const v16i zero = {};
                    v16i& dd = d[CH == 0 ? j : 0];
                    if (first)  // a branch: a select is 16 operations a block
                        dd = mfma2(a, w[j], zero);
                    else
                        dd = mfma2(a, w[j], dd);
                    if (last)
                        rescale(dd, acc[j], &s_sc[slot][u][wm * 32 + 4 * h], s_sc[slot][u][W4_BM + wrow + 32 * j]);
                }
                cg = last ? 0 : cg + 1;
            }
        }
        if (st + 1 < nst) store_sc(slot ^ 1);
    }

    typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
    const int mb = m0 + wm * 32;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wrow + 32 * j;
        v16f low;
#pragma unroll
        for (int e = 0; e < 16; ++e) low[e] = 0.0f;
        if (lr != nullptr) {
            const int ml = mb + (lane & 31) < M ? mb + (lane & 31) : M - 1;
            const uint16_t* pl = lr + static_cast<int64_t>(ml) * r + 8 * h;
            const uint16_t* pu = up + static_cast<int64_t>(n < N ? n : N - 1) * r + 8 * h;
            for (int k = 0; k < r; k += 16)
                low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const v8bf*>(pl + k),
                                                              *reinterpret_cast<const v8bf*>(pu + k), low, 0, 0, 0);
        }
        if (n >= N) continue;
        const float b = bias != nullptr ? bf16_to_f32(bias[n]) : 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = mb + 8 * (e >> 2) + 4 * h + (e & 3);
            if (m >= M) continue;
            float* o = out + static_cast<int64_t>(m) * N + n;
            float v;
            {
#pragma clang fp contract(off)
                v = acc[j][e] + b;
                if (lr != nullptr) v = low[e] + v;
                if (accumulate) v = *o + v;
            }
            *o = GELU ? gelu_tanh(v) : v;
        }
    }
}

// ---- AWQ ----------------------------------------------------------------
// AWQ kInterleave=4 nibble address (cuda_kernels.cu:3072-3085).
__device__ __forceinline__ int awq_nibble(const int32_t* qw, int IC, int oc, int ic) {
    const int i16 = ((ic >> 6) << 6) + (oc & 3) * 16 + (((ic & 63) >> 5) << 3) + (ic & 7);
    const int bit = ((i16 & 1) << 4) + (((ic >> 3) & 3) << 2);
    return static_cast<int>((static_cast<uint32_t>(qw[static_cast<int64_t>(oc >> 2) * (IC / 2) + (i16 >> 1)]) >> bit) &
                            0xF);
}

// repack_awq_kernel (cuda_kernels.cu:3059-3091): [OC/4, IC/2] -> [IC/8, OC].
__global__ __launch_bounds__(256) void awq_repack_kernel(const int32_t* __restrict__ qw, int32_t* __restrict__ out,
                                                         int OC, int IC) {
    const int oc = blockIdx.x * blockDim.x + threadIdx.x;
    const int ig = blockIdx.y;
    if (oc >= OC) return;
    uint32_t w = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) w |= static_cast<uint32_t>(awq_nibble(qw, IC, oc, ig * 8 + k)) << (4 * k);
    out[static_cast<int64_t>(ig) * OC + oc] = static_cast<int32_t>(w);
}

// dequantize_awq_to_bf16_kernel (cuda_kernels.cu:3002-3038).
__global__ __launch_bounds__(256) void awq_dequant_kernel(const int32_t* __restrict__ qw,
                                                          const uint16_t* __restrict__ wscales,
                                                          const uint16_t* __restrict__ wzeros,
                                                          uint16_t* __restrict__ out, int OC, int IC, int gs,
                                                          int ncomp) {
    const int64_t total = static_cast<int64_t>(OC) * IC;
    const int dim = OC / ncomp;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int so = static_cast<int>(i / IC);
        const int ic = static_cast<int>(i % IC);
        const int nk = (so % dim) * ncomp + so / dim;
        const int g = ic / gs;
        const float s = bf16_to_f32(wscales[static_cast<int64_t>(g) * OC + nk]);
        const float z = bf16_to_f32(wzeros[static_cast<int64_t>(g) * OC + nk]);
        float w;
        {
#pragma clang fp contract(off)
            w = static_cast<float>(awq_nibble(qw, IC, nk, ic)) * s + z;
        }
        out[i] = f32_to_bf16(w);
    }
}

// awq_gemv_repacked_kernel (cuda_kernels.cu:3106-3153), M = 1, gs = 64. The
// sum over ic runs in order, so each output channel is one dependent chain of
// IC additions, and a dependent v_add_f32 takes 8.25 cycles: 3072 of them are
// 10.6 us at 2.4 GHz. Everything else is taken off that chain. A workgroup
// owns 64 channels, one per lane: eight waves load the weight words, form the
// products and put them in a two-slot LDS ring of 128 inputs; a ninth wave, first
// in the issue order, reads them (16 bytes a lane, the next 32 inputs while it
// adds the last) and adds. From the second stage on the words are loaded
// AWQ_DEPTH stages ahead; the compiler sinks the first loads below the barrier
// that x waits for, which the ninth wave copies alone, so a launch starts with
// both latencies in a row. q * s is exact in fp32 (4 bits x a bf16's 8), so
// fma(q, s, z) is the reference's q * s + z.
// 18432 x 3072 (32 MB of weights and scales): 22.4 us; one wave per 64 channels
// doing all of it took 74.6. With x in scalar registers, whose load latency
// falls on every stage's barrier, 32.7; with the last sums' operands read in
// one go (134 registers, so that two workgroups do not share a CU), 36.
constexpr int AWQ_PW = 8;     // producer waves
constexpr int AWQ_DEPTH = 4;  // stages of weight words in flight per producer
constexpr int AWQ_THR = 64 * (AWQ_PW + 1);
constexpr int AWQ_RING = 2 * 32 * 64;  // [slot][4 inputs][channel], 16 bytes each

__global__ __launch_bounds__(AWQ_THR, 5) void awq_gemv_kernel(const float* __restrict__ x, const int32_t* __restrict__ qw,
                                                           const uint16_t* __restrict__ wscales,
                                                           const uint16_t* __restrict__ wzeros,
                                                           const uint16_t* __restrict__ bias, float* __restrict__ out,
                                                           int OC, int IC, int ncomp) {
    constexpr int WPP = 16 / AWQ_PW;  // words of 8 inputs per producer and stage
    extern __shared__ __attribute__((aligned(16))) v4f awq_lds[];  // the ring, then x
    v4f* sx = awq_lds + AWQ_RING;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nk_raw = blockIdx.x * 64 + lane;
    const bool live = nk_raw < OC;
    const int nk = live ? nk_raw : OC - 1;
    const int G = IC / 64;
    // Stages in whole rounds of AWQ_DEPTH, so that the producers' loop has no
    // exit inside a round and the loads in flight are counted exactly.
    const int nst = ((G + 1) / 2 + AWQ_DEPTH - 1) / AWQ_DEPTH * AWQ_DEPTH;
    // one barrier a stage: slot st & 1 is full, and the other one is read
    auto stage_barrier = [] {
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    if (wave < AWQ_PW) {
        const int w0 = wave * WPP;  // first of the stage's 16 words
        uint32_t q[AWQ_DEPTH][WPP];
        uint16_t s16[AWQ_DEPTH], z16[AWQ_DEPTH];
        // Stages past the end (and the half stage past an odd G) read the
        // last group again; its products are never added.
        auto group_of = [&](int st) {
            const int g = 2 * st + (w0 >> 3);
            return g < G ? g : G - 1;
        };
        auto load = [&](int d, int st) {
            const int g = group_of(st);
            const int32_t* p = qw + static_cast<int64_t>(g * 8 + (w0 & 7)) * OC + nk;
#pragma unroll
            for (int i = 0; i < WPP; ++i) q[d][i] = static_cast<uint32_t>(p[static_cast<int64_t>(i) * OC]);
            s16[d] = wscales[static_cast<int64_t>(g) * OC + nk];
            z16[d] = wzeros[static_cast<int64_t>(g) * OC + nk];
        };
#pragma unroll
        for (int d = 0; d < AWQ_DEPTH; ++d) load(d, d);
        stage_barrier();  // x is in LDS
        v4f xs[2 * WPP];
        auto load_x = [&](int st) {
            const v4f* xg = sx + group_of(st) * 16 + (w0 & 7) * 2;
#pragma unroll
            for (int i = 0; i < 2 * WPP; ++i) xs[i] = xg[i];
        };
        load_x(0);
        for (int st0 = 0; st0 < nst; st0 += AWQ_DEPTH) {
#pragma unroll
            for (int d = 0; d < AWQ_DEPTH; ++d) {
                const int st = st0 + d;
                v4f v[2 * WPP];
                const float s = bf16_to_f32(s16[d]), z = bf16_to_f32(z16[d]);
#pragma unroll
                for (int i = 0; i < WPP; ++i) {
                    const uint32_t ev = q[d][i] & 0x0F0F0F0Fu, od = (q[d][i] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const float n = static_cast<float>(((k & 1 ? od : ev) >> (8 * (k >> 1))) & 0xFFu);
                        v[2 * i + (k >> 2)][k & 3] = __builtin_fmaf(n, s, z) * xs[2 * i + (k >> 2)][k & 3];
                    }
                }
                load(d, st + AWQ_DEPTH);
                v4f* ring = awq_lds + (st & 1) * (AWQ_RING / 2) + 2 * w0 * 64 + lane;
#pragma unroll
                for (int i = 0; i < 2 * WPP; ++i) ring[i * 64] = v[i];
                load_x(st + 1);
                stage_barrier();
            }
        }
        return;
    }
    for (int i = lane; i < IC / 4; i += 64) sx[i] = reinterpret_cast<const v4f*>(x)[i];
    stage_barrier();
    __builtin_amdgcn_s_setprio(3);
    float acc = 0.0f;
    v4f va[8], vb[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) vb[c] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    auto read = [&](v4f (&v)[8], int st, int u) {
        const v4f* p = awq_lds + (st & 1) * (AWQ_RING / 2) + 8 * u * 64 + lane;
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = p[c * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const v4f (&v)[8]) {
#pragma clang fp contract(off)
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = acc + v[c][e];
        __builtin_amdgcn_sched_barrier(0);
    };
    int st = 0;
    for (; st < G / 2; ++st) {
        stage_barrier();
        read(va, st, 0);
        add(vb);  // the last stage's last quarter (zeros at first)
        read(vb, st, 1);
        add(va);
        read(va, st, 2);
        add(vb);
        read(vb, st, 3);
        add(va);
    }
    add(vb);
    for (; st < nst; ++st) {
        stage_barrier();
        if (2 * st < G) {  // the last of an odd number of groups
            read(va, st, 0);
            read(vb, st, 1);
            add(va);
            add(vb);
        }
    }
    if (!live) return;
    const int dim = OC / ncomp;
    const int so = (nk % ncomp) * dim + nk / ncomp;
    if (bias != nullptr) acc = acc + bf16_to_f32(bias[so]);
    out[so] = acc;
}

// The same with one wave per 64 channels doing all of it, the next group's
// eight words loaded while this one is summed: for a few groups, where the
// ring's prologue costs more than the chain, and for more channels than the
// ring's workgroups can be on the chip at once (awq_short has the line).
__global__ __launch_bounds__(64) void awq_gemv_short_kernel(const float* __restrict__ x, const int32_t* __restrict__ qw,
                                                            const uint16_t* __restrict__ wscales,
                                                            const uint16_t* __restrict__ wzeros,
                                                            const uint16_t* __restrict__ bias, float* __restrict__ out,
                                                            int OC, int IC, int ncomp) {
    extern __shared__ float s_x[];
    for (int i = threadIdx.x; i < IC; i += blockDim.x) s_x[i] = x[i];
    __syncthreads();
    const int nk_raw = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = nk_raw < OC;
    const int nk = live ? nk_raw : OC - 1;
    const int G = IC / 64;
    auto load = [&](int g, uint32_t* p, uint16_t& s, uint16_t& z) {
#pragma unroll
        for (int io = 0; io < 8; ++io) p[io] = static_cast<uint32_t>(qw[static_cast<int64_t>(g * 8 + io) * OC + nk]);
        s = wscales[static_cast<int64_t>(g) * OC + nk];
        z = wzeros[static_cast<int64_t>(g) * OC + nk];
    };
    uint32_t p[8], pn[8];
    uint16_t s16, z16, sn16 = 0, zn16 = 0;
    load(0, p, s16, z16);
    float acc = 0.0f;
    for (int g = 0; g < G; ++g) {
        if (g + 1 < G) load(g + 1, pn, sn16, zn16);
        const float s = bf16_to_f32(s16);
        const float z = bf16_to_f32(z16);
        const v4f* xv = reinterpret_cast<const v4f*>(s_x + g * 64);
#pragma unroll
        for (int io = 0; io < 8; ++io) {
            const v4f x0 = xv[2 * io], x1 = xv[2 * io + 1];
            const float xs[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
#pragma clang fp contract(off)
                const float w = static_cast<float>((p[io] >> (4 * k)) & 0xF) * s + z;
                acc = acc + w * xs[k];
            }
        }
#pragma unroll
        for (int io = 0; io < 8; ++io) p[io] = pn[io];
        s16 = sn16;
        z16 = zn16;
    }
    if (!live) return;
    const int dim = OC / ncomp;
    const int so = (nk % ncomp) * dim + nk / ncomp;
    if (bias != nullptr) acc = acc + bf16_to_f32(bias[so]);
    out[so] = acc;
}

// ---- nunchaku layouts ----------------------------------------------------
// MMA-swizzled nibble and scale addresses (cuda_kernels.cu:2945-2973).
__device__ __forceinline__ int nk_nibble(const uint8_t* q, int K, int row, int col) {
    const int kt = K / 64, nt = row / 128, nw = row % 128;
    const int np = nw / 16, ps = (nw % 16) / 8, nl = nw % 8;
    const int ktile = col / 64, kps = (col % 64) / 32, kl = (col % 32) / 8, rk = col % 8;
    const int64_t i32 = static_cast<int64_t>(nt) * (kt * 1024) + ktile * 1024 + np * 128 + nl * 16 + kl * 4 + ps * 2 + kps;
    return (q[i32 * 4 + rk / 2] >> ((rk % 2) * 4)) & 0xF;
}

__device__ __forceinline__ int64_t nk_scale_off(int G, int row, int g) {
    const int nt = row / 128, nw = row % 128;
    return static_cast<int64_t>(nt) * G * 128 + g * 128 + (nw / 16) * 16 + ((nw % 8) / 2) * 4 + ((nw % 16) / 8) * 2 +
           nw % 2;
}

// unswizzle_nunchaku_weights_kernel (cuda_kernels.cu:3431-3487).
__global__ __launch_bounds__(256) void nk_unswizzle_kernel(const uint8_t* __restrict__ q_sw,
                                                           const uint16_t* __restrict__ s_sw,
                                                           uint8_t* __restrict__ q_rm, float* __restrict__ s_rm,
                                                           int N, int K, int G) {
    const int64_t total = static_cast<int64_t>(N) * (K / 2);
    const int gs = K / G;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int row = static_cast<int>(i / (K / 2));
        const int c0 = static_cast<int>(i % (K / 2)) * 2;
        q_rm[i] = static_cast<uint8_t>(nk_nibble(q_sw, K, row, c0) | (nk_nibble(q_sw, K, row, c0 + 1) << 4));
        if (c0 % gs == 0) s_rm[static_cast<int64_t>(c0 / gs) * N + row] = bf16_to_f32(s_sw[nk_scale_off(G, row, c0 / gs)]);
    }
}

// dequantize_nunchaku_to_bf16_kernel (cuda_kernels.cu:2932-2978).
__global__ __launch_bounds__(256) void nk_dequant_kernel(const uint8_t* __restrict__ q_sw,
                                                         const uint16_t* __restrict__ s_sw,
                                                         uint16_t* __restrict__ out, int N, int K, int G) {
    const int64_t total = static_cast<int64_t>(N) * K;
    const int gs = K / G;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int row = static_cast<int>(i / K);
        const int col = static_cast<int>(i % K);
        const float s = bf16_to_f32(s_sw[nk_scale_off(G, row, col / gs)]);
        out[i] = f32_to_bf16(static_cast<float>(nib_signed(nk_nibble(q_sw, K, row, col))) * s);
    }
}

// unswizzle_lora_weights_kernel (cuda_kernels.cu:3503-3562).
__global__ __launch_bounds__(256) void lora_unswizzle_kernel(const uint16_t* __restrict__ packed,
                                                             uint16_t* __restrict__ out, int rows, int cols,
                                                             int is_down) {
    const int64_t total = static_cast<int64_t>(rows) * cols;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int row = static_cast<int>(i / cols);
        const int col = static_cast<int>(i % cols);
        const int sr = is_down ? col : row, sc = is_down ? row : col;
        const int cf = is_down ? sc / 16 : sr / 16, rf = is_down ? sr / 16 : sc / 16;
        const int ln = sr % 16, lk = sc % 16;
        const int64_t f = static_cast<int64_t>(cf) * 16 * cols + rf * 256 + (ln % 8) * 32 + ((lk % 8) / 2) * 8 +
                          (ln / 8) * 4 + (lk / 8) * 2 + lk % 2;
        out[i] = packed[f];
    }
}

// bf16 transpose [R, C] -> [C, R] (the low-rank down projection is stored
// [K, r]; the GEMM takes its weight as [r, K]).
__global__ __launch_bounds__(256) void transpose_u16_kernel(const uint16_t* __restrict__ in,
                                                            uint16_t* __restrict__ out, int R, int C) {
    const int64_t total = static_cast<int64_t>(R) * C;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int c = static_cast<int>(i / R);
        const int r = static_cast<int>(i % R);
        out[i] = in[static_cast<int64_t>(r) * C + c];
    }
}

// fp32 -> bf16, round to nearest even (fp32_to_bf16, cuda_kernels.cu:33-42).
__global__ __launch_bounds__(256) void f32_to_bf16_kernel(const float* __restrict__ in, uint16_t* __restrict__ out,
                                                          int64_t n) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        out[i] = f32_to_bf16(in[i]);
}

// bf16 -> fp32 (bf16_to_fp32, cuda_kernels.cu:22-31): exact widening.
__global__ __launch_bounds__(256) void bf16_to_f32_kernel(const uint16_t* __restrict__ in, float* __restrict__ out,
                                                          int64_t n) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        out[i] = bf16_to_f32(in[i]);
}

int grid_for(int64_t n, int per_block = 256) {
    const int64_t b = (n + per_block - 1) / per_block;
    return static_cast<int>(b < 65536 ? (b > 0 ? b : 1) : 65536);
}

// Parts of a row and grid of a row pass with `per` threads a row, at most
// `most` workgroups (below 2^24: a launch holds fewer than 2^32 threads).
struct RowGrid {
    int nb;
    unsigned blocks;
};
RowGrid row_grid(int rows, int per, bool is_short, int threads, int most) {
    if (is_short) {
        const int rpw = SHORT_THR / per, parts = (rows - 1) / rpw + 1;
        return {1, static_cast<unsigned>(std::min(parts, most))};
    }
    const int nb = (per + threads - 1) / threads;
    return {nb, static_cast<unsigned>(nb) * std::min(rows, nb < most ? most / nb : 1)};
}

}  // namespace

hipError_t launch_dequant_int4_bf16(const uint8_t* qw, const float* scales, uint16_t* out, int N, int K, int gs,
                                    int nf4, int scales_gn, int signed_int4, hipStream_t stream) {
    return launch_dequant_int4_bf16_ext(qw, scales, out, N, K, gs, nf4, scales_gn, signed_int4, nullptr, 0, 0, stream);
}

hipError_t launch_dequant_int4_bf16_ext(const uint8_t* qw, const float* scales, uint16_t* out, int N, int K, int gs,
                                        int nf4, int scales_gn, int signed_int4, const uint16_t* up, int r, int pad,
                                        hipStream_t stream) {
    if (N == 0 || K == 0) return hipSuccess;
    if (K % 8 != 0 || gs <= 0 || K % gs != 0 || pad < r || pad % 8 != 0) return hipErrorInvalidValue;
    // at most 4096 workgroups: each loads its table for a few rows
    const int per = (K + pad) / 8;
    // short: rows that would leave more than half of ROW_THR idle (us, one row
    // a workgroup / side by side: 50000 x 8 8.7 / 2.6, 12288 x 64 5.3 / 2.8,
    // 3072 x 256 4.0 / 2.8; 12288 x 512 6.5 / 7.4)
    const bool is_short = per < 64;
    const RowGrid g = row_grid(N, per, is_short, ROW_THR, 4096);
    if (is_short)
        hipLaunchKernelGGL(dequant_int4_bf16_kernel<true>, dim3(g.blocks), dim3(SHORT_THR), 0, stream, qw, scales, out,
                           N, K, gs, nf4, scales_gn, signed_int4, up, r, pad, g.nb);
    else
        hipLaunchKernelGGL(dequant_int4_bf16_kernel<false>, dim3(g.blocks), dim3(ROW_THR), 0, stream, qw, scales, out,
                           N, K, gs, nf4, scales_gn, signed_int4, up, r, pad, g.nb);
    return hipGetLastError();
}

hipError_t launch_quant_int4_weight(const float* r, uint8_t* qw, float* scales, int N, int K, int gs, int nf4,
                                    hipStream_t stream) {
    if (N == 0 || K == 0) return hipSuccess;
    if (gs <= 0 || gs % 2 != 0 || K % gs != 0) return hipErrorInvalidValue;
    const int64_t tasks = static_cast<int64_t>(N) * (K / gs);
    const int blocks = static_cast<int>((tasks + 3) / 4);
    if (nf4)
        hipLaunchKernelGGL(quant_int4_weight_kernel<true>, dim3(blocks), dim3(256), 0, stream, r, qw, scales, N, K, gs);
    else
        hipLaunchKernelGGL(quant_int4_weight_kernel<false>, dim3(blocks), dim3(256), 0, stream, r, qw, scales, N, K,
                           gs);
    return hipGetLastError();
}

template <int GS, int V>
static void run_quant_act(const float* x, const float* smooth, uint16_t* bf16_out, uint8_t* packed, float* scales,
                          int M, int K, hipStream_t stream) {
    constexpr int THR = V == 2 ? 256 : ROW_THR;
    // 8 columns: as in the dequantization (30000 x 64 13.0 -> 2.9 us, 4352 x 128
    // 3.8 -> 2.5)
    const bool is_short = K / V < (V == 2 ? SHORT_THR : 64);
    const RowGrid g = row_grid(M, K / V, is_short, THR, 1 << 23);
    if (is_short)
        hipLaunchKernelGGL((quant_act_int4_kernel<GS, V, true>), dim3(g.blocks), dim3(SHORT_THR), 0, stream, x, smooth,
                           bf16_out, packed, scales, M, K, g.nb);
    else
        hipLaunchKernelGGL((quant_act_int4_kernel<GS, V, false>), dim3(g.blocks), dim3(THR), 0, stream, x, smooth,
                           bf16_out, packed, scales, M, K, g.nb);
}

hipError_t launch_quant_act_int4(const float* x, const float* smooth, uint16_t* bf16_out, uint8_t* packed,
                                 float* scales, int M, int K, int gs, hipStream_t stream) {
    if (M == 0 || K == 0) return hipSuccess;
    if ((gs != 32 && gs != 64 && gs != 128) || K % gs != 0) return hipErrorInvalidValue;
    // us, 2 / 8 columns a thread: 16 x 3072 2.19 / 2.37, 128 x 3072 2.5 / 2.6,
    // 128 x 128 2.1 / 2.4; past the line 192 x 3072 2.8 / 2.7, 512 x 1024 2.8 /
    // 2.7; rows that are no whole workgroups of 8 columns 128 x 1056 2.5 / 2.3,
    // 128 x 1536 2.5 / 2.25
    const bool few = static_cast<int64_t>(M) * K <= 3 << 17 && (K < 512 || K % 1024 == 0);
    auto* run = few
                    ? (gs == 32 ? run_quant_act<32, 2> : gs == 64 ? run_quant_act<64, 2> : run_quant_act<128, 2>)
                    : (gs == 32 ? run_quant_act<32, 8> : gs == 64 ? run_quant_act<64, 8> : run_quant_act<128, 8>);
    run(x, smooth, bf16_out, packed, scales, M, K, stream);
    return hipGetLastError();
}

template <int CH>
static void run_w4a4(unsigned tiles, const uint8_t* act, const uint8_t* wgt, const float* as, const float* ws, float* out,
                     int M, int N, int K, int gs, int accumulate, const uint16_t* bias, const uint16_t* lr,
                     const uint16_t* up, int r, int gelu, hipStream_t stream) {
    if (gelu)
        hipLaunchKernelGGL((w4a4_gemm_kernel<CH, true>), dim3(tiles), dim3(W4_THR), 0, stream, act, wgt, as, ws, out,
                           M, N, K, gs / 64, accumulate, bias, lr, up, r);
    else
        hipLaunchKernelGGL((w4a4_gemm_kernel<CH, false>), dim3(tiles), dim3(W4_THR), 0, stream, act, wgt, as, ws, out,
                           M, N, K, gs / 64, accumulate, bias, lr, up, r);
}

hipError_t launch_w4a4_gemm(const uint8_t* act, const uint8_t* wgt, const float* as, const float* ws, float* out,
                            int M, int N, int K, int gs, int accumulate, const uint16_t* bias, const uint16_t* lr,
                            const uint16_t* up, int r, int gelu, hipStream_t stream) {
    if (M == 0 || N == 0) return hipSuccess;
    if (gs <= 0 || gs % 64 != 0 || K % gs != 0 || (lr != nullptr && (up == nullptr || r <= 0 || r % 16 != 0)))
        return hipErrorInvalidValue;
    const int64_t tiles = static_cast<int64_t>((M + W4_BM - 1) / W4_BM) * ((N + W4_BN - 1) / W4_BN);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    auto* run = gs == 64 ? run_w4a4<1> : gs == 128 ? run_w4a4<2> : run_w4a4<0>;
    run(static_cast<unsigned>(tiles), act, wgt, as, ws, out, M, N, K, gs, accumulate, bias, lr, up, r, gelu, stream);
    return hipGetLastError();
}

hipError_t launch_awq_repack(const int32_t* qw, int32_t* out, int OC, int IC, hipStream_t stream) {
    if (OC == 0 || IC == 0) return hipSuccess;
    if (OC % 4 != 0 || IC % 64 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(awq_repack_kernel, dim3((OC + 255) / 256, IC / 8), dim3(256), 0, stream, qw, out, OC, IC);
    return hipGetLastError();
}

hipError_t launch_awq_dequant(const int32_t* qw, const uint16_t* wscales, const uint16_t* wzeros, uint16_t* out,
                              int OC, int IC, int gs, int ncomp, hipStream_t stream) {
    if (OC == 0 || IC == 0) return hipSuccess;
    if (OC % 4 != 0 || IC % 64 != 0 || gs <= 0 || IC % gs != 0 || ncomp <= 0 || OC % ncomp != 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(awq_dequant_kernel, dim3(grid_for(static_cast<int64_t>(OC) * IC)), dim3(256), 0, stream, qw,
                       wscales, wzeros, out, OC, IC, gs, ncomp);
    return hipGetLastError();
}

// Which AWQ kernel, by how often over the ring's workgroups fill the chip (two
// fit a CU up to 4096 inputs, later one). us, awq_gemv_short_kernel / the ring:
// up to once, 18432 channels of 128 inputs 4.1 / 5.1, of 192 5.4 / 5.3, of 256
// 6.4 / 5.3; to 1.5 times, 36864 of 320 7.8 / 8.1, of 384 9.0 / 8.1; to 2.5
// times, 64000 of 768 15.5 / 19.1, 73728 of 1024 27.4 / 22.6; from there 98304
// of 896 24 / 28, of 3072 75 / 77, 147456 of 2048 65 / 74.
static bool awq_short(int OC, int IC) {
    const int at_once = 256 * (IC <= 4096 ? 2 : 1), wgs = (OC + 63) / 64;
    return 2 * wgs > 5 * at_once || IC <= 64 * (wgs <= at_once ? 2 : 2 * wgs <= 3 * at_once ? 5 : 12);
}

hipError_t launch_awq_gemv(const float* x, const int32_t* qw_rep, const uint16_t* wscales, const uint16_t* wzeros,
                           const uint16_t* bias, float* out, int OC, int IC, int gs, int ncomp, hipStream_t stream) {
    if (OC == 0) return hipSuccess;
    // the reference's GEMV reads 8 words (64 inputs) per group
    if (gs != 64 || IC % 64 != 0 || ncomp <= 0 || OC % ncomp != 0 || IC > 16384) return hipErrorInvalidValue;
    if (awq_short(OC, IC)) {
        hipLaunchKernelGGL(awq_gemv_short_kernel, dim3((OC + 63) / 64), dim3(64), IC * sizeof(float), stream, x, qw_rep,
                           wscales, wzeros, bias, out, OC, IC, ncomp);
        return hipGetLastError();
    }
    const int lds = AWQ_RING * 16 + IC * 4;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(awq_gemv_kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(awq_gemv_kernel, dim3((OC + 63) / 64), dim3(AWQ_THR), lds, stream, x, qw_rep, wscales, wzeros,
                       bias, out, OC, IC, ncomp);
    return hipGetLastError();
}

hipError_t launch_nk_unswizzle(const uint8_t* q_sw, const uint16_t* s_sw, uint8_t* q_rm, float* s_rm, int N, int K,
                               int G, hipStream_t stream) {
    if (N == 0 || K == 0) return hipSuccess;
    if (K % 64 != 0 || G <= 0 || K % G != 0 || N % 128 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(nk_unswizzle_kernel, dim3(grid_for(static_cast<int64_t>(N) * (K / 2))), dim3(256), 0, stream,
                       q_sw, s_sw, q_rm, s_rm, N, K, G);
    return hipGetLastError();
}

hipError_t launch_nk_dequant(const uint8_t* q_sw, const uint16_t* s_sw, uint16_t* out, int N, int K, int G,
                             hipStream_t stream) {
    if (N == 0 || K == 0) return hipSuccess;
    if (K % 64 != 0 || G <= 0 || K % G != 0 || N % 128 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(nk_dequant_kernel, dim3(grid_for(static_cast<int64_t>(N) * K)), dim3(256), 0, stream, q_sw,
                       s_sw, out, N, K, G);
    return hipGetLastError();
}

hipError_t launch_lora_unswizzle(const uint16_t* packed, uint16_t* out, int rows, int cols, int is_down,
                                 hipStream_t stream) {
    if (rows == 0 || cols == 0) return hipSuccess;
    if (rows % 16 != 0 || cols % 16 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(lora_unswizzle_kernel, dim3(grid_for(static_cast<int64_t>(rows) * cols)), dim3(256), 0, stream,
                       packed, out, rows, cols, is_down);
    return hipGetLastError();
}

hipError_t launch_transpose_u16(const uint16_t* in, uint16_t* out, int R, int C, hipStream_t stream) {
    if (R == 0 || C == 0) return hipSuccess;
    hipLaunchKernelGGL(transpose_u16_kernel, dim3(grid_for(static_cast<int64_t>(R) * C)), dim3(256), 0, stream, in,
                       out, R, C);
    return hipGetLastError();
}

hipError_t launch_f32_to_bf16(const float* in, uint16_t* out, int64_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(f32_to_bf16_kernel, dim3(grid_for(n)), dim3(256), 0, stream, in, out, n);
    return hipGetLastError();
}

hipError_t launch_bf16_to_f32(const uint16_t* in, float* out, int64_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(bf16_to_f32_kernel, dim3(grid_for(n)), dim3(256), 0, stream, in, out, n);
    return hipGetLastError();
}

}  // namespace qimg
