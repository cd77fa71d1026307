// router.hip -- MoE router of a decoder layer on gfx950: affine-Q8 logits
// and top-8 expert selection.
//
// Reference: QwenQ4ActiveExpertStreamingRunner.swift:1177-1190 dispatches
// qwen_router_q8_logits_simd_f32 (deltanet.metal:2229-2281: one SIMD group
// per expert row, the factored accumulation scale * sum(q x) + bias * sum(x)
// per 64-column group) and qwen_router_top8_logits_f32 (:2283-2329: the eight
// largest logits by insertion, ties keeping the lower expert index, softmax
// over all logits, the eight probabilities renormalised).
//
// Format (MLX affine Q8, group 64, deltanet.metal:863-900): element c of row
// r is byte c of the row, i.e. byte c % 4 (lowest first) of uint32 word
// w[r * cols/4 + c/4]; value = byte * scale[r, c/64] + bias[r, c/64].
//
// Kernels:
//   router_logits_kernel  one token, or a few bf16 ones, on the vector units:
//       one wave per (expert row, block of NT tokens); lane l holds bytes
//       32l .. 32l+31 of each 2048-column piece (two 16-B loads), converts
//       them with v_cvt_f32_ubyte and accumulates in fp32 in the factored
//       form; a lane-group sum per token. x stays fp32. All NT tokens' x
//       loads are issued together and the logits stored at the end (a store
//       between tokens would hold the next token's loads: vmcnt counts
//       stores too).
//   router_logits_mfma_kernel  several tokens, as matrix products on bf16
//       operands: the bytes become the integers q - 128, an fp32 x three
//       terms that add up to it bit for bit, a bf16 x stays as it is, and per
//       group logit += s P + (b + 128 s) sum(x) in fp32. The products are
//       exact and a stored bias of ~-128 times the scale no longer cancels,
//       so the logits are closer to the fp64 product than the vector form's
//       (2000 tokens of fp32 x, 2-norm: 0.92e-7 against 2.5e-7; bf16 x 0.81e-7
//       against 0.91e-7). x as an fp16 hi + lo pair (22 bits) took two thirds
//       of the products and 1.05e-7: 25.6 us at 2000 tokens either way, 54.4
//       against 58.5 at 8192. NW waves split K.
//       What bounded the first form of it, at 25-30 us a block, was the
//       operand order itself: a lane per matrix row makes a 16-byte load
//       touch 64 different lines (38 B/ns per CU from L2 against 125-148
//       where each four lanes read 64 consecutive bytes, measured), so tiles
//       are read in quads and turned through LDS.
//   router_logits_block_kernel  many tokens: the same products, 16 tokens by
//       all experts per workgroup, x converted once, top-8 included.
//   router_top8_kernel    one wave per token: the logits in registers (up to
//       4 per lane), eight rounds of a wave maximum (DPP) and a ballot for
//       the lowest index holding it, then the reference's softmax and
//       renormalisation.
#include "common.hpp"
#include "internal.hpp"
#include "mfma.hpp"

namespace qff {

template <int I>
__device__ __forceinline__ float rt_ubyte(uint32_t v) { return static_cast<float>((v >> (8 * I)) & 0xffu); }

// x[i .. i + 31] as fp32
template <int X_DT>
__device__ __forceinline__ void rt_load_x32(const void* x, size_t i, float (&xv)[32]) {
    if (X_DT == 1) {
        const uint16_t* xp = static_cast<const uint16_t*>(x) + i;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x4_t u = *reinterpret_cast<const u32x4_t*>(xp + 8 * q);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                xv[8 * q + 2 * j] = __uint_as_float(u[j] << 16);
                xv[8 * q + 2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u);
            }
        }
    } else {
        const float4* xp = reinterpret_cast<const float4*>(static_cast<const float*>(x) + i);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 f = xp[q];
            xv[4 * q] = f.x;
            xv[4 * q + 1] = f.y;
            xv[4 * q + 2] = f.z;
            xv[4 * q + 3] = f.w;
        }
    }
}

// acc + scale * sum(q x) + bias * sum(x) of half a group: 32 weight bytes and x
__device__ __forceinline__ float rt_half_group(const u32x4_t (&wq)[2], const float (&xv)[32], float scale, float bias,
                                               float acc) {
    float dot = 0.0f, sum = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t wd = wq[j >> 2][j & 3];
        dot = fmaf(rt_ubyte<0>(wd), xv[4 * j], dot);
        dot = fmaf(rt_ubyte<1>(wd), xv[4 * j + 1], dot);
        dot = fmaf(rt_ubyte<2>(wd), xv[4 * j + 2], dot);
        dot = fmaf(rt_ubyte<3>(wd), xv[4 * j + 3], dot);
        sum += (xv[4 * j] + xv[4 * j + 1]) + (xv[4 * j + 2] + xv[4 * j + 3]);
    }
    acc = fmaf(scale, dot, acc);
    return fmaf(bias, sum, acc);
}

// One logit by one wave, in the operations and order of router_logits_kernel.
template <int SB_DT, int X_DT>
__device__ __forceinline__ float rt_vector_logit(const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                                                 const void* x, int cols, int m, int e, int lane) {
    const int G = cols / 64, npc = cols / 32;
    float acc = 0.0f;
    for (int p0 = 0; p0 < npc; p0 += 64) {
        const int pc = min(p0 + lane, npc - 1);
        const bool live = p0 + lane < npc;
        const u32x4_t* src = reinterpret_cast<const u32x4_t*>(w + static_cast<size_t>(e) * (cols / 4) + 8 * pc);
        const u32x4_t wq[2] = {src[0], src[1]};
        const size_t gi = static_cast<size_t>(e) * G + pc / 2;
        float xv[32];
        rt_load_x32<X_DT>(x, static_cast<size_t>(m) * cols + 32 * pc, xv);
        acc = rt_half_group(wq, xv, live ? elem<SB_DT>::load(scales, gi) : 0.0f,
                            live ? elem<SB_DT>::load(biases, gi) : 0.0f, acc);
    }
    return group_sum<64>(acc);
}

// grid (ceil(E / 4), ceil(batch / NT)), 256 threads; KW = 2048-column pieces
template <int SB_DT, int X_DT, int KW, int NT>
__global__ __launch_bounds__(256) void router_logits_kernel(const uint32_t* __restrict__ w,
                                                            const uint16_t* __restrict__ scales,
                                                            const uint16_t* __restrict__ biases,
                                                            const void* __restrict__ x, float* __restrict__ logits,
                                                            int experts, int cols, int batch) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = blockIdx.x * 4 + wave;
    const int ec = min(e, experts - 1);
    const int m0 = blockIdx.y * NT;
    const int G = cols / 64, W4 = cols / 4, npc = cols / 32;   // 32-byte pieces per row
    u32x4_t wq[KW][2];
    float sv[KW], bv[KW];
    bool live[KW];
#pragma unroll
    for (int k = 0; k < KW; ++k) {
        const int pc = lane + 64 * k;
        live[k] = pc < npc;
        const int pcc = min(pc, npc - 1);
        const uint32_t* src = w + static_cast<size_t>(ec) * W4 + 8 * pcc;
        wq[k][0] = *reinterpret_cast<const u32x4_t*>(src);
        wq[k][1] = *reinterpret_cast<const u32x4_t*>(src + 4);
        sv[k] = elem<SB_DT>::load(scales, static_cast<size_t>(ec) * G + pcc / 2);
        bv[k] = elem<SB_DT>::load(biases, static_cast<size_t>(ec) * G + pcc / 2);
    }
    // every token of the block, its index clamped into the batch, so no load
    // waits behind a branch or a store
    float accs[NT];
#pragma unroll
    for (int mi = 0; mi < NT; ++mi) {
        const int m = min(m0 + mi, batch - 1);
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int pcc = min(lane + 64 * k, npc - 1);
            float xv[32];
            rt_load_x32<X_DT>(x, static_cast<size_t>(m) * cols + 32 * pcc, xv);
            // half a group per lane; pieces past the row end (cols < 2048) add nothing
            acc = rt_half_group(wq[k], xv, live[k] ? sv[k] : 0.0f, live[k] ? bv[k] : 0.0f, acc);
        }
        accs[mi] = group_sum<64>(acc);
    }
    if (lane == 0 && e < experts) {
#pragma unroll
        for (int mi = 0; mi < NT; ++mi)
            if (m0 + mi < batch) logits[static_cast<size_t>(m0 + mi) * experts + e] = accs[mi];
    }
}

// bf16 operands that hold an x of type X_DT
template <int X_DT> constexpr int rt_terms = X_DT == 1 ? 1 : 3;

// 4 weight bytes -> the bf16 pairs q - 128: integers of at most 8 bits, whose
// fp32 form has them in its upper half
__device__ __forceinline__ void rt_bytes_to_bf16(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const uint32_t v = w ^ 0x80808080u;   // q - 128 as signed bytes
    uint32_t f[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        f[c] = __float_as_uint(static_cast<float>(static_cast<int8_t>(static_cast<uint8_t>(v >> (8 * c)))));
    lo = __builtin_amdgcn_perm(f[1], f[0], 0x07060302u);
    hi = __builtin_amdgcn_perm(f[3], f[2], 0x07060302u);
}

// One group (64 columns) of one token, held by the four lanes j of a quad (fp32:
// columns 16 i + 4 j .. +3 in piece i; bf16: 32 i + 8 j .. +7), as bf16
// operands: a bf16 x as it is, an fp32 x as the three terms that cutting 8
// significant bits off at a time leaves, hi + mid + lo == x with every bit (of
// |x| >= 2^-110: below that the last term meets bf16's smallest step, 2^-133).
// Term k goes to xo[k], LDS rows [token][row] at 16-byte pieces p0 + c,
// swizzled by the token. Returns the sum of x.
template <int X_DT, int XL>
__device__ __forceinline__ float rt_stage_x(const u32x4_t (&xr)[XL], uint16_t* const (&xo)[rt_terms<X_DT>], int row,
                                            int tok, int p0, int j) {
    const int sw = tok & (row / 8 - 1) & 15;
    float sum = 0.0f;
    if constexpr (X_DT == 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                sum += __uint_as_float(xr[i][c] << 16);
                sum += __uint_as_float(xr[i][c] & 0xffff0000u);
            }
            *reinterpret_cast<u32x4_t*>(xo[0] + tok * row + 8 * ((p0 + 4 * i + j) ^ sw)) = xr[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t f[3][4];   // fp32 forms of the terms: the upper halves hold them
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float v = __uint_as_float(xr[i][c]);
                sum += v;
                f[0][c] = xr[i][c];
                const float r1 = v - __uint_as_float(f[0][c] & 0xffff0000u);
                f[1][c] = __float_as_uint(r1);
                f[2][c] = __float_as_uint(r1 - __uint_as_float(f[1][c] & 0xffff0000u));
            }
            const int o = tok * row + 8 * ((p0 + 2 * i + (j >> 1)) ^ sw) + 4 * (j & 1);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                *reinterpret_cast<u32x2_t*>(xo[k] + o) = u32x2_t{__builtin_amdgcn_perm(f[k][1], f[k][0], 0x07060302u),
                                                                 __builtin_amdgcn_perm(f[k][3], f[k][2], 0x07060302u)};
        }
    }
    return group_sum<4>(sum);
}

// sum over one group of (q - 128) x for 16 experts (weight bytes wd in operand
// order) x 16 tokens, the smallest terms of x first
template <int TERMS>
__device__ __forceinline__ f32x4_t rt_products(u32x4_t wd, const u32x4_t (&xo)[TERMS][2]) {
    u32x4_t a[2];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        uint32_t lo, hi;
        rt_bytes_to_bf16(wd[d], lo, hi);
        a[d >> 1][2 * (d & 1)] = lo;
        a[d >> 1][2 * (d & 1) + 1] = hi;
    }
    f32x4_t P = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = TERMS - 1; k >= 0; --k) {
        P = mfma_16x16x32_bf16(a[0], xo[k][0], P);
        P = mfma_16x16x32_bf16(a[1], xo[k][1], P);
    }
    return P;
}

// Logits that the products leave infinite or NaN, from the vector form: an
// infinite x has no terms (inf - inf), and (q - 128) x can pass fp32's range
// where q x does not. Lane l holds logit v of (token m, expert e), if ok.
template <int SB_DT, int X_DT>
__device__ __forceinline__ float rt_finite_or_vector(float v, bool ok, int m, int e, const uint32_t* w,
                                                     const uint16_t* scales, const uint16_t* biases, const void* x,
                                                     int cols, int lane) {
    for (uint64_t bad = __ballot(ok && !(fabsf(v) <= 3.4028235e38f)); bad != 0; bad &= bad - 1) {   // wave-uniform
        const int src = __builtin_ctzll(bad);
        const float r = rt_vector_logit<SB_DT, X_DT>(w, scales, biases, x, cols, __builtin_amdgcn_readlane(m, src),
                                                     __builtin_amdgcn_readlane(e, src), lane);
        if (lane == src) v = r;
    }
    return v;
}

// acc += s P + (b + 128 s) sum(x) for the lane's four experts, sb their (s, b + 128 s)
__device__ __forceinline__ void rt_accumulate(f32x4_t& acc, f32x4_t P, float sum, const f32x4_t* sb) {
    const f32x4_t c0 = sb[0], c1 = sb[1];
    acc[0] = fmaf(c0[0], P[0], fmaf(c0[1], sum, acc[0]));
    acc[1] = fmaf(c0[2], P[1], fmaf(c0[3], sum, acc[1]));
    acc[2] = fmaf(c1[0], P[2], fmaf(c1[1], sum, acc[2]));
    acc[3] = fmaf(c1[2], P[3], fmaf(c1[3], sum, acc[3]));
}

// A 16-row x 64-byte tile from the load's lane order (lane l: row l / 4, piece
// l % 4, so four lanes read 64 consecutive bytes) into the MFMA operand's (lane
// l: row l % 16, piece l / 16) through 1 KB of the wave's own LDS, the pieces
// of a row rotated so that 16 lanes meet every bank group.
__device__ __forceinline__ u32x4_t rt_tile_turn(uint32_t* buf, u32x4_t v, int lane) {
    const int r = lane >> 2, n = lane & 15;
    *reinterpret_cast<u32x4_t*>(buf + 4 * (4 * r + ((lane & 3) ^ (r >> 2)))) = v;
    __builtin_amdgcn_wave_barrier();
    const u32x4_t o = *reinterpret_cast<const u32x4_t*>(buf + 4 * (4 * n + ((lane >> 4) ^ (n >> 2))));
    __builtin_amdgcn_wave_barrier();
    return o;
}

// Several tokens. grid (ceil(E / (16 NT)), ceil(batch / 16)), NW waves.
template <int SB_DT, int X_DT, int NT, int NW>
__global__ __launch_bounds__(64 * NW) void router_logits_mfma_kernel(const uint32_t* __restrict__ w,
                                                                     const uint16_t* __restrict__ scales,
                                                                     const uint16_t* __restrict__ biases,
                                                                     const void* __restrict__ x,
                                                                     float* __restrict__ logits, int experts, int cols,
                                                                     int batch, int gmagic) {
    constexpr int TERMS = rt_terms<X_DT>, XB = X_DT == 1 ? 2 : 4;   // operands and bytes of an x
    constexpr int RE = 16 * NT;   // experts per workgroup
    constexpr int XL = XB;        // 16-byte x loads per lane and group
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int n = lane & 15, kb = lane >> 4;
    const int G = cols / 64;
    const int E0 = static_cast<int>(blockIdx.x) * RE, M0 = static_cast<int>(blockIdx.y) * 16;
    // (s, b + 128 s) of the workgroup's experts, [G][RE]; afterwards the waves' partial logits [NW][RE x 16]
    constexpr int kSb = 64 * (RE + 2) * 2, kPart = NW * RE * 16;
    __shared__ __attribute__((aligned(16))) float lds[kSb > kPart ? kSb : kPart];
    // per wave: a weight tile, the group's x operands [16 tokens][64] and each token's sum
    __shared__ __attribute__((aligned(16))) uint32_t wl[NW][256];
    __shared__ __attribute__((aligned(16))) uint16_t xl[NW][TERMS][16 * 64];
    __shared__ float xf[NW][16];

    const char* xrow = static_cast<const char*>(x) +
                       static_cast<size_t>(min(M0 + (lane >> 2), batch - 1)) * cols * XB + 16 * (lane & 3);
    const uint32_t* wrow[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
        wrow[i] = w + static_cast<size_t>(min(E0 + 16 * i + (lane >> 2), experts - 1)) * (cols / 4) + 4 * (lane & 3);

    u32x4_t xr[2][XL], wr[2][NT];
    auto fetch = [&](int s, int g) {
        const char* xp = xrow + 64 * g * XB;
#pragma unroll
        for (int q = 0; q < XL; ++q) xr[s][q] = *reinterpret_cast<const u32x4_t*>(xp + 64 * q);
#pragma unroll
        for (int i = 0; i < NT; ++i) wr[s][i] = *reinterpret_cast<const u32x4_t*>(wrow[i] + 16 * g);
    };
    // the wave's first two groups and the scales, all requested before any is
    // used (indices clamped, so every load is issued)
    fetch(0, min(wave, G - 1));
    fetch(1, min(wave + NW, G - 1));
    constexpr int SBT = RE / NW;   // entries per thread at the largest G, 64
    float sv[SBT], bv[SBT];
#pragma unroll
    for (int k = 0; k < SBT; ++k) {
        const int idx = min(t + 64 * NW * k, RE * G - 1), e = (idx * gmagic) >> 20;
        const size_t gi = static_cast<size_t>(min(E0 + e, experts - 1)) * G + (idx - e * G);
        sv[k] = elem<SB_DT>::load(scales, gi);
        bv[k] = elem<SB_DT>::load(biases, gi);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < SBT; ++k) {
        const int idx = min(t + 64 * NW * k, RE * G - 1), e = (idx * gmagic) >> 20, g = idx - e * G;
        *reinterpret_cast<float2*>(&lds[(g * (RE + 2) + e) * 2]) = make_float2(sv[k], fmaf(128.0f, sv[k], bv[k]));
    }
    __syncthreads();

    f32x4_t acc[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int s, int g) {
        uint16_t* xo[TERMS];
#pragma unroll
        for (int k = 0; k < TERMS; ++k) xo[k] = xl[wave][k];
        const float xs = rt_stage_x<X_DT>(xr[s], xo, 64, lane >> 2, 0, lane & 3);
        if ((lane & 3) == 0) xf[wave][lane >> 2] = xs;
        __builtin_amdgcn_wave_barrier();
        const float sum = xf[wave][n];
        u32x4_t xv[TERMS][2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int o = n * 64 + 8 * ((2 * kb + ks) ^ (n & 7));
#pragma unroll
            for (int k = 0; k < TERMS; ++k) xv[k][ks] = *reinterpret_cast<const u32x4_t*>(&xl[wave][k][o]);
        }
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const f32x4_t P = rt_products<TERMS>(rt_tile_turn(wl[wave], wr[s][i], lane), xv);
            // experts 16 i + 4 kb .. +3
            rt_accumulate(acc[i], P, sum, reinterpret_cast<const f32x4_t*>(&lds[(g * (RE + 2) + 16 * i + 4 * kb) * 2]));
        }
        __builtin_amdgcn_wave_barrier();
    };
    for (int g = wave; g < G; g += 2 * NW) {   // wave-uniform
        step(0, g);
        if (g + 2 * NW < G) fetch(0, g + 2 * NW);
        if (g + NW < G) step(1, g + NW);
        if (g + 3 * NW < G) fetch(1, g + 3 * NW);
    }
    __syncthreads();   // the scales are consumed; their bytes take the partial sums
#pragma unroll
    for (int i = 0; i < NT; ++i) *reinterpret_cast<f32x4_t*>(&lds[wave * RE * 16 + (i * 64 + lane) * 4]) = acc[i];
    __syncthreads();
    for (int o = t; o < RE * 16; o += 64 * NW) {   // wave-uniform
        float v = lds[o];
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) v += lds[ww * RE * 16 + o];
        const int l = (o >> 2) & 63, e = E0 + 16 * (o >> 8) + 4 * (l >> 4) + (o & 3), m = M0 + (l & 15);
        const bool ok = m < batch && e < experts;
        v = rt_finite_or_vector<SB_DT, X_DT>(v, ok, m, e, w, scales, biases, x, cols, lane);
        if (ok) logits[static_cast<size_t>(m) * experts + e] = v;
    }
}

// One wave ranks token m's logits lg[0 .. experts): the eight largest (ties to
// the lower index) and their renormalised softmax weights.
__device__ __forceinline__ void router_top8(const float* lg, int32_t* __restrict__ indices,
                                            float* __restrict__ scores, int m, int experts, int lane) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = lane + 64 * j;
        v[j] = i < experts ? lg[i] : -INFINITY;
    }
    bool taken[4] = {false, false, false, false};
    float top_v[8];
    int top_i[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        // the largest untaken logit, then its lowest index: the index blocks
        // j hold experts 64j .. 64j+63 in lane order, so the first block
        // whose ballot hits gives the lowest index through its lowest lane
        float lm = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j < experts && !taken[j]) lm = fmaxf(lm, v[j]);
        const float wm = group_max<64>(lm);
        int idx = -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const unsigned long long hit = __ballot(lane + 64 * j < experts && !taken[j] && v[j] == wm);
            if (idx < 0 && hit) idx = 64 * j + __ffsll(static_cast<long long>(hit)) - 1;
        }
        top_v[k] = wm;
        top_i[k] = idx;
#pragma unroll
        for (int j = 0; j < 4; ++j) taken[j] = taken[j] || idx == lane + 64 * j;
    }
    // softmax over all logits with the top value as the shift, eight
    // probabilities renormalised
    const float mx = top_v[0];
    float den = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (lane + 64 * j < experts) den += expf(v[j] - mx);
    den = group_sum<64>(den);
    float p[8], tot = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        p[k] = expf(top_v[k] - mx) / den;
        tot += p[k];
    }
    if (lane < 8) {
        float pk = p[0];
        int ik = top_i[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) {
            pk = lane == k ? p[k] : pk;
            ik = lane == k ? top_i[k] : ik;
        }
        indices[static_cast<size_t>(m) * 8 + lane] = ik;
        scores[static_cast<size_t>(m) * 8 + lane] = pk / tot;
    }
}


// grid ceil(batch / 4), 256 threads: wave w ranks token 4 blockIdx.x + w.
__global__ __launch_bounds__(256) void router_top8_kernel(const float* __restrict__ logits,
                                                          int32_t* __restrict__ indices, float* __restrict__ scores,
                                                          int experts, int batch) {
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= batch) return;   // wave-uniform
    router_top8(logits + static_cast<size_t>(m) * experts, indices, scores, m, experts, threadIdx.x & 63);
}

// Enough tokens for every CU: a workgroup takes 16 tokens and all experts (wave
// w experts 16 w .. 16 w + 15, one MFMA tile over all of K) and ranks its
// tokens itself, one per wave. Each slab of 512 columns of x is converted
// once per workgroup (thread quads, rt_stage_x) into LDS; the weights are
// requested four groups ahead into registers (a slab ahead ten registers
// spill: 21 MB of scratch writes, 64 against 58.5 us at 8192 tokens). LDS is
// active half of the time at 8192 tokens, a fifth of that on bank conflicts, and
// the matrix cores 16 %: every wave reads the slab's x (3 MB a block in all, 1
// MB of bf16) and turns its weights there. Eight waves with two tiles each: 3-8
// % slower than these sixteen, 10 % with bf16 x.
constexpr int kRtSlab = 8;          // groups per slab
constexpr int kRtAhead = 4;         // groups between a weight tile's request and its use
constexpr int kRtBlockWaves = 16;   // a token and a tile of 16 experts each

template <int SB_DT, int X_DT>
__global__ __launch_bounds__(64 * kRtBlockWaves) void router_logits_block_kernel(
    const uint32_t* __restrict__ w, const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
    const void* __restrict__ x, float* __restrict__ logits, int32_t* __restrict__ indices,
    float* __restrict__ scores, int experts, int cols, int batch) {
    constexpr int TERMS = rt_terms<X_DT>, XB = X_DT == 1 ? 2 : 4;                   // operands and bytes of an x
    constexpr int NW = kRtBlockWaves, RE = 16 * NW, XL = XB;
    constexpr int SBT = RE * kRtSlab / (64 * NW);                                   // scale entries per thread and slab
    constexpr int XS = 16 * 512;                                                    // values of a slab
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int n = lane & 15, kb = lane >> 4;
    const int G = cols / 64, NS = (G + kRtSlab - 1) / kRtSlab;
    const int M0 = static_cast<int>(blockIdx.x) * 16;

    __shared__ __attribute__((aligned(16))) uint16_t xs[2][TERMS][XS];
    __shared__ __attribute__((aligned(16))) float sbl[2][kRtSlab * (RE + 2) * 2];
    __shared__ __attribute__((aligned(16))) uint32_t wl[NW][256];   // per wave: a tile's 16 rows x 64 bytes
    __shared__ float xf[2][kRtSlab][16];   // sum of (group, token)

    // this thread's x quads and scale entries of a slab, and this wave's
    // weights of it: lane l the 16 bytes l % 4 of row l / 4 of each group
    u32x4_t xr[XL], wr[kRtAhead];
    float sv[SBT], bv[SBT];
    // the first eight waves' threads hold a slab's 128 (token, group) quads
    const bool stager = __builtin_amdgcn_readfirstlane(wave) < 8;   // wave-uniform
    const uint32_t* const wrow = w + static_cast<size_t>(min(16 * wave + (lane >> 2), experts - 1)) * (cols / 4) + 4 * (lane & 3);
    auto fetch_x = [&](int sl) {
        if (!stager) return;
        const int q = t >> 2, tok = q >> 3, g = min(kRtSlab * sl + (q & 7), G - 1);
        const char* src = static_cast<const char*>(x) +
                          (static_cast<size_t>(min(M0 + tok, batch - 1)) * cols + 64 * g) * XB + 16 * (t & 3);
#pragma unroll
        for (int i = 0; i < XL; ++i) xr[i] = *reinterpret_cast<const u32x4_t*>(src + 64 * i);
    };
    auto fetch_sb = [&](int sl) {
#pragma unroll
        for (int k = 0; k < SBT; ++k) {
            const int idx = t + 64 * NW * k, e = idx >> 3, g = kRtSlab * sl + (idx & 7);
            const size_t gi = static_cast<size_t>(min(e, experts - 1)) * G + min(g, G - 1);
            sv[k] = elem<SB_DT>::load(scales, gi);
            bv[k] = elem<SB_DT>::load(biases, gi);
        }
    };
    auto fetch_w = [&](int g) { wr[g & (kRtAhead - 1)] = *reinterpret_cast<const u32x4_t*>(wrow + 16 * min(g, G - 1)); };
    // the fetched slab into LDS buffer buf (groups past the last get zero scales)
    auto stage = [&](int sl, int buf) {
#pragma unroll
        for (int k = 0; k < SBT; ++k) {
            const int idx = t + 64 * NW * k, e = idx >> 3, gl = idx & 7;
            const bool live = kRtSlab * sl + gl < G;
            *reinterpret_cast<float2*>(&sbl[buf][(gl * (RE + 2) + e) * 2]) =
                make_float2(live ? sv[k] : 0.0f, live ? fmaf(128.0f, sv[k], bv[k]) : 0.0f);
        }
        if (stager) {
            const int q = t >> 2, tok = q >> 3, gl = q & 7, j = t & 3;
            uint16_t* xo[TERMS];
#pragma unroll
            for (int k = 0; k < TERMS; ++k) xo[k] = xs[buf][k];
            const float sum = rt_stage_x<X_DT>(xr, xo, 512, tok, 8 * gl, j);
            if (j == 0) xf[buf][gl][tok] = sum;
        }
    };

    fetch_x(0);
    fetch_sb(0);
#pragma unroll
    for (int g = 0; g < kRtAhead; ++g) fetch_w(g);
    // (a clobber after each slab's requests: otherwise the compiler moves the
    // loads to the top of the iteration that uses them)
    asm volatile("" ::: "memory");
    f32x4_t tot = f32x4_t{0.f, 0.f, 0.f, 0.f};   // lane: token n, experts 16 wave + 4 kb .. +3
    for (int sl = 0; sl < NS; ++sl) {
        const int buf = sl & 1;
        f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};   // the slab's own sums: shorter fp32 chains
        stage(sl, buf);
        __syncthreads();
        // the next slab (the last again at the end: no branch around loads)
        const int nx = min(sl + 1, NS - 1);
        fetch_x(nx);
        fetch_sb(nx);
#pragma unroll
        for (int gl = 0; gl < kRtSlab; ++gl) {
            const float sum = xf[buf][gl][n];
            u32x4_t xv[TERMS][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {   // columns 16 kb + 8 ks .. +7 of the group
                const int o = n * 512 + 8 * ((8 * gl + 2 * kb + ks) ^ n);
#pragma unroll
                for (int k = 0; k < TERMS; ++k) xv[k][ks] = *reinterpret_cast<const u32x4_t*>(&xs[buf][k][o]);
            }
            const f32x4_t P = rt_products<TERMS>(rt_tile_turn(wl[wave], wr[gl % kRtAhead], lane), xv);
            rt_accumulate(acc, P, sum, reinterpret_cast<const f32x4_t*>(&sbl[buf][(gl * (RE + 2) + 16 * wave + 4 * kb) * 2]));
            fetch_w(kRtSlab * sl + gl + kRtAhead);
        }
        tot += acc;
        asm volatile("" ::: "memory");
    }
    // every expert of the 16 tokens is here: logits through LDS (the staging
    // buffers are idle once every wave is past its last slab)
    __syncthreads();
    float* lg = reinterpret_cast<float*>(xs);   // [16][RE + 4]
    *reinterpret_cast<f32x4_t*>(&lg[n * (RE + 4) + 16 * wave + 4 * kb]) = tot;
    __syncthreads();
    const int m = M0 + wave;
    if (m >= batch) return;   // wave-uniform
    lg += wave * (RE + 4);
    for (int e0 = 0; e0 < experts; e0 += 64) {
        const int e = e0 + lane;
        const bool ok = e < experts;
        const float v = rt_finite_or_vector<SB_DT, X_DT>(lg[e], ok, m, e, w, scales, biases, x, cols, lane);
        if (ok) logits[static_cast<size_t>(m) * experts + e] = lg[e] = v;
    }
    __builtin_amdgcn_wave_barrier();
    router_top8(lg, indices, scores, m, experts, lane);
}

// Q8 dequant test hook: one word (4 bytes) per thread -> 4 floats.
template <int SB_DT>
__global__ __launch_bounds__(256) void q8_dequant_kernel(const uint32_t* __restrict__ w,
                                                         const uint16_t* __restrict__ scales,
                                                         const uint16_t* __restrict__ biases,
                                                         float* __restrict__ out, int rows, int cols) {
    const size_t words = static_cast<size_t>(rows) * (cols / 4);
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= words) return;
    const int r = static_cast<int>(i / (cols / 4));
    const int c0 = static_cast<int>(i % (cols / 4)) * 4;
    const size_t gi = static_cast<size_t>(r) * (cols / 64) + c0 / 64;
    const float s = elem<SB_DT>::load(scales, gi);
    const float b = elem<SB_DT>::load(biases, gi);
    const uint32_t word = w[i];
    reinterpret_cast<float4*>(out + static_cast<size_t>(r) * cols + c0)[0] =
        make_float4(rt_ubyte<0>(word) * s + b, rt_ubyte<1>(word) * s + b, rt_ubyte<2>(word) * s + b,
                    rt_ubyte<3>(word) * s + b);
}

hipError_t launch_q8_dequant(hipStream_t stream, const uint32_t* w, const void* scales, const void* biases,
                             qff_dtype sb_dtype, float* out, int rows, int cols) {
    const size_t words = static_cast<size_t>(rows) * (cols / 4);
    const unsigned blocks = static_cast<unsigned>((words + 255) / 256);
    const uint16_t* s = static_cast<const uint16_t*>(scales);
    const uint16_t* b = static_cast<const uint16_t*>(biases);
    if (sb_dtype == QFF_BF16) q8_dequant_kernel<1><<<blocks, 256, 0, stream>>>(w, s, b, out, rows, cols);
    else q8_dequant_kernel<2><<<blocks, 256, 0, stream>>>(w, s, b, out, rows, cols);
    return hipGetLastError();
}

hipError_t launch_router_top8(qff_ctx* ctx, hipStream_t stream, const uint32_t* w, const void* scales,
                              const void* biases, qff_dtype sb_dtype, const void* x, qff_dtype x_dtype,
                              float* logits, int32_t* indices, float* scores, int experts, int cols, int batch) {
    const uint16_t* s = static_cast<const uint16_t*>(scales);
    const uint16_t* b = static_cast<const uint16_t*>(biases);
    // The kernel by the number of 16-token blocks nb (batch 8192 / 4096 / 2560 /
    // 2000 / 512 / 256 / 16 at 256 x 2048, both launches, us; fp32 x, then bf16):
    //   vector units   1835 / 923 / 580 / 454 / 123 / 64.5 / 10.9    504 / 258 / 164 / 130 / 39.8 / 24.3 / 8.9
    //   MFMA, 1 tile    161 / 85.3 / 57.0 / 46.4 / 17.1 / 11.8 / 11.0  103 / 55.5 / 37.9 / 31.3 / 12.8 / 10.2 / 9.5
    //   MFMA, 2 tiles   120 / 67.1 / 46.6 / 37.9 / 14.2 / 12.9 / 12.4   65 / 36.6 / 26.4 / 22.5 / 11.4 / 11.1 / 10.7
    //   MFMA, 4 tiles    82 / 43.9 / 35.1 / 25.2 / 17.3 / 17.3 / 17.0   58 / 33.8 / 25.6 / 20.4 / 15.4 / 15.4 / 14.8
    //   whole blocks   58.5 / 31.1 / 28.9 / 30.3 / 29.1 / 28.9 / 27.7   45 / 24.2 / 23.0 / 22.8 / 23.1 / 23.0 / 21.8
    // so the tiles per workgroup grow once the grid covers the chip, and whole
    // blocks take over where they do so themselves.
    const int nb = (batch + 15) / 16, cu = ctx->num_cu;
    const bool k2 = cols > 2048, vec = batch == 1 || (x_dtype == QFF_BF16 && batch <= 16);
    if (8 * nb > 5 * cu) {
        ProfScope prof(ctx, stream, "router_logits");
#define QFF_RB(S, X) \
    router_logits_block_kernel<S, X><<<nb, 64 * kRtBlockWaves, 0, stream>>>(w, s, b, x, logits, indices, scores, experts, \
                                                                           cols, batch)
        if (sb_dtype == QFF_BF16) {
            if (x_dtype == QFF_BF16) QFF_RB(1, 1); else QFF_RB(1, 0);
        } else {
            if (x_dtype == QFF_BF16) QFF_RB(2, 1); else QFF_RB(2, 0);
        }
#undef QFF_RB
        return hipGetLastError();
    }
    {
        ProfScope prof(ctx, stream, "router_logits");
        const dim3 vgrid((experts + 3) / 4, (batch + 3) / 4);
        const int gmagic = (1 << 20) / (cols / 64) + 1;   // idx / G = idx gmagic >> 20 for idx < 4096, G <= 64
        const auto tiles = [&](int nt) { return (experts + 16 * nt - 1) / (16 * nt); };
#define QFF_RV(S, X, K, NT) \
    router_logits_kernel<S, X, K, NT><<<vgrid, 256, 0, stream>>>(w, s, b, x, logits, experts, cols, batch)
#define QFF_RM(S, X, NT, NW)                                                                              \
    router_logits_mfma_kernel<S, X, NT, NW><<<dim3(tiles(NT), nb), 64 * NW, 0, stream>>>(w, s, b, x, logits, \
                                                                                        experts, cols, batch, gmagic)
#define QFF_RL(S, X)                                            \
    if (vec) {                                                  \
        if (batch == 1) {                                       \
            if (k2) QFF_RV(S, X, 2, 1); else QFF_RV(S, X, 1, 1); \
        } else { /* bf16 x */                                   \
            if (k2) QFF_RV(S, 1, 2, 4); else QFF_RV(S, 1, 1, 4); \
        }                                                       \
    } else if (tiles(1) * nb <= cu) {                           \
        QFF_RM(S, X, 1, 16);                                    \
    } else if (tiles(2) * nb <= cu) {                           \
        QFF_RM(S, X, 2, 8);                                     \
    } else {                                                    \
        QFF_RM(S, X, 4, 4);                                     \
    }
#define QFF_RL_X(S) \
    if (x_dtype == QFF_BF16) { QFF_RL(S, 1); } else { QFF_RL(S, 0); }
        if (sb_dtype == QFF_BF16) { QFF_RL_X(1); } else { QFF_RL_X(2); }
#undef QFF_RL_X
#undef QFF_RL
#undef QFF_RM
#undef QFF_RV
    }
    ProfScope prof(ctx, stream, "router_top8");
    router_top8_kernel<<<(batch + 3) / 4, 256, 0, stream>>>(logits, indices, scores, experts, batch);
    return hipGetLastError();
}

}  // namespace qff
