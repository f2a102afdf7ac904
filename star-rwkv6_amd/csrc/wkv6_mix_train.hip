// The whole input side of the time-mix layer with gradients (rwkv6_model.py:134-146; notation of wkv6_mix.hip):
//
//   h      = tanh(x_mix A^T)                         x_mix = x + xx mix_x, A the five stacked (R, C) first weights
//   x_s    = x + xx (h_s W_s^T + bias_s)             (shift_mix_five of wkv6_mix.hip)
// backward, from the gradients g_s of the five outputs, gcoef_s = g_s xx:
//   gh_s   = gcoef_s W_s                             summed over channels
//   gpre   = gh (1 - h^2),  gxm = gpre A             gradients of x_mix A^T and of x_mix
//   gW_s   = gcoef_s^T h_s,  gbias_s = sum gcoef_s,  gA = gpre^T x_mix,  gmix = sum gxm xx      summed over tokens
//   gx[t]  = sum_s g_s - gxx + gxm (1 - mix_x) + z[t+1],   gxx = sum_s g_s coef_s,  z = gxx + gxm mix_x
//
// All of it is bound by the traffic of the (B,T,C) tensors, so none of the products that appear between them is ever
// written: x_mix, the five coefficients and the five gcoef live in registers (and, where a product sums over tokens, in
// a wave's own LDS tile).  A sum over channels and a sum over tokens of the same gcoef cannot both be finished by one
// workgroup, so the gradients g_s are read twice: mix_reduce_kernel<grad> takes whole rows of a few tokens (gpre
// complete, nothing to combine between workgroups), mix_grads_kernel takes 64 channels of many tokens (the weight
// gradients stay in accumulators, one partial per workgroup).
// B8 T1024 C2048, forward and backward: 178 us of kernels at R32 (x and the gradients read twice more than once: 501 MB in, 232 MB
// out), 381 us at R64; R32 as four elementwise kernels around six library products (gcoef written and read twice, x_mix
// written and read) 504 us, of which 235 us the skinny products.
#include "wkv6_common.h"
#include "wkv6_kernels.h"
#include "wkv6_mfma.h"

#include <type_traits>

namespace wkv6 {

constexpr int kMix = 5;          // mixers
constexpr int kFragElems = 512;  // one operand fragment of a 16x16x32 MFMA: 64 lanes x 8 elements

typedef Raw8<bf16_t> Row8;
// eight elements at a uniform base and a 32-bit byte offset per lane (the scalar-base addressing form)
__device__ __forceinline__ void load_row8(Row8 &r, const bf16_t *base, uint32_t byteoff) {
    r.a = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(base) + byteoff);
}

// a value that is the same in every lane, pinned to scalar registers (the compiler keeps some in vector registers)
__device__ __forceinline__ int64_t uniform64(int64_t x) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)x >> 32));
    return (int64_t)((uint64_t)hi << 32 | lo);
}
// ---- DPP moves inside a row of 16 lanes (lane l16 = token): the previous / the next token's value -----------------
__device__ __forceinline__ uint32_t prev_lane(uint32_t first, uint32_t x) {   // lane 0 keeps `first`
    return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)x, 0x111, 0xF, 0xF, false);   // row_shr:1
}
__device__ __forceinline__ float next_lane(float last, float x) {             // lane 15 keeps `last`
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(last), __float_as_int(x), 0x101, 0xF, 0xF, false));   // row_shl:1
}
__device__ __forceinline__ uint32_t last_to_first(uint32_t x) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x121, 0xF, 0xF, false); }   // row_ror:1
__device__ __forceinline__ float first_to_last(float x) {                                                                                     // row_ror:15
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x12F, 0xF, 0xF, false));
}
__device__ __forceinline__ Row8 prev_rows(const Row8 &first, const Row8 &x) {
    Row8 p;
    p.a.x = prev_lane(first.a.x, x.a.x); p.a.y = prev_lane(first.a.y, x.a.y);
    p.a.z = prev_lane(first.a.z, x.a.z); p.a.w = prev_lane(first.a.w, x.a.w);
    return p;
}
__device__ __forceinline__ Row8 last_row_first(const Row8 &x) {
    Row8 p;
    p.a.x = last_to_first(x.a.x); p.a.y = last_to_first(x.a.y); p.a.z = last_to_first(x.a.z); p.a.w = last_to_first(x.a.w);
    return p;
}
// the values are final here: nothing of their computation moves past this point
__device__ __forceinline__ void pin8(float (&v)[8]) {
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
}
__device__ __forceinline__ bf16x8 pack_operand(const float (&v)[8]) {
    return make_bf16x8(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
}

// ------------------------------------------------------------------------------------------
// The weights in the forms the kernels read, once per call: two MB of traffic, bound by its launch.
//   a_frag  [C/32][5R/16][64 lanes][8]      A as operand fragments with the k-slots along 32 channels
//   wt_frag [C/32][5][R/16][64 lanes][8]    W_s transposed, the same
//   a_t     (C, 5R)                         A transposed
//   w       (5, C, R)                       W in bf16
// One workgroup per 32 channels and matrix (blockIdx.y).
// ------------------------------------------------------------------------------------------
template <typename Tw, int R>
__global__ __launch_bounds__(256) void mix_weights_kernel(int C, const Tw *__restrict__ a, const Tw *__restrict__ w2t,
        bf16_t *__restrict__ a_frag, bf16_t *__restrict__ wt_frag, bf16_t *__restrict__ a_t, bf16_t *__restrict__ w)
{
    constexpr int rows = kMix * R;
    __shared__ bf16_t tile[rows][40];   // [stacked row (s, r)][channel of the 32]
    const int c0 = (int)blockIdx.x * 32;
    const bool is_a = blockIdx.y == 0;
    if (is_a) {
#pragma unroll
        for (int j = 0; j < rows * 8 / 256; ++j) {
            const int i = j * 256 + threadIdx.x;
            float v[4];
            load4(a + (size_t)(i >> 3) * C + c0 + 4 * (i & 7), v);
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[i >> 3][4 * (i & 7) + e] = (bf16_t)v[e];
        }
    } else {
        constexpr int per = R / 4;   // 4-element pieces of a row of W
#pragma unroll
        for (int j = 0; j < kMix * 32 * per / 256; ++j) {
            const int i = j * 256 + threadIdx.x;
            const int r = (i % per) * 4, c = (i / per) % 32, s = i / (per * 32);
            float v[4];
            load4(w2t + ((size_t)s * C + c0 + c) * R + r, v);
            store4(w + ((size_t)s * C + c0 + c) * R + r, v[0], v[1], v[2], v[3]);
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[s * R + r + e][c] = (bf16_t)v[e];
        }
    }
    __syncthreads();
    bf16_t *frag = (is_a ? a_frag : wt_frag) + (size_t)blockIdx.x * rows * 32;
    for (int i = threadIdx.x; i < rows * 4; i += 256) {   // fragment i / 64, lane i % 64
        const int l = i & 63;
        *reinterpret_cast<uint4 *>(frag + (size_t)i * 8) = *reinterpret_cast<const uint4 *>(&tile[(i >> 6) * 16 + (l & 15)][8 * (l >> 4)]);
    }
    if (is_a)
        for (int i = threadIdx.x; i < 32 * (rows / 8); i += 256) {
            const int c = i / (rows / 8), r = (i % (rows / 8)) * 8;
            uint16_t v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(uint16_t, tile[r + e][c]);
            *reinterpret_cast<uint4 *>(a_t + (size_t)(c0 + c) * rows + r) =
                make_uint4(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16, v[4] | (uint32_t)v[5] << 16, v[6] | (uint32_t)v[7] << 16);
        }
}

// tanh to well under half a unit of bf16 (2^-9): 1 - 2 / (e^{2x} + 1), and where that difference cancels the series
// x (1 - x^2/3 + 2 x^4/15), whose next term is 17 x^6/315 < 3e-5 below |x| = 1/4.
__device__ __forceinline__ float tanh_bf16(float x) {
    const float x2 = x * x;
    const float small = x * fmaf(x2, fmaf(x2, 2.f / 15.f, -1.f / 3.f), 1.f);
    const float big = 1.f - 2.f * __builtin_amdgcn_rcpf(exp2_fast(x * (2.f * kLog2e)) + 1.f);
    return x2 < 0.0625f ? small : big;
}

// ------------------------------------------------------------------------------------------
// Sums over channels:  forward  h = tanh(x_mix A^T);  kGrad  gpre = (gcoef_s W_s)_s (1 - h^2).
// One workgroup takes all channels of 32 tokens (16 at R = 64: the accumulators), so nothing is left to combine; its
// eight waves take 32-channel chunks in turn and add up through LDS at the end.  The weights' fragments come from L2 once
// per workgroup (16 tokens per workgroup, i.e. twice that traffic: 30 and 73 us instead of 21 and 50).  A chunk's x and
// g are fetched while the chunk before it is worked on.  B8 T1024 C2048 in a pass, R32: 17 us forward, latencies of a launch of one
// workgroup per compute unit (12 us with nothing fetched in the loop); 41 us backward for 204 MB read, part of it still in the
// last-level cache.  R64: 39 and 58 us.
// ------------------------------------------------------------------------------------------
constexpr int kReduceWaves = 8;
template <int R> struct MixReduce {
    static constexpr int kBlocks = R == 32 ? 2 : 1;          // 16-token blocks per workgroup
    static constexpr int kTiles = kMix * R / 16;             // 16-row tiles of the stacked rank
    static constexpr int kRound = kTiles * kBlocks / 2;      // accumulator tiles combined per round
    static constexpr int kLds = kReduceWaves * kRound * 64 * 16;
};

template <int R, bool kGrad>
__global__ __launch_bounds__(kReduceWaves * 64) void mix_reduce_kernel(int64_t n_tok, int T, int C,
        const bf16_t *__restrict__ x, const float *__restrict__ mix_x, const bf16_t *__restrict__ frags,
        const bf16_t *__restrict__ g0, const bf16_t *__restrict__ g1, const bf16_t *__restrict__ g2, const bf16_t *__restrict__ g3,
        const bf16_t *__restrict__ g4, const bf16_t *__restrict__ h, bf16_t *__restrict__ out)
{
    typedef MixReduce<R> M;
    constexpr int NB = M::kBlocks, NT = M::kTiles, RT = R / 16;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t tok0 = (int64_t)blockIdx.x * (16 * NB);
    const bf16_t *const gs[kMix] = {g0, g1, g2, g3, g4};
    const int64_t base = tok0 * C;
    const int left = (int)(n_tok - 1 - tok0 < 16 * NB ? n_tok - 1 - tok0 : 16 * NB);   // (rows past the end: the last one once more, not stored)
    uint32_t row[NB];
    bool first[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int t = min(16 * b + l16, left);
        row[b] = ((uint32_t)t * (uint32_t)C + 8 * g) * 2u;
        first[b] = (tok0 + t) % T == 0;
    }
    const bool before = l16 == 0 && tok0 % T != 0;
    // one chunk's operands; each is fetched anew for the wave's next chunk as soon as the current one is done with it
    Row8 xr[NB], xp, gr[kGrad ? kMix : 1][NB];
    Raw8<float> mix;
    bf16x8 wf[NT];
    auto fetch_x = [&](int c) {
#pragma unroll
        for (int b = 0; b < NB; ++b) load_row8(xr[b], x + base + c, row[b]);
        if (before) load_row8(xp, x + base - C + c, row[0]);
        if (!kGrad) mix.load(mix_x + c + 8 * g);
    };
    auto fetch_g = [&](int s, int c) {
#pragma unroll
        for (int b = 0; b < NB; ++b) load_row8(gr[kGrad ? s : 0][b], gs[s] + base + c, row[b]);
    };
    auto fetch_w = [&](int i, int c) {
        wf[i] = *reinterpret_cast<const bf16x8 *>(reinterpret_cast<const char *>(frags + ((size_t)(c >> 5) * NT + i) * kFragElems) + (uint32_t)lane * 16u);
    };
    f32x4 acc[NT][NB];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[i][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // Every workgroup starts at another place of its rows: in step from the first channel on, all of them would be at
    // the same 512 bytes of every 4 KiB row at any time, i.e. at two of the 16 memory channels those rows cover.
    const int nchunk = C / 32, nturn = (nchunk + kReduceWaves - 1) / kReduceWaves;
    const int n_my = nchunk % kReduceWaves == 0 || wave < nchunk % kReduceWaves ? nturn : nturn - 1;   // the wave's chunks
    auto my_chunk = [&](int i) {
        return (i + (int)(blockIdx.x % n_my)) % n_my * kReduceWaves + wave;
    };
    if (n_my > 0) {
        const int c = 32 * my_chunk(0);
        xp.zero();
        fetch_x(c);
#pragma unroll
        for (int i = 0; i < NT; ++i) fetch_w(i, c);
        if (kGrad) {
#pragma unroll
            for (int s = 0; s < kMix; ++s) fetch_g(s, c);
        }
    }
    for (int turn = 0; turn < n_my; ++turn) {
        const int next = 32 * my_chunk(min(turn + 1, n_my - 1));   // (the last one once more: no branch around the loads)
        Row8 carry = xp;
        float mx[8], xx[NB][8];
        bf16x8 xmix[NB] = {};
        if (!kGrad) mix.to_float(mx);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float xv[8];
            xr[b].to_float(xv);
            prev_rows(carry, xr[b]).to_float(xx[b]);
            carry = last_row_first(xr[b]);
#pragma unroll
            for (int e = 0; e < 8; ++e) xx[b][e] = (first[b] ? 0.f : xx[b][e]) - xv[e];
            if (!kGrad) {
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[e] = fmaf(xx[b][e], mx[e], xv[e]);
                xmix[b] = pack_operand(xv);
            } else {
                pin8(xx[b]);
            }
        }
        fetch_x(next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < kMix; ++s) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                bf16x8 o = xmix[b];
                if (kGrad) {
                    float gv[8];
                    gr[kGrad ? s : 0][b].to_float(gv);
#pragma unroll
                    for (int e = 0; e < 8; ++e) gv[e] *= xx[b][e];
                    o = pack_operand(gv);
                }
#pragma unroll
                for (int q = s * RT; q < (s + 1) * RT; ++q) acc[q][b] = mfma32(wf[q], o, acc[q][b]);
            }
            if (kGrad) fetch_g(s, next);
#pragma unroll
            for (int q = s * RT; q < (s + 1) * RT; ++q) fetch_w(q, next);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // add up over the waves, two rounds of kRound tiles; thread (tile, lane) then holds four neighbouring rows of one token
    f32x4 *red = reinterpret_cast<f32x4 *>(smem);
#pragma unroll
    for (int rd = 0; rd < 2; ++rd) {
        if (rd) __syncthreads();
#pragma unroll
        for (int i = 0; i < M::kRound; ++i) {
            const int tile = rd * M::kRound + i;
            red[(wave * M::kRound + i) * 64 + lane] = acc[tile / NB][tile % NB];
        }
        __syncthreads();
        for (int j = threadIdx.x; j < M::kRound * 64; j += kReduceWaves * 64) {
            f32x4 s = red[j];
#pragma unroll
            for (int q = 1; q < kReduceWaves; ++q) s += red[q * M::kRound * 64 + j];
            const int tile = rd * M::kRound + (j >> 6), l = j & 63;
            const int64_t t = tok0 + 16 * (tile % NB) + (l & 15);
            if (t >= n_tok) continue;
            const size_t o = (size_t)t * (kMix * R) + 16 * (tile / NB) + 4 * (l >> 4);
            if (kGrad) {
                float hv[4];
                load4(h + o, hv);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] *= fmaf(-hv[e], hv[e], 1.f);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = tanh_bf16(s[e]);
            }
            store4(out + o, s[0], s[1], s[2], s[3]);
        }
    }
}

// ------------------------------------------------------------------------------------------
// Everything else of the backward: gx, and the sums over tokens.
//
// Workgroup: 64 channels, two token ranges side by side, each walked in steps of 32 tokens (the k-slots of one MFMA).
// A lane holds 8 neighbouring channels of a token (16-byte accesses), the order in which coef and gxm come out of their
// MFMAs when W's and A's rows are assigned as in wkv6_mix.hip; the neighbouring tokens are neighbouring lanes (DPP),
// across steps they are carried in registers.  Three waves take the same 32 channels of a range, one of each role on
// every SIMD:
//   gx waves:  coef, gxx, gxm and from them gx and gmix;
//   W waves:   gcoef, transposed through a tile of their own in LDS (the transposing read), for gW and gbias;
//   A waves:   x_mix, the same way, for gA; they also bring the h and gpre rows that all roles read from LDS.
// (The roles read the same x and g: the later reads find the lines in L1 or L2.  One wave doing everything had a SIMD to
// itself for its 440 registers and every LDS and MFMA latency in the open: 84 us at B8 T1024 C2048 R32 against 75 so.  The
// traffic alone, 256 MB, would take 50 us; the roles alone take 45, 44 and 32 us: vector instructions and LDS on top.)
// R = 64: the W and A waves hold accumulators for half of the rank's columns, a second launch without gx waves (kGx false) does the
// other half.  The gx waves need all of them: a step of the first launch has two parts of 160 columns (32 of each mixer) that go
// through the same two tiles as at R = 32, and gxx and gxm take each part's share (both are linear in it).  B8 T1024 C2048: 136 + 60 us.
// (Tiles of all 320 columns fit once: filled from memory between two barriers in every step, 181 + 63 us.  Now 15 registers of the first
// launch are in scratch memory, 3 at R = 32.)
// ------------------------------------------------------------------------------------------
constexpr int kGradTok = 32;
template <int R, bool kGx> struct MixGrads {
    static constexpr int kThreads = kGx ? 768 : 512;
    static constexpr int kParts = kGx ? R / 32 : 1;          // parts of a step: 32 columns of each mixer go through the tiles at a time
    static constexpr int kCols = kMix * 32;
    static constexpr int kPitch = kCols + 8;                 // elements per token row of their tiles: 8 rows on 8 different bank groups
    static constexpr int kBufs = 2;
    static constexpr int kStagePitch = 40;
    static constexpr bool kLdsA = R == 32;                   // A's fragments in LDS, too (R = 64: from L2)
    static constexpr int kTile = kGradTok * kPitch * 2;      // bytes of one range's rows
    static constexpr int kW = 0;                                                 // [5][R/32][4][64][8]
    static constexpr int kA = kW + (kGx ? kMix * R * 64 * 2 : 0);                // [5R/32][4][64][8]
    static constexpr int kBias = kA + (kGx && kLdsA ? kMix * R * 64 * 2 : 0);    // [5][64] fp32
    static constexpr int kMixX = kBias + kMix * 64 * 4;                          // [64] fp32
    static constexpr int kTiles = kMixX + 64 * 4;                                // [kBufs][2 ranges][h, gpre][32][kPitch]
    static constexpr int kStage = kTiles + kBufs * 4 * kTile;                    // [8 waves][32][kStagePitch]
    static constexpr int kBytes0 = kStage + 8 * kGradTok * kStagePitch * 2;
    static constexpr int kFold = 2 * 40 * 64 * 16;                               // the ranges' accumulators are added up here at the end
    static constexpr int kBytes = kBytes0 > kFold ? kBytes0 : kFold;
    static_assert(kBytes <= 160 * 1024, "LDS of mix_grads_kernel");
};

struct MixGradArgs {
    int64_t n_tok;
    int T, C, nruns, steps;      // a range is steps * 32 tokens, a run two ranges, ranges in token order
    int r0;                      // first column of the rank for the W and A waves
    const bf16_t *x, *h, *gpre, *w, *a_t, *g[kMix];
    const float *bias, *mix_x;
    bf16_t *gx;
    float *edge_first, *edge_last;   // (ranges, C): z of a range's first token; gx of its last token without the next token's z
    float *part_w, *part_a;          // [nruns][C/64][2 halves][20 tiles][64 lanes][4] accumulator tiles
    float *part_bias, *part_mix;     // (ranges, 5, C), (ranges, C)
};

// What a wave walks: its range's tokens, its 32 channels, and the step's x and g, each fetched again for the next step as
// soon as the current one is done with it (the last step fetches itself once more: no branch, and its lines are at hand).
// Tokens past the end read the last token's rows; their x and previous-token values are taken as zero.
struct MixWalk {
    const MixGradArgs &p;
    const int l16, g, c0;
    const int64_t first_tok;
    int64_t base;                // element offset of the step last aimed at
    uint32_t off[2];             // the lane's byte offset in its two 16-token blocks
    int pos[2], pos_step;        // the lane's tokens' positions in their sequences
    int64_t left;                // tokens from the current step's first to the end
    Row8 xr[2], gr[kMix][2], before;   // before: in lane 0, the row of the token before the step
    bool valid[2], last[2];      // of the current step's tokens: not past the end, the last of a sequence

    __device__ __forceinline__ MixWalk(const MixGradArgs &a, int range, int chan, int lane)
        : p(a), l16(lane & 15), g(lane >> 4), c0(chan), first_tok((int64_t)range * a.steps * kGradTok) {
#pragma unroll
        for (int b = 0; b < 2; ++b) pos[b] = (int)((first_tok + 16 * b + l16) % p.T);
        pos_step = kGradTok % p.T;
        left = p.n_tok - first_tok;
        before.zero();
        if (l16 == 0 && left > 0 && pos[0] != 0) before.load(p.x + (first_tok - 1) * p.C + c0 + 8 * g);
        aim(0);
        fetch_x();
    }
    __device__ __forceinline__ void aim(int step) {
        const int64_t t0 = min(first_tok + step * kGradTok, p.n_tok - 1), rest = p.n_tok - 1 - t0;
        const int most = rest < kGradTok ? (int)rest : kGradTok;
        base = uniform64(t0 * p.C + c0);
#pragma unroll
        for (int b = 0; b < 2; ++b) off[b] = ((uint32_t)min(16 * b + l16, most) * (uint32_t)p.C + 8 * g) * 2u;
    }
    __device__ __forceinline__ void fetch_x() {
#pragma unroll
        for (int b = 0; b < 2; ++b) load_row8(xr[b], p.x + base, off[b]);
    }
    __device__ __forceinline__ void fetch_g(int s) {
#pragma unroll
        for (int b = 0; b < 2; ++b) load_row8(gr[s][b], p.g[s] + base, off[b]);
    }
    // x and xx of the step's tokens; moves on to the next step's positions
    __device__ __forceinline__ void x_and_xx(float (&xv)[2][8], float (&xx)[2][8]) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            valid[b] = 16 * b + l16 < left;
            last[b] = pos[b] == p.T - 1;
            Row8 prev = prev_rows(before, xr[b]), cur = xr[b];
            before = last_row_first(xr[b]);
            const bool use_prev = valid[b] && pos[b] != 0;
            prev.a.x = use_prev ? prev.a.x : 0; prev.a.y = use_prev ? prev.a.y : 0; prev.a.z = use_prev ? prev.a.z : 0; prev.a.w = use_prev ? prev.a.w : 0;
            cur.a.x = valid[b] ? cur.a.x : 0; cur.a.y = valid[b] ? cur.a.y : 0; cur.a.z = valid[b] ? cur.a.z : 0; cur.a.w = valid[b] ? cur.a.w : 0;
            cur.to_float(xv[b]);
            prev.to_float(xx[b]);
#pragma unroll
            for (int e = 0; e < 8; ++e) xx[b][e] -= xv[b][e];
            pos[b] += pos_step;
            if (pos[b] >= p.T) pos[b] -= p.T;
        }
        left -= kGradTok;
    }
};

__device__ __forceinline__ void load8(const float *p, float (&v)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4 *>(p), b = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
}
__device__ __forceinline__ void store8(float *p, const float (&v)[8]) {
    *reinterpret_cast<f32x4 *>(p) = (f32x4){v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4 *>(p + 4) = (f32x4){v[4], v[5], v[6], v[7]};
}

// Rows of h or gpre for a range's tile: 128 threads, four per token, 32 columns (of one mixer) at a time.  `r0`: the first of them
template <int R, bool kGx> struct MixTile {
    u32x4 v[kMix];
    __device__ __forceinline__ void fetch(const MixGradArgs &p, const bf16_t *src, int64_t first_tok, int step, int r0, int tid) {
        const int64_t t0 = uniform64(min(first_tok + step * kGradTok, p.n_tok - 1)), rest = p.n_tok - 1 - t0;
        const uint32_t o = (uint32_t)(min(tid >> 2, (int)(rest < kGradTok ? rest : kGradTok)) * (kMix * R) + (tid & 3) * 8 + (kGx ? 0 : r0)) * 2u;
        const char *b = reinterpret_cast<const char *>(src + t0 * (kMix * R) + (kGx ? r0 : 0));
#pragma unroll
        for (int j = 0; j < kMix; ++j) v[j] = *reinterpret_cast<const u32x4 *>(b + o + j * 2 * R);
    }
    __device__ __forceinline__ void put(bf16_t *tile, int tid) const {
#pragma unroll
        for (int j = 0; j < kMix; ++j)
            *reinterpret_cast<u32x4 *>(tile + (tid >> 2) * MixGrads<R, kGx>::kPitch + (tid & 3) * 8 + 32 * j) = v[j];
    }
};
// where a range's h (which = 0) or gpre (1) rows are of part number `turn` (step * kParts + part)
template <int R, bool kGx> __device__ __forceinline__ bf16_t *mix_tile(unsigned char *smem, int turn, int rg, int which) {
    typedef MixGrads<R, kGx> L;
    return reinterpret_cast<bf16_t *>(smem + L::kTiles + (((turn & 1) * 2 + rg) * 2 + which) * L::kTile);
}
// operand fragment with the k-slots along a step's 32 tokens: column n0 + l16 of a tile.  A lane group's four slots are
// tokens two apart: with 20 banks from row to row, their four 32-byte pieces then lie on all 32 different banks.
__device__ __forceinline__ bf16x8 mix_frag_tokens(const bf16_t *tile, int pitch, int n0, int l16, int g) {
    const bf16_t *q = tile + (8 * (g >> 1) + (g & 1) + 2 * (l16 >> 2)) * pitch + n0 + 4 * (l16 & 3);
    typedef s16x4 __attribute__((address_space(3))) *lds4;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)q));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(q + 16 * pitch)));
    return make_bf16x8(lo[0], lo[1], hi[0], hi[1]);
}

// operand row l of tile ct <-> this channel of the workgroup's 64
__device__ __forceinline__ int mix_frag_channel(int ct, int l) { return 32 * (ct >> 1) + 8 * (l >> 2) + 4 * (ct & 1) + (l & 3); }

template <int R>
__device__ __forceinline__ void mix_gx_wave(const MixGradArgs &p, unsigned char *smem, int range, int rg, int cg, int half, int lane)
{
    typedef MixGrads<R, true> L;
    constexpr int kParts = L::kParts, kPitch = L::kPitch;
    const int l16 = lane & 15, g = lane >> 4, C = p.C;
    const bf16_t *wf = reinterpret_cast<const bf16_t *>(smem + L::kW), *af = reinterpret_cast<const bf16_t *>(smem + L::kA);
    const float *bias_l = reinterpret_cast<const float *>(smem + L::kBias) + 32 * half + 8 * g;
    const float *mix_l = reinterpret_cast<const float *>(smem + L::kMixX) + 32 * half + 8 * g;
    const int64_t first_tok = (int64_t)range * p.steps * kGradTok;
    // (R = 64) A's columns of the workgroup, and the lane's place in them: tile 2 half, the other tile's rows are four channels on
    const char *a_cols = reinterpret_cast<const char *>(p.a_t + (size_t)cg * 64 * (kMix * R));
    const uint32_t a_off = (uint32_t)(mix_frag_channel(2 * half, l16) * (kMix * R) + 8 * g) * 2u;
    MixWalk wk(p, range, cg * 64 + half * 32, lane);
#pragma unroll
    for (int s = 0; s < kMix; ++s) wk.fetch_g(s);
    float gmix[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float pend[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // gx of the step's last token, waiting for the next token's z
    bool pend_valid = false, pend_last = false;
    auto put = [&](int64_t base, uint32_t o, const float (&v)[8]) {
        *reinterpret_cast<bf16x8 *>(reinterpret_cast<char *>(p.gx + base) + o) = pack_operand(v);
    };
    for (int step = 0; step < p.steps; ++step) {
        const int next = min(step + 1, p.steps - 1);
        const int64_t cur_base = wk.base, step_tok = first_tok + step * kGradTok;
        const uint32_t cur_off[2] = {wk.off[0], wk.off[1]};
        float xx[2][8], gsum[2][8], gxx[2][8];
        f32x4 xm[2][2];   // gxm, the same lane order as coef
        auto take_x = [&]() {
            float xv[2][8];
            wk.x_and_xx(xv, xx);
            if (kParts == 1) wk.aim(next);
            wk.fetch_x();
        };
#pragma unroll
        for (int part = 0; part < kParts; ++part) {
            __syncthreads();
            const bf16_t *ht = mix_tile<R, true>(smem, step * kParts + part, rg, 0), *gt = mix_tile<R, true>(smem, step * kParts + part, rg, 1);
            if (kParts == 1) take_x();
            else if (part == kParts - 1) wk.aim(next);
            if (part > 0) {   // (as loaded: not the values unpacked for the part before, twice the registers)
#pragma unroll
                for (int s = 0; s < kMix; ++s)
#pragma unroll
                    for (int b = 0; b < 2; ++b) asm volatile("" : "+v"(wk.gr[s][b].a.x), "+v"(wk.gr[s][b].a.y), "+v"(wk.gr[s][b].a.z), "+v"(wk.gr[s][b].a.w));
            }
#pragma unroll
            for (int s = 0; s < kMix; ++s) {
                f32x4 cf[2][2];
                bf16x8 wfr[2];
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    cf[0][m] = cf[1][m] = part == 0 ? *reinterpret_cast<const f32x4 *>(bias_l + 64 * s + 4 * m) : (f32x4){0.f, 0.f, 0.f, 0.f};
                    wfr[m] = *reinterpret_cast<const bf16x8 *>(wf + (size_t)(((s * kParts + part) * 4 + 2 * half + m) * 64 + lane) * 8);
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const bf16x8 hr = *reinterpret_cast<const bf16x8 *>(ht + (16 * b + l16) * kPitch + s * 32 + 8 * g);
#pragma unroll
                    for (int m = 0; m < 2; ++m) cf[b][m] = mfma32(wfr[m], hr, cf[b][m]);
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    float gv[8];
                    wk.gr[s][b].to_float(gv);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (part == kParts - 1) gsum[b][e] = s == 0 ? gv[e] : gsum[b][e] + gv[e];
                        gxx[b][e] = part == 0 && s == 0 ? gv[e] * cf[b][e >> 2][e & 3] : fmaf(gv[e], cf[b][e >> 2][e & 3], gxx[b][e]);
                    }
                    if (part == kParts - 1) pin8(gsum[b]);   // (or the sums sink to their use behind the branches below, with every g still in registers)
                    pin8(gxx[b]);
                }
                if (part == kParts - 1) wk.fetch_g(s);
                if (s & 1) __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (part == 0) {
#pragma unroll
                for (int b = 0; b < 2; ++b) xm[b][0] = xm[b][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int s = 0; s < kMix; ++s) {
                const int kk = s * kParts + part;   // 32 of A's stacked rows
                bf16x8 afr[2];
#pragma unroll
                for (int m = 0; m < 2; ++m)
                    afr[m] = L::kLdsA ? *reinterpret_cast<const bf16x8 *>(af + (size_t)((kk * 4 + 2 * half + m) * 64 + lane) * 8)
                                      : *reinterpret_cast<const bf16x8 *>(a_cols + a_off + m * 4 * (kMix * R) * 2 + 64 * kk);
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const bf16x8 gq = *reinterpret_cast<const bf16x8 *>(gt + (16 * b + l16) * kPitch + 32 * s + 8 * g);
#pragma unroll
                    for (int m = 0; m < 2; ++m) xm[b][m] = mfma32(afr[m], gq, xm[b][m]);
                }
                if (s & 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (kParts > 1) take_x();   // (here, not ahead of the products: xx is not needed before, and its sixteen registers are)
        float o[2][8], mx[8];
        load8(mix_l, mx);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float m = xm[b][e >> 2][e & 3];
                gmix[e] = fmaf(m, xx[b][e], gmix[e]);
                gxx[b][e] = fmaf(m, mx[e], gxx[b][e]);             // z
                o[b][e] = (gsum[b][e] + m) - gxx[b][e];
            }
        pin8(o[0]); pin8(o[1]); pin8(gmix);
        __builtin_amdgcn_sched_barrier(0);
        if (step == 0 && l16 == 0) store8(p.edge_first + (size_t)range * C + wk.c0 + 8 * g, gxx[0]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {                  // lane 15: z of this step's first token
            const float z = first_to_last(gxx[0][e]);  // (with all lanes: a lane that is switched off is not read)
            pend[e] += pend_last ? 0.f : z;
        }
        if (step > 0 && pend_valid && l16 == 15) {
            put((step_tok - 1) * C + wk.c0, 16u * g, pend);
        }
        float zn[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) zn[e] = next_lane(first_to_last(gxx[1][e]), gxx[0][e]);
        if (!wk.last[0]) {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[0][e] += zn[e];
        }
        if (wk.valid[0]) put(cur_base, cur_off[0], o[0]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            pend[e] = o[1][e];
            zn[e] = next_lane(0.f, gxx[1][e]);
        }
        if (!wk.last[1]) {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[1][e] += zn[e];
        }
        if (wk.valid[1] && l16 < 15) put(cur_base, cur_off[1], o[1]);
        pend_valid = wk.valid[1]; pend_last = wk.last[1];
    }
    if (pend_valid && l16 == 15) {   // the range's last token: complete if a sequence ends with it
        if (pend_last) put((first_tok + (int64_t)p.steps * kGradTok - 1) * C + wk.c0, 16u * g, pend);
        else store8(p.edge_last + (size_t)range * C + wk.c0 + 8 * g, pend);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) gmix[e] += __shfl_xor(gmix[e], m);
    if (l16 == 0) store8(p.part_mix + (size_t)range * C + wk.c0 + 8 * g, gmix);
    __syncthreads();   // (the other waves fold their accumulators in two phases)
    __syncthreads();
}

// The second range's accumulators through LDS to the first's wave, then one partial per workgroup.
template <int N>
__device__ __forceinline__ void mix_fold(const f32x4 (&acc)[N], f32x4 *fold, float *part, size_t tile0, int rg, int lane)
{
    __syncthreads();
    if (rg == 1) {
#pragma unroll
        for (int i = 0; i < N; ++i) fold[i * 64 + lane] = acc[i];
    }
    __syncthreads();
    if (rg == 0) {
        f32x4 *q = reinterpret_cast<f32x4 *>(part) + tile0 * 64 + lane;
#pragma unroll
        for (int i = 0; i < N; ++i) q[i * 64] = acc[i] + fold[i * 64 + lane];
    }
}

template <int R, bool kGx>
__device__ __forceinline__ void mix_w_wave(const MixGradArgs &p, unsigned char *smem, int range, int rg, int run, int cg, int half, int lane)
{
    typedef MixGrads<R, kGx> L;
    const int l16 = lane & 15, g = lane >> 4, C = p.C;
    bf16_t *stage = reinterpret_cast<bf16_t *>(smem + L::kStage) + (2 * rg + half) * kGradTok * L::kStagePitch;
    f32x4 acc[4 * kMix];                                      // (s, rank tile, channel tile): rows = rank, columns = channels
    f32x4 acc_b[2];                                           // row s: gbias of mixer s
#pragma unroll
    for (int i = 0; i < 4 * kMix; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    acc_b[0] = acc_b[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
    MixWalk wk(p, range, cg * 64 + half * 32, lane);
    // g_s is fetched only while g_{s-kAhead} is worked on, for the registers' sake: the gx waves brought its lines to L2
    constexpr int kAhead = 2;
#pragma unroll
    for (int s = 0; s < kAhead; ++s) wk.fetch_g(s);
    for (int step = 0; step < p.steps; ++step) {
        __syncthreads();
        const bf16_t *ht = mix_tile<R, kGx>(smem, step * L::kParts, rg, 0);   // (the part with this launch's columns)
        float xx[2][8];
        {
            float xv[2][8];
            wk.x_and_xx(xv, xx);
            pin8(xx[0]); pin8(xx[1]);
        }
#pragma unroll
        for (int s = 0; s < kMix; ++s) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                float gv[8];
                wk.gr[s][b].to_float(gv);
#pragma unroll
                for (int e = 0; e < 8; ++e) gv[e] *= xx[b][e];
                *reinterpret_cast<bf16x8 *>(stage + (16 * b + l16) * L::kStagePitch + 8 * g) = pack_operand(gv);
            }
            if (s + kAhead == kMix) { wk.aim(min(step + 1, p.steps - 1)); wk.fetch_x(); }
            wk.fetch_g((s + kAhead) % kMix);
            const bf16x8 gc[2] = {mix_frag_tokens(stage, L::kStagePitch, 0, l16, g), mix_frag_tokens(stage, L::kStagePitch, 16, l16, g)};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x8 hq = mix_frag_tokens(ht, L::kPitch, s * 32 + 16 * i, l16, g);
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[4 * s + 2 * i + j] = mfma32(hq, gc[j], acc[4 * s + 2 * i + j]);
            }
            uint32_t one = l16 == s ? 0x3f803f80u : 0u;         // bf16 ones in row s alone: the mixers' sums share a tile
            asm volatile("" : "+v"(one));                       // (made where it is used: five operands kept across the loop are 20 registers)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc_b[j] = mfma32(make_bf16x8(one, one, one, one), gc[j], acc_b[j]);
            if (s & 1) __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (L::kParts == 2) __syncthreads();   // (the other part is the gx waves')
    }
    if (p.r0 == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * g + e < kMix) p.part_bias[((size_t)range * kMix + 4 * g + e) * C + wk.c0 + 16 * j + l16] = acc_b[j][e];
    }
    mix_fold(acc, reinterpret_cast<f32x4 *>(smem) + half * 40 * 64, p.part_w, ((size_t)(run * (C / 64) + cg) * 2 + half) * 20, rg, lane);
}

template <int R, bool kGx>
__device__ __forceinline__ void mix_a_wave(const MixGradArgs &p, unsigned char *smem, int range, int rg, int run, int cg, int half, int lane)
{
    typedef MixGrads<R, kGx> L;
    const int l16 = lane & 15, g = lane >> 4, tid = half * 64 + lane, C = p.C;
    const float *mix_l = reinterpret_cast<const float *>(smem + L::kMixX) + 32 * half + 8 * g;
    bf16_t *stage = reinterpret_cast<bf16_t *>(smem + L::kStage) + (4 + 2 * rg + half) * kGradTok * L::kStagePitch;
    f32x4 acc[4 * kMix];                                      // (s, rank tile, channel tile): rows = channels, columns = rank
#pragma unroll
    for (int i = 0; i < 4 * kMix; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int64_t first_tok = (int64_t)range * p.steps * kGradTok;
    MixTile<R, kGx> tile;
    constexpr int kParts = L::kParts;
    const int r0 = kGx ? 0 : p.r0;
    tile.fetch(p, p.h, first_tok, 0, r0, tid);
    tile.put(mix_tile<R, kGx>(smem, 0, rg, 0), tid);
    tile.fetch(p, p.gpre, first_tok, 0, r0, tid);
    tile.put(mix_tile<R, kGx>(smem, 0, rg, 1), tid);
    MixWalk wk(p, range, cg * 64 + half * 32, lane);
    // one part of a step, the tiles of the part behind it brought meanwhile
    auto take = [&](auto part, int step) {
        constexpr int kPart = decltype(part)::value;
        __syncthreads();
        const int next = min(step + 1, p.steps - 1);
        const int bstep = kPart + 1 < kParts ? step : next, br0 = kParts == 2 ? 32 * (1 - kPart) : r0;
        tile.fetch(p, p.h, first_tok, bstep, br0, tid);
        if constexpr (kPart == 0) {
            float xv[2][8], xx[2][8], mx[8];
            wk.x_and_xx(xv, xx);
            wk.aim(next);
            wk.fetch_x();
            load8(mix_l, mx);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int e = 0; e < 8; ++e) xv[b][e] = fmaf(xx[b][e], mx[e], xv[b][e]);
                *reinterpret_cast<bf16x8 *>(stage + (16 * b + l16) * L::kStagePitch + 8 * g) = pack_operand(xv[b]);
            }
        }
        tile.put(mix_tile<R, kGx>(smem, step * kParts + kPart + 1, rg, 0), tid);
        tile.fetch(p, p.gpre, first_tok, bstep, br0, tid);
        if constexpr (kPart == 0) {
            const bf16x8 xt[2] = {mix_frag_tokens(stage, L::kStagePitch, 0, l16, g), mix_frag_tokens(stage, L::kStagePitch, 16, l16, g)};
            const bf16_t *gt = mix_tile<R, kGx>(smem, step * kParts + kPart, rg, 1);
#pragma unroll
            for (int i = 0; i < 2 * kMix; ++i) {
                const bf16x8 gq = mix_frag_tokens(gt, L::kPitch, 16 * i, l16, g);
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[2 * i + j] = mfma32(xt[j], gq, acc[2 * i + j]);
                if (i % 5 == 4) __builtin_amdgcn_sched_barrier(0);
            }
        }
        tile.put(mix_tile<R, kGx>(smem, step * kParts + kPart + 1, rg, 1), tid);
    };
    for (int step = 0; step < p.steps; ++step) {
        take(std::integral_constant<int, 0>{}, step);
        if constexpr (kParts == 2) take(std::integral_constant<int, 1>{}, step);
    }
    mix_fold(acc, reinterpret_cast<f32x4 *>(smem) + (half * 40 + 20) * 64, p.part_a, ((size_t)(run * (C / 64) + cg) * 2 + half) * 20, rg, lane);
}

template <int R, bool kGx>
__global__ __launch_bounds__(kGx ? 768 : 512) void mix_grads_kernel(MixGradArgs p)
{
    typedef MixGrads<R, kGx> L;
    constexpr int KW = R / 32, KA = kMix * R / 32;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = wave & 1, rg = (wave >> 1) & 1;
    const int run = (int)blockIdx.x % p.nruns, cg = (int)blockIdx.x / p.nruns, range = run * 2 + rg;
    bf16_t *wf = reinterpret_cast<bf16_t *>(smem + L::kW), *af = reinterpret_cast<bf16_t *>(smem + L::kA);
    float *bias_l = reinterpret_cast<float *>(smem + L::kBias), *mix_l = reinterpret_cast<float *>(smem + L::kMixX);
    if (kGx) {
        for (int i = threadIdx.x; i < kMix * KW * 4 * 64; i += L::kThreads) {
            const int l = i & 63, ct = (i >> 6) & 3, kk = (i >> 8) % KW, s = (i >> 8) / KW;
            *reinterpret_cast<uint4 *>(wf + (size_t)i * 8) =
                *reinterpret_cast<const uint4 *>(p.w + ((size_t)s * p.C + cg * 64 + mix_frag_channel(ct, l & 15)) * R + 32 * kk + 8 * (l >> 4));
        }
        if (L::kLdsA)
            for (int i = threadIdx.x; i < KA * 4 * 64; i += L::kThreads) {
                const int l = i & 63, ct = (i >> 6) & 3, kk = i >> 8;
                *reinterpret_cast<uint4 *>(af + (size_t)i * 8) =
                    *reinterpret_cast<const uint4 *>(p.a_t + (size_t)(cg * 64 + mix_frag_channel(ct, l & 15)) * (kMix * R) + 32 * kk + 8 * (l >> 4));
            }
        for (int i = threadIdx.x; i < kMix * 64; i += L::kThreads) bias_l[i] = p.bias[(size_t)(i >> 6) * p.C + cg * 64 + (i & 63)];
    }
    if (threadIdx.x < 64) mix_l[threadIdx.x] = p.mix_x[cg * 64 + threadIdx.x];
    __syncthreads();
    // (the waves that fetch from memory and fill the tiles go first where a SIMD has a choice)
    if (wave < 4) {
        __builtin_amdgcn_s_setprio(3);
        mix_a_wave<R, kGx>(p, smem, range, rg, run, cg, half, lane);
    } else if (wave < 8) {
        mix_w_wave<R, kGx>(p, smem, range, rg, run, cg, half, lane);
    } else if (kGx) {
        __builtin_amdgcn_s_setprio(3);
        mix_gx_wave<R>(p, smem, range, rg, cg, half, lane);
    }
}

// Sums of the workgroups' partials -> gradients of the weights, and gx of the tokens at the ends of the ranges.
// blockIdx.y: 0 gW, 1 gA (columns r0..r0+31 of the rank), 2 gbias and gmix, 3 the ranges' ends.
template <typename Tw>
__global__ __launch_bounds__(256) void mix_finish_kernel(MixGradArgs p, int R, Tw *__restrict__ gw, Tw *__restrict__ ga,
                                                         float *__restrict__ gbias, float *__restrict__ gmix)
{
    const int C = p.C, nranges = 2 * p.nruns;
    const int i = (int)blockIdx.x * 256 + threadIdx.x;
    if (blockIdx.y < 2) {
        const int per_run = (C / 64) * 2 * 20 * 64;
        if (i >= per_run) return;
        const f32x4 *src = reinterpret_cast<const f32x4 *>(blockIdx.y == 0 ? p.part_w : p.part_a) + i;
        f32x4 s = src[0];
#pragma unroll 8
        for (int q = 1; q < p.nruns; ++q) s += src[(size_t)q * per_run];
        const int lane = i & 63, l16 = lane & 15, g = lane >> 4, tile = (i >> 6) % 20, c0 = (i / (64 * 20)) * 32;
        if (blockIdx.y == 0) {   // tile (s, rank tile, channel tile): rows = rank, columns = channels
            const int r = p.r0 + 16 * ((tile >> 1) & 1) + 4 * g, c = c0 + 16 * (tile & 1) + l16;
            store4(gw + ((size_t)(tile >> 2) * C + c) * R + r, s[0], s[1], s[2], s[3]);
        } else {                 // tile (s, rank tile, channel tile): rows = channels, columns = rank
            const int r = (tile >> 2) * R + p.r0 + 16 * ((tile >> 1) & 1) + l16, c = c0 + 16 * (tile & 1) + 4 * g;
            store4(ga + (size_t)r * C + c, s[0], s[1], s[2], s[3]);
        }
    } else if (blockIdx.y == 2) {
        if (i >= (kMix + 1) * C) return;
        const bool is_mix = i >= kMix * C;
        float s = 0.f;
#pragma unroll 8
        for (int q = 0; q < nranges; ++q) s += is_mix ? p.part_mix[(size_t)q * C + i - kMix * C] : p.part_bias[(size_t)q * kMix * C + i];
        if (is_mix) gmix[i - kMix * C] = s; else gbias[i] = s;
    } else {
        const int per = C / 4;
        for (int j = i; j < (nranges - 1) * per; j += (int)gridDim.x * 256) {
            const int e = j / per, c = (j % per) * 4;
            const int64_t t = (int64_t)(e + 1) * p.steps * kGradTok - 1;
            if (t >= p.n_tok || t % p.T == p.T - 1) continue;
            const float4 a = *reinterpret_cast<const float4 *>(p.edge_last + (size_t)e * C + c);
            const float4 z = *reinterpret_cast<const float4 *>(p.edge_first + (size_t)(e + 1) * C + c);
            store4(p.gx + (size_t)t * C + c, a.x + z.x, a.y + z.y, a.z + z.z, a.w + z.w);
        }
    }
}

// ---- host side ----------------------------------------------------------------------------
static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

size_t shift_mix_weights_bytes(int64_t C, int64_t R) { return 4 * align256((size_t)(kMix * R * C) * sizeof(bf16_t)); }

struct MixWeightForms {
    bf16_t *a_frag, *wt_frag, *a_t, *w;
    MixWeightForms(void *block, int64_t C, int64_t R) {
        char *b = reinterpret_cast<char *>(block);
        const size_t n = align256((size_t)(kMix * R * C) * sizeof(bf16_t));
        a_frag = (bf16_t *)b; wt_frag = (bf16_t *)(b + n); a_t = (bf16_t *)(b + 2 * n); w = (bf16_t *)(b + 3 * n);
    }
};

template <int R, bool kGrad>
static hipError_t launch_reduce(hipStream_t st, int64_t n, int64_t T, int64_t C, const void *x, const float *mix_x, const bf16_t *frags,
                                const void *const g[5], const void *h, void *out) {
    constexpr auto kern = mix_reduce_kernel<R, kGrad>;
    hipError_t e = allow_dynamic_lds<kern>(MixReduce<R>::kLds);
    if (e != hipSuccess) return e;
    auto gp = [&](int i) { return g ? (const bf16_t *)g[i] : nullptr; };
    const int64_t per = 16 * MixReduce<R>::kBlocks;
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + per - 1) / per)), dim3(kReduceWaves * 64), MixReduce<R>::kLds, st, n, (int)T, (int)C,
                       (const bf16_t *)x, mix_x, frags, gp(0), gp(1), gp(2), gp(3), gp(4), (const bf16_t *)h, (bf16_t *)out);
    return hipGetLastError();
}

hipError_t shift_mix_forward(hipStream_t st, int weight_dtype, int64_t B, int64_t T, int64_t C, int64_t R, const void *x, const float *mix_x,
                             const void *a, const void *w2t, const float *bias, void *weights, void *h, void *const out[5]) {
    const MixWeightForms w(weights, C, R);
    const dim3 grid((unsigned)(C / 32), 2);
    auto pack = [&](auto kernel, auto *tag) {
        typedef std::remove_pointer_t<decltype(tag)> Tw;
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, (int)C, (const Tw *)a, (const Tw *)w2t, w.a_frag, w.wt_frag, w.a_t, w.w);
    };
    if (weight_dtype == kF32) R == 32 ? pack(mix_weights_kernel<float, 32>, (float *)nullptr) : pack(mix_weights_kernel<float, 64>, (float *)nullptr);
    else R == 32 ? pack(mix_weights_kernel<bf16_t, 32>, (bf16_t *)nullptr) : pack(mix_weights_kernel<bf16_t, 64>, (bf16_t *)nullptr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = R == 32 ? launch_reduce<32, false>(st, B * T, T, C, x, mix_x, w.a_frag, nullptr, nullptr, h)
                : launch_reduce<64, false>(st, B * T, T, C, x, mix_x, w.a_frag, nullptr, nullptr, h);
    if (e != hipSuccess) return e;
    return shift_mix_five(st, B, T, C, R, x, h, w.w, bias, out);
}

// how the tokens are cut for mix_grads_kernel: runs of two ranges each, as many as the chip holds at once and no more (a
// partial of every weight gradient per run; and a workgroup's LDS leaves no room for a second one on its compute unit, so
// that one workgroup too many is a second round of full length).  Backward at 8192 tokens, one run less than needed to give
// every compute unit something / one more than fits: H12 68 / 91 us, H24 104 / 137, H40 198 / 251, H48 231 / 300.
struct MixCut {
    int nruns, steps;
    MixCut(int64_t n, int64_t C) {
        const int64_t groups = C / 64, fit = compute_units() / groups, want = fit > 1 ? fit : 1;   // runs that the chip holds at once
        const int64_t most = (n + 2 * kGradTok - 1) / (2 * kGradTok);                       // runs of one step per range
        const int64_t runs = want < most ? want : most;
        steps = (int)((n + runs * 2 * kGradTok - 1) / (runs * 2 * kGradTok));
        nruns = (int)((n + (int64_t)steps * 2 * kGradTok - 1) / ((int64_t)steps * 2 * kGradTok));
    }
};

struct MixWorkspace {
    size_t gpre, part_w, part_a, part_bias, part_mix, edge_first, edge_last, bytes;
    MixWorkspace(int64_t n, int64_t C, int64_t R, const MixCut &cut) {
        size_t o = 0;
        auto take = [&](size_t b) { const size_t at = o; o += align256(b); return at; };
        gpre = take((size_t)(n * kMix * R) * 2);
        part_w = take((size_t)cut.nruns * kMix * 32 * C * 4);
        part_a = take((size_t)cut.nruns * kMix * 32 * C * 4);
        part_bias = take((size_t)2 * cut.nruns * kMix * C * 4);
        part_mix = take((size_t)2 * cut.nruns * C * 4);
        edge_first = take((size_t)2 * cut.nruns * C * 4);
        edge_last = take((size_t)2 * cut.nruns * C * 4);
        bytes = o;
    }
};

size_t shift_mix_backward_workspace_bytes(int64_t B, int64_t T, int64_t C, int64_t R) {
    return MixWorkspace(B * T, C, R, MixCut(B * T, C)).bytes;
}

template <int R, bool kGx>
static hipError_t launch_grads(hipStream_t st, const MixGradArgs &p) {
    constexpr auto kern = mix_grads_kernel<R, kGx>;
    typedef MixGrads<R, kGx> L;
    hipError_t e = allow_dynamic_lds<kern>(L::kBytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.nruns * (p.C / 64))), dim3(L::kThreads), L::kBytes, st, p);
    return hipGetLastError();
}

hipError_t shift_mix_backward(hipStream_t st, int weight_dtype, int64_t B, int64_t T, int64_t C, int64_t R, const void *x, const float *mix_x,
                              const float *bias, const void *weights, const void *h, const void *const gout[5],
                              void *gx, float *gmix_x, void *ga, void *gw2t, float *gbias, void *workspace) {
    const MixWeightForms w(const_cast<void *>(weights), C, R);
    const int64_t n = B * T;
    const MixCut cut(n, C);
    const MixWorkspace ws(n, C, R, cut);
    char *base = reinterpret_cast<char *>(workspace);
    void *gpre = base + ws.gpre;
    hipError_t e = R == 32 ? launch_reduce<32, true>(st, n, T, C, x, mix_x, w.wt_frag, gout, h, gpre)
                           : launch_reduce<64, true>(st, n, T, C, x, mix_x, w.wt_frag, gout, h, gpre);
    if (e != hipSuccess) return e;
    MixGradArgs p = {};
    p.n_tok = n; p.T = (int)T; p.C = (int)C; p.nruns = cut.nruns; p.steps = cut.steps;
    p.x = (const bf16_t *)x; p.h = (const bf16_t *)h; p.gpre = (const bf16_t *)gpre; p.w = w.w; p.a_t = w.a_t;
    for (int s = 0; s < kMix; ++s) p.g[s] = (const bf16_t *)gout[s];
    p.bias = bias; p.mix_x = mix_x; p.gx = (bf16_t *)gx;
    p.edge_first = (float *)(base + ws.edge_first); p.edge_last = (float *)(base + ws.edge_last);
    p.part_w = (float *)(base + ws.part_w); p.part_a = (float *)(base + ws.part_a);
    p.part_bias = (float *)(base + ws.part_bias); p.part_mix = (float *)(base + ws.part_mix);
    auto finish = [&](unsigned rows) {
        // (blockIdx.y counts from 0; with rows = 2 only the weights' sums)
        const dim3 grid((unsigned)(((C / 64) * 2 * 20 * 64 + 255) / 256), rows);
        if (weight_dtype == kF32)
            hipLaunchKernelGGL(mix_finish_kernel<float>, grid, dim3(256), 0, st, p, (int)R, (float *)gw2t, (float *)ga, gbias, gmix_x);
        else
            hipLaunchKernelGGL(mix_finish_kernel<bf16_t>, grid, dim3(256), 0, st, p, (int)R, (bf16_t *)gw2t, (bf16_t *)ga, gbias, gmix_x);
        return hipGetLastError();
    };
    e = R == 32 ? launch_grads<32, true>(st, p) : launch_grads<64, true>(st, p);
    if (e == hipSuccess) e = finish(4);
    if (R == 64 && e == hipSuccess) {
        p.r0 = 32;
        e = launch_grads<64, false>(st, p);
        if (e == hipSuccess) e = finish(2);
    }
    return e;
}

}  // namespace wkv6
