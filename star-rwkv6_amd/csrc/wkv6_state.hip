// What a time segment leaves alone: the state it builds from zero and the decay over it, for gfx950 (bf16 tensors).  The first
// pass over the segments of a sequence, forward (k, v) and, read back to front with r and gy in their place, backward.
//
// Nothing but the state is wanted, so a chunk of 64 tokens is one step:
//   S <- e^{c_64} o S + K^^T V ,   K^_s = k_s e^{c_64 - c_{s+1}}     (c: running sum of the log decays)
// with every exponent <= 0: no reference inside the chunk, no range to leave, two exponentials per element of k, one scaling of the
// state and eight MFMAs per wave and chunk.  (As the tile form's kernel without y, four tiles of 16 tokens to a chunk, each with a
// scaling of its own: training pair of B1 T8192 H32 164 us, so 155, B2 T4096 H16 96.7 / 90.0, T1000 H8 36.6 / 33.2, with the output
// stage T4096 H32 100.7 / 94.1; prompt T1337 H32 23.7 / 22.0, with the output stage T3000 36.7 / 34.0.)
//
// Bound by the reading of k, v and w where the segments fill the chip (B1 T8192 H32: 100 MB), by a launch and the latency of the
// first loads where they are short.  More in flight is slower: rows four, five and six chunks ahead 156, 157 and 160 us for
// the pair above instead of 155, 92, 93 and 96 instead of 90.
// One workgroup per (segment, head): four loading waves (wave p <-> tokens 16p .. 16p+15 of every chunk) bring the rows straight
// into LDS three chunks ahead and form K^; a wave's sums over its 16 tokens go to the others through LDS, so a chunk's operands take
// two steps: the sums, and a barrier later K^.  Four consumer waves (q): value columns 16q .. of the state.
#include "wkv6_mfma.h"
#include "wkv6_kernels.h"
#include "wkv6_block.h"

namespace wkv6 {

struct StateLds {
    static constexpr int kAhead = 3;                                 // chunks between the request of the rows and their use
    static constexpr int kV = 0;                                     // [chunk % (kAhead + 1)] v tiles
    static constexpr int kKW = kV + (kAhead + 1) * kTileBytes;       // [chunk % (kAhead - 1)][k, w] tiles (done with two chunks before use)
    static constexpr int kOp = kKW + (kAhead - 1) * 2 * kTileBytes;  // [2] K^
    static constexpr int kTot = kOp + 2 * kTileBytes;                // [2][4 waves][64] exponents over each wave's tokens
    static constexpr int kG = kTot + 2 * 4 * kN * 4;                 // [2][64] decay over the chunk
    static constexpr int kBytes = kG + 2 * kN * 4;
};
static_assert(StateLds::kAhead >= 3 && StateLds::kBytes <= 160 * 1024, "LDS of state_kernel");

struct StateArgs {
    int T, H;                    // longest row; heads
    int reverse;                 // the row is read back to front
    RowCut cut;
    const bf16_t *k, *v, *w;
    float *states, *decay;       // [rows][H][64 key][64 value], [rows][H][64] (may be null)
};

// sum over the rows of lanes behind the lane's own (row g: rows g+1 .. 3)
__device__ __forceinline__ float suffix_rows(float x, int g) {
    const uint32_t xi = __float_as_uint(x);
    const u32x2 a = __builtin_amdgcn_permlane16_swap(xi, xi, false, false);   // a[0] = rows (0,0,2,2), a[1] = rows (1,1,3,3)
    const uint32_t si = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
    const u32x2 b = __builtin_amdgcn_permlane32_swap(si, si, false, false);   // b[1] = rows 2+3 everywhere
    return ((g & 1) ? 0.f : __uint_as_float(a[1])) + ((g & 2) ? 0.f : __uint_as_float(b[1]));
}

__global__ __launch_bounds__(512) void state_kernel(StateArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    typedef StateLds L;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, l16 = lane & 15;
    const int pair = (int)blockIdx.x, row = pair / a.H, h = pair - row * a.H;
    const int64_t C = (int64_t)a.H * kN;
    if (a.cut.segments) {
        const RowView rv = row_view(a.cut, row, a.T);
        a.T = rv.tokens;
        move_rows(a.k, rv.shift * C); move_rows(a.v, rv.shift * C); move_rows(a.w, rv.shift * C);
    }
    const int T = a.T, nvisit = (T + kBlockTokens - 1) / kBlockTokens;
    float *tot_l = reinterpret_cast<float *>(smem + L::kTot), *g_l = reinterpret_cast<float *>(smem + L::kG);

    if (wave < 4) {
        // ---------------- loading waves ----------------
        const int p = wave;
        const int64_t base = (int64_t)row * T * C + (int64_t)h * kN;
        const bf16_t *kb = a.k + base, *vb = a.v + base, *wb = a.w + base;
        const uint32_t rowbytes = (uint32_t)C * 2u, lds0 = lds_address(smem);
        const int lrow = lane >> 3;
        const uint32_t lpiece = (uint32_t)(((lane & 7) ^ lrow) << 4);
        auto issue = [&](int it) {   // six loads; rows past the end read the last one
            const uint32_t own = 16 * p * kTileRow;
            const uint32_t kk = lds0 + L::kKW + (it % (L::kAhead - 1)) * 2 * kTileBytes + own, vv = lds0 + L::kV + (it % (L::kAhead + 1)) * kTileBytes + own;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int i = min(it * kBlockTokens + 16 * p + 8 * hf + lrow, T - 1), t = a.reverse ? T - 1 - i : i;
                const uint32_t o = (uint32_t)t * rowbytes + lpiece;
                load_rows8_to_lds(wb, o, kk + kTileBytes + 8 * hf * kTileRow);
                load_rows8_to_lds(kb, o, kk + 8 * hf * kTileRow);
                load_rows8_to_lds(vb, o, vv + 8 * hf * kTileRow);
            }
        };
        // lane (l16, g): channels 4 l16 .. +3 of tokens 16p + 4g .. +3
        float fk[4][4], ew2[4][4], after[4];   // k; exp(w) log2(e); exponents of the wave's later tokens behind the lane's
        float all[4] = {0.f, 0.f, 0.f, 0.f};   // exponents over the row so far
        // k and w of chunk `it` into registers, the sums of its exponents to LDS; `younger`: chunks requested behind it
        auto start = [&](int it, int younger) {
            const unsigned char *kt = smem + L::kKW + (it % (L::kAhead - 1)) * 2 * kTileBytes, *wt = kt + kTileBytes;
            wait_in_flight(6 * younger);
            uint2 qk[4], qw[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t o = tile_off(16 * p + 4 * g + e, 4 * l16);
                qk[e] = *reinterpret_cast<const uint2 *>(kt + o);
                qw[e] = *reinterpret_cast<const uint2 *>(wt + o);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (their tiles may be filled again)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float fw[4];
                unpack4(make_s16x4(qk[e].x, qk[e].y), fk[e]);
                unpack4(make_s16x4(qw[e].x, qw[e].y), fw);
                const bool valid = it * kBlockTokens + 16 * p + 4 * g + e < T;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    ew2[e][c] = valid ? exp2_fast(fmaf(fw[c], kLog2e, kLog2Log2e)) : 0.f;
                    if (!valid) fk[e][c] = 0.f;
                }
            }
            float tot[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float lt = (ew2[0][c] + ew2[1][c]) + (ew2[2][c] + ew2[3][c]);
                tot[c] = sum_rows(lt);
                after[c] = suffix_rows(lt, g);
            }
            if (g == 0) *reinterpret_cast<f32x4 *>(tot_l + ((it & 1) * 4 + p) * kN + 4 * l16) = (f32x4){tot[0], tot[1], tot[2], tot[3]};
        };
        // K^ of the chunk in registers, behind a barrier of all waves' sums
        auto finish = [&](int it) {
            unsigned char *op = smem + L::kOp + (it & 1) * kTileBytes;
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const f32x4 x = *reinterpret_cast<const f32x4 *>(tot_l + ((it & 1) * 4 + w) * kN + 4 * l16);
                sum += x;
                if (w > p) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) after[c] += x[c];
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) all[c] += sum[c];
            if (p == 0 && g == 0)
                *reinterpret_cast<f32x4 *>(g_l + (it & 1) * kN + 4 * l16) = (f32x4){exp2_fast(-sum[0]), exp2_fast(-sum[1]), exp2_fast(-sum[2]), exp2_fast(-sum[3])};
#pragma unroll
            for (int e = 3; e >= 0; --e) {
                float x[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    x[c] = fk[e][c] * exp2_fast(-after[c]);
                    after[c] += ew2[e][c];
                }
                *reinterpret_cast<uint2 *>(op + tile_off(16 * p + 4 * g + e, 4 * l16)) = make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]));
            }
        };
        auto younger = [&](int issued, int it) { return min(issued, nvisit - 1) - it; };   // issued: the last chunk asked for so far
        for (int i = 0; i < min(nvisit, L::kAhead - 1); ++i) issue(i);
        start(0, younger(L::kAhead - 2, 0));
        if (L::kAhead - 1 < nvisit) issue(L::kAhead - 1);
        __syncthreads();
        finish(0);
        if (nvisit > 1) start(1, younger(L::kAhead - 1, 1));
        for (int it = 0; it < nvisit; ++it) {
            __syncthreads();
            // free again: v of chunk it - 1, k and w of chunk it + 1
            if (it + L::kAhead < nvisit) issue(it + L::kAhead);
            if (it + 1 < nvisit) finish(it + 1);
            if (it + 2 < nvisit) start(it + 2, younger(it + L::kAhead, it + 2));
        }
        if (a.decay && p == 0 && g == 0)
            *reinterpret_cast<f32x4 *>(a.decay + (int64_t)pair * kN + 4 * l16) = (f32x4){exp2_fast(-all[0]), exp2_fast(-all[1]), exp2_fast(-all[2]), exp2_fast(-all[3])};
    } else {
        // ---------------- consumer waves ----------------
        const int q = wave - 4;
        f32x4 S[4];   // S[m][rr]: key row block_row_channel(m, g) + rr, value column 16q + l16
#pragma unroll
        for (int m = 0; m < 4; ++m) S[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
        __syncthreads();
        for (int it = 0; it < nvisit; ++it) {
            __syncthreads();
            const unsigned char *kt = smem + L::kOp + (it & 1) * kTileBytes, *vt = smem + L::kV + (it % (L::kAhead + 1)) * kTileBytes;
            const float *gv = g_l + (it & 1) * kN;
#pragma unroll
            for (int m = 0; m < 4; ++m) S[m] *= *reinterpret_cast<const f32x4 *>(gv + block_row_channel(m, g));
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                s16x4 vf[2], kq[2][4];
#pragma unroll
                for (int pp = 0; pp < 2; ++pp) {
                    vf[pp] = tile_frag_tok(vt, 16 * q, 32 * blk + 16 * pp, l16, g);
#pragma unroll
                    for (int m = 0; m < 4; ++m) kq[pp][m] = block_frag_tok_rows(kt, m, 32 * blk + 16 * pp, l16, g);
                }
#pragma unroll
                for (int m = 0; m < 4; ++m) S[m] = mfma32(both16(kq[0][m], kq[1][m]), both16(vf[0], vf[1]), S[m]);
            }
            settle(S[0], S[1], S[2], S[3]);
        }
        float *out = a.states + (int64_t)pair * (kN * kN) + 16 * q + l16;
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) out[(block_row_channel(m, g) + rr) * kN] = S[m][rr];
    }
}

hipError_t segment_states(hipStream_t st, int64_t rows, int64_t L, int64_t H, const void *k, const void *v, const void *w,
                          float *states, float *decay, bool reverse, RowCut cut)
{
    StateArgs a = {};
    a.T = (int)L; a.H = (int)H; a.reverse = reverse; a.cut = cut;
    a.k = (const bf16_t *)k; a.v = (const bf16_t *)v; a.w = (const bf16_t *)w;
    a.states = states; a.decay = decay;
    const hipError_t e = allow_dynamic_lds<state_kernel>(StateLds::kBytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(state_kernel, dim3((unsigned)(rows * H)), dim3(512), StateLds::kBytes, st, a);
    return hipGetLastError();
}

}  // namespace wkv6
