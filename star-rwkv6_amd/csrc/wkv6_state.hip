// What a time segment leaves alone: the state it builds from zero and the decay over it, for gfx950 (bf16 tensors).  The first
// pass over the segments of a sequence, forward (k, v) and, read back to front with r and gy in their place, backward.
//
// Nothing but the state is wanted, so of the tile form (wkv6_chunk_fwd.hip) only its update is left, 16 tokens at a time:
//   S <- diag(g) S + K^^T V ,   K^_s = k_s e^{c_16 - c_{s+1}} ,   g = e^{c_16}     (c: running sum of the log decays in the tile)
// in the tile form's arithmetic and order, so that what a segment hands on has the bits it would have there; and, as there, a row of
// which a tile leaves the range of e^{-c} is redone one timestep at a time, in fp32 (wkv6_scan_body.h).  (64 tokens as one step need
// half as many MFMAs and no range, but round every k of such a row to bf16: the final state of a prompt with one strong decay in
// every 64 tokens was 1.4e-3 from float64, and is 5.5e-8.)
//
// Bound by the reading of k, v and w where the segments fill the chip (B1 T8192 H32: 100 MB), by a launch and the latency of the
// first loads where they are short.  Through the torch flavour, the tile form's kernel without y / 64 tokens as one step / this:
// prompt B1 T1337 H32 19.6 / 17.9 / 18.3 us, training B1 T8192 H32 164 / 159.7 / 162.1.  Rows three and four chunks ahead: 18.6
// and 18.6, 164.6 and 165.3.
// One workgroup per (segment, head): four loading waves (wave p <-> tile p of every chunk, lane = channel) bring the rows straight
// into LDS two chunks ahead and form K^ and g; four consumer waves (q): value columns 16q .. of the state.
#include "wkv6_mfma.h"
#include "wkv6_kernels.h"
#include "wkv6_block.h"
#include "wkv6_scan_body.h"

namespace wkv6 {

struct StateLds {
    static constexpr int kAhead = 2;                                 // chunks between the request of the rows and their use
    static constexpr int kV = 0;                                     // [chunk % (kAhead + 1)] v tiles
    static constexpr int kKW = kV + (kAhead + 1) * kTileBytes;       // [chunk % kAhead][k, w] tiles (done with a chunk before use)
    static constexpr int kOp = kKW + kAhead * 2 * kTileBytes;        // [2] K^
    static constexpr int kG = kOp + 2 * kTileBytes;                  // [2][4 tiles][64] decay over each tile
    static constexpr int kDecay = kG + 2 * 4 * kN * 4;               // [4 waves][64] exponents over each wave's tiles of the row
    static constexpr int kBytes = kDecay + 4 * kN * 4;
};
static_assert(StateLds::kBytes <= 160 * 1024 && sizeof(ScanFwdLds) <= StateLds::kBytes, "LDS of state_kernel");

struct StateArgs {
    int T, H;                    // longest row; heads
    int reverse;                 // the row is read back to front
    RowCut cut;
    const bf16_t *k, *v, *w;
    const bf16_t *u;             // (read by the pass one timestep at a time, for a y that it does not write)
    float *states, *decay;       // [rows][H][64 key][64 value], [rows][H][64] (may be null)
    GivenStates given;
    int P, unused;               // the segments of a sequence, and which of them nobody asks for (P = 0: all are wanted)
};

// kUnused: a segment of every sequence is not wanted (asked at run time, prompts, of which all are, took 0.1 us longer: 18.26 / 18.35)
template <bool kUnused>
__global__ __launch_bounds__(512) void state_kernel(StateArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    typedef StateLds L;
    __shared__ int s_wild;       // a tile of the row left the range
    if (threadIdx.x == 0) s_wild = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pair = (int)blockIdx.x, row = pair / a.H, h = pair - row * a.H;
    const int64_t C = (int64_t)a.H * kN;
    // Without states at the ends of a sequence its last segment (read back to front, its first) hands nothing on: only a decay is left, for
    // the other direction's walk, which begins there from zero.  Half of the reading with two segments, an eighth with eight:
    // forward and backward, all passes run / so: B4 T3000 H32 (two) 236.8 / 224.1 us, B10 T1685 H12 (two) 143.3 / 136.7, B1 T3908 H48 (five) 132.3 / 129.0,
    // eight of B1 T8192 H32 165.8 / 164.7.
    if (kUnused && row % a.P == a.unused) {
        if (a.decay && threadIdx.x < kN) a.decay[(int64_t)pair * kN + threadIdx.x] = 0.f;
        return;
    }
    if (a.cut.segments) {
        const RowView rv = row_view(a.cut, row, a.T);
        a.T = rv.tokens;
        move_rows(a.k, rv.shift * C); move_rows(a.v, rv.shift * C); move_rows(a.w, rv.shift * C);
    }
    const int T = a.T, nvisit = (T + kBlockTokens - 1) / kBlockTokens;
    float *decay_l = reinterpret_cast<float *>(smem + L::kDecay);

    if (wave < 4) {
        // ---------------- loading waves: lane = channel, wave p <-> tile p of every chunk ----------------
        const int p = wave;
        const int64_t base = (int64_t)row * T * C + (int64_t)h * kN;
        const bf16_t *kb = a.k + base, *vb = a.v + base, *wb = a.w + base;
        const uint32_t rowbytes = (uint32_t)C * 2u, lds0 = lds_address(smem);
        const int lrow = lane >> 3;
        const uint32_t lpiece = (uint32_t)(((lane & 7) ^ lrow) << 4);
        auto issue = [&](int it) {   // six loads; rows past the end read the last one
            const uint32_t own = 16 * p * kTileRow;
            const uint32_t kk = lds0 + L::kKW + (it % L::kAhead) * 2 * kTileBytes + own, vv = lds0 + L::kV + (it % (L::kAhead + 1)) * kTileBytes + own;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int i = min(it * kBlockTokens + 16 * p + 8 * hf + lrow, T - 1), t = a.reverse ? T - 1 - i : i;
                const uint32_t o = (uint32_t)t * rowbytes + lpiece;
                load_rows8_to_lds(wb, o, kk + kTileBytes + 8 * hf * kTileRow);
                load_rows8_to_lds(kb, o, kk + 8 * hf * kTileRow);
                load_rows8_to_lds(vb, o, vv + 8 * hf * kTileRow);
            }
        };
        // byte offsets of the lane's channel inside a tile row, for the 8 swizzle phases
        uint32_t choff[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) choff[s] = (uint32_t)((((lane >> 3) ^ s) << 4) + ((lane & 7) << 1)) + (uint32_t)(16 * p * kTileRow);
        float all = 0.f;   // base-2 exponent summed over this wave's tiles
        // K^ and the decay of the wave's tile of chunk `it`; `younger`: chunks requested behind it.  The same arithmetic in the
        // same order as the tile form's (fwd_producer in wkv6_chunk_fwd.hip): the same bits.
        auto prepare = [&](int it, int younger) {
            const unsigned char *kt = smem + L::kKW + (it % L::kAhead) * 2 * kTileBytes, *wt = kt + kTileBytes;
            unsigned char *op = smem + L::kOp + (it & 1) * kTileBytes;
            wait_in_flight(6 * younger);
            float xk[16], fw[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t o = choff[e & 7] + e * kTileRow;
                uint32_t rk = *reinterpret_cast<const uint16_t *>(kt + o), rw = *reinterpret_cast<const uint16_t *>(wt + o);
                if (it * kBlockTokens + 16 * p + e >= T) { rk = 0u; rw = neg_inf_bits<bf16_t>(); }
                xk[e] = bf16_bits_to_float(rk); fw[e] = bf16_bits_to_float(rw);
            }
            float cs2 = 0.f, pa = 1.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float ew2 = exp2_fast(fmaf(fw[e], kLog2e, kLog2Log2e));   // exp(w) log2(e)
                cs2 += ew2;
                xk[e] *= exp2_fast(cs2);   // k exp(+c_{t+1})
                pa *= exp2_fast(-ew2);
            }
#pragma unroll
            for (int e = 0; e < 16; e += 2) {
                const uint32_t x = pack_bf16x2(xk[e] * pa, xk[e + 1] * pa);
                *reinterpret_cast<uint16_t *>(op + choff[e & 7] + e * kTileRow) = (uint16_t)x;
                *reinterpret_cast<uint16_t *>(op + choff[(e + 1) & 7] + (e + 1) * kTileRow) = (uint16_t)(x >> 16);
            }
            if (__builtin_amdgcn_ballot_w64(!(cs2 <= kWildLimit * kLog2e)) != 0ull && lane == 0) s_wild = 1;
            reinterpret_cast<float *>(smem + L::kG)[((it & 1) * 4 + p) * kN + lane] = pa;
            all += cs2;
        };
        auto younger = [&](int issued, int it) { return min(issued, nvisit - 1) - it; };   // issued: the last chunk asked for so far
        for (int i = 0; i < min(nvisit, L::kAhead); ++i) issue(i);
        prepare(0, younger(L::kAhead - 1, 0));
        for (int it = 0; it < nvisit; ++it) {
            __syncthreads();
            // free again: v of chunk it - 1, k and w of chunk it
            if (it + L::kAhead < nvisit) issue(it + L::kAhead);
            if (it + 1 < nvisit) prepare(it + 1, younger(it + L::kAhead, it + 1));
        }
        decay_l[p * kN + lane] = all;
    } else {
        // ---------------- consumer waves ----------------
        const int q = wave - 4, g = lane >> 4, l16 = lane & 15;
        // the given state of a sequence's first segment: 16 of the 4096 elements to a thread, asked for here and left behind the chunks
        const bool give = a.given.states && row % a.given.P == 0;
        const int first = 4 * (64 * q + lane);
        float given[4][4];
        if (give) {
            const int b = row / a.given.P;
            const int64_t from = ((a.given.map ? a.given.map[b] : (int64_t)b) * a.H + h) * (kN * kN) + first;
            if (a.given.bf16) {
#pragma unroll
                for (int i = 0; i < 4; ++i) load4(reinterpret_cast<const bf16_t *>(a.given.states) + from + 1024 * i, given[i]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) load4(reinterpret_cast<const float *>(a.given.states) + from + 1024 * i, given[i]);
            }
        }
        f32x4 S[4];   // S[m][rr]: key row 16m + 4g + rr, value column 16q + l16
#pragma unroll
        for (int m = 0; m < 4; ++m) S[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
        for (int it = 0; it < nvisit; ++it) {
            __syncthreads();
            const unsigned char *kt = smem + L::kOp + (it & 1) * kTileBytes, *vt = smem + L::kV + (it % (L::kAhead + 1)) * kTileBytes;
            const float *gv = reinterpret_cast<const float *>(smem + L::kG) + (it & 1) * 4 * kN;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const s16x4 vf = tile_frag_tok(vt, 16 * q, 16 * p, l16, g);
                s16x4 kf[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) kf[m] = tile_frag_tok(kt, 16 * m, 16 * p, l16, g);
#pragma unroll
                for (int m = 0; m < 4; ++m) S[m] *= *reinterpret_cast<const f32x4 *>(gv + p * kN + 16 * m + 4 * g);
#pragma unroll
                for (int m = 0; m < 4; ++m) S[m] = mfma16(kf[m], vf, S[m]);
                settle(S[0], S[1], S[2], S[3]);
            }
        }
        if (give) {
#pragma unroll
            for (int i = 0; i < 4; ++i) store4(a.given.start + (int64_t)pair * (kN * kN) + first + 1024 * i, given[i][0], given[i][1], given[i][2], given[i][3]);
        }
        if (!s_wild) {   // (complete: the last chunk was prepared before the last barrier)
            float *out = a.states + (int64_t)pair * (kN * kN) + 16 * q + l16;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) out[(16 * m + 4 * g + rr) * kN] = S[m][rr];
        }
    }
    __syncthreads();
    if (a.decay && threadIdx.x < kN) {
        const float *e = decay_l + threadIdx.x;
        a.decay[(int64_t)pair * kN + threadIdx.x] = exp2_fast(-((e[0] + e[kN]) + (e[2 * kN] + e[3 * kN])));
    }
    if (s_wild) {
        __syncthreads();
        scan_fwd_body<bf16_t, bf16_t, float>(*reinterpret_cast<ScanFwdLds *>(smem), row, h, T, a.H, a.k, a.k, a.v, a.w, a.u, nullptr, nullptr,
                                             nullptr, a.states, a.reverse != 0);
    }
}

hipError_t segment_states(hipStream_t st, int64_t rows, int64_t L, int64_t H, const void *k, const void *v, const void *w, const void *u,
                          float *states, float *decay, bool reverse, RowCut cut, const GivenStates &given, int P)
{
    StateArgs a = {};
    a.T = (int)L; a.H = (int)H; a.reverse = reverse; a.cut = cut;
    a.k = (const bf16_t *)k; a.v = (const bf16_t *)v; a.w = (const bf16_t *)w; a.u = (const bf16_t *)u;
    a.states = states; a.decay = decay; a.given = given;
    a.P = P; a.unused = reverse ? 0 : P - 1;
    if (P && given.states) return hipErrorInvalidValue;   // (the workgroups of the first segments pass them on)
    auto launch = [&](auto kernel, hipError_t e) -> hipError_t {
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, dim3((unsigned)(rows * H)), dim3(512), StateLds::kBytes, st, a);
        return hipGetLastError();
    };
    return P ? launch(state_kernel<true>, allow_dynamic_lds<state_kernel<true>>(StateLds::kBytes))
             : launch(state_kernel<false>, allow_dynamic_lds<state_kernel<false>>(StateLds::kBytes));
}

}  // namespace wkv6
