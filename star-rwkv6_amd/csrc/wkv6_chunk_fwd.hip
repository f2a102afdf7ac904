// WKV6 in chunk-parallel form for gfx950: bf16 MFMA for the dense products, fp32 state.
//
// One workgroup (12 waves) per (batch, head) pair, or -- with more pairs than compute units -- one
// workgroup per compute unit that runs its pairs back to back through the same pipeline.  Time is
// cut into chunks of 64 tokens, each chunk into 4 tiles of 16 tokens.  The fp32 state S[j][i] lives in the MFMA accumulators of the
// "consumer" waves (wave q of a group owns value columns 16q..16q+15) and is advanced one tile at a time:
//
//   c_t = sum_{s<t} exp(w_s) inside the tile (so exp(-c_t) is the decay from the tile start to t)
//   R~[t][j] = r_t[j] exp(-c_t[j])            K~[t][j] = k_t[j] exp(+c_{t+1}[j])
//   g[j] = exp(-c_16[j])
//   A[t][s]  = R~_t . K~_s  (s < t),  A[t][t] = sum_j r_t[j] u[j] k_t[j]
//   Y        = R~ S + A V          (16x64x64 and 16x16x16 MFMA, K index j resp. s)
//   S       <- diag(g) (S + K~^T V)   (64x16x16 MFMA, K index s)
//
// Data path.  The raw r, k, w, v rows of a chunk go from global memory straight into LDS tiles
// (16-byte pieces, no registers), two chunks ahead of their use.  The four "producer" waves (one per
// tile, lane = channel) read r, k, w from there, compute R~, K~, g and the diagonal
// in fp32 for the NEXT chunk and write them back as bf16 tiles while the consumers run the MFMAs of
// the current one; the consumers (two groups of four waves that both carry the state but share out
// the per-tile output work) take V directly from its raw tile.  Every tile is stored once,
// [token][channel]; fragments with the k-slots along the tokens come from the transposing LDS read.
// The two roles meet at one barrier per chunk.  HBM traffic is exactly the algorithmic minimum
// (r,k,v,w read once, y written once).
//
// exp(+c) needs the decay accumulated inside one 16-token tile to stay in range.  A producer wave
// that meets a tile whose summed exp(w) exceeds kWildLimit in any channel raises a flag in LDS, and
// the workgroup then redoes ITS (batch, head) pair with the exact per-timestep code
// (wkv6_scan_body.h) before the kernel ends; other workgroups are unaffected.
#include "wkv6_mfma.h"
#include "wkv6_kernels.h"
#include "wkv6_scan_body.h"

#include <type_traits>

namespace wkv6 {

constexpr int CL = 64;   // tokens per chunk

// LDS map of the forward kernel (byte offsets into the dynamic block)
struct FwdLds {
    static constexpr int kRawRKW = 0;                                   // [2 chunk parities][r,k,w] raw tiles
    static constexpr int kRawV = kRawRKW + 2 * 3 * kTileBytes;          // [3] raw v tiles (chunk % 3)
    static constexpr int kOp = kRawV + 3 * kTileBytes;                  // [2] operand blocks
    static constexpr int kOpRt = 0, kOpKt = kTileBytes, kOpG = 2 * kTileBytes, kOpRuk = kOpG + 4 * kN * 4;
    static constexpr int kOpBytes = kOpRuk + CL * 4;
    static constexpr int kBytes0 = kOp + 2 * kOpBytes;
    // only WITHOUT the fused output stage: [2] K^ = K~ g, k decayed to the END of its tile (exponents <= 0)
    static constexpr int kKg = kBytes0;
    static constexpr int kDecay = kKg + 2 * kTileBytes;                 // [4 tiles][64] floats: see FwdArgs::decay
    static constexpr int kBytes = kDecay + 4 * kN * 4;
    // only with the fused output stage (group norm and gate):
    static constexpr int kYStage = kBytes0;                             // [2 visit parities] y of one chunk, bf16
    static constexpr int kRawG = kYStage + 2 * kTileBytes;              // [4] raw gate tiles (visit & 3)
    static constexpr int kGnTab = kRawG + 4 * kTileBytes;               // [4][scale, offset][64] floats of the visit's head
    static constexpr int kBytesFused = kGnTab + 4 * 2 * kN * 4;
};

// With the fused output stage y does not go to global memory: the consumers leave each chunk in LDS
// as [token][64 channels] rows of 128 bytes, and a producer wave reads whole rows (lane = channel)
// one visit later.  The 32-byte slot of a consumer wave's 16 channels is XORed with bits 2..3 of the
// token, so that the four token rows one accumulator store touches fall into different banks.
__device__ __forceinline__ uint32_t ystage_off(int t, int ch) {
    return ((uint32_t)t << 7) + (((((uint32_t)ch >> 4) ^ ((uint32_t)t >> 2)) & 3u) << 5) + (((uint32_t)ch & 15u) << 1);
}

// Wave layout: 12 waves, four per role, one wave of each role per SIMD:
//   loader/producer (wave p <-> tile p) | consumer group 0 (y of tiles 0, 2) | consumer group 1 (tiles 1, 3)
constexpr int kFwdThreads = 12 * 64;

struct FwdArgs {
    int T, H;
    int nitems;      // B * H (batch, head) pairs; with kMulti a workgroup takes every gridDim.x-th of them
    int split;       // 1, 2 or 4 workgroups per pair, each with the consumer waves of 4 / split column slices
    int reverse;     // 1: the time axis is read back to front (row T-1-t in the place of row t)
    int slice;       // chunks of a pair's slice of `ckpt` (those of the longest row)
    RowCut cut;      // rows that are time segments (one pair per workgroup and kRagged)
    float *decay;    // null, or [pairs][64]: per pair exp(-sum of exp(w) over its tokens) (one pair per workgroup, no output stage)
    const bf16_t *r, *k, *v, *w, *u;   // 16-bit elements: bf16, or fp16 with v a bf16 copy (see OutOf)
    const void *v_orig;                // v as the caller holds it (the exact per-timestep pass reads this one)
    const void *s0;
    const int64_t *map;
    bf16_t *y;
    void *sT;
    float *ckpt;
    int *arrivals;   // with ckpt: per-head counters the backward's fused gu sum starts from zero
    // fused output stage: out = (group_norm_head(y) * gn_scale + gn_offset) * gate, y itself is not written
    const bf16_t *gate;
    const float *gn_scale, *gn_offset;   // (H, 64)
    float gn_eps;
    bf16_t *out;
    // training with the fused output stage (then y above is written as well, for the norm's backward):
    float *stats;    // null, or (B, T, H, 2) fp32: mean and 1/sqrt(var + eps) of y over each head's channels
    GnSums sums;
};

// ------------------------------------------------------------------------------------------
// Consumer group GRP of two: both groups carry the state through every tile (4 MFMAs and a
// scaling), group 0 produces y for tiles 0 and 2, group 1 for tiles 1 and 3.
// ------------------------------------------------------------------------------------------
template <typename Tin, typename Ts, bool kSave, bool kRagged, bool kMulti, bool kFuse, int GRP>
__device__ __forceinline__ void fwd_consumer(const FwdArgs &a, const unsigned char *smem, const int *s_wild, int bh0, int q, int lane)
{
    const int T = a.T, H = a.H;
    const int g = lane >> 4, l16 = lane & 15;
    const int64_t C = (int64_t)H * kN;
    const int nchunk = (T + CL - 1) / CL;
    const int stride = (int)gridDim.x;
    const int n_my = kMulti ? (a.nitems - bh0 + stride - 1) / stride : 1;
    const Ts *s0 = reinterpret_cast<const Ts *>(a.s0);
    // initial state of a (batch, head) pair as stored (converted when the pair starts)
    Ts Sraw[16];
    auto request_state = [&](int bh) {
        const int b = bh / H, h = bh - b * H;
        const int64_t row = a.map ? a.map[b] : (int64_t)b;
        const Ts *p = s0 + (row * H + h) * kN * kN + 16 * q + l16;
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) Sraw[4 * m + rr] = p[(16 * m + 4 * g + rr) * kN];
    };
    if (s0 != nullptr) request_state(bh0);
    int it = 0;   // chunk visits of this workgroup so far: picks the LDS buffers
    for (int n = 0, bh = bh0; n < n_my; ++n, bh += stride) {
        const int b = bh / H, h = bh - b * H;
        const int64_t base = (int64_t)b * T * C + (int64_t)h * kN;
        f32x4 S[4];
        if (s0 != nullptr) {
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) S[m][rr] = (float)Sraw[4 * m + rr];
        } else {
#pragma unroll
            for (int m = 0; m < 4; ++m) S[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
        typedef typename OutOf<Tin>::type Tout;
        Tout *y_h = reinterpret_cast<Tout *>(a.y) + base;
        if (kSave && GRP == 0 && b == 0 && q == 0 && lane == 0 && a.arrivals) a.arrivals[h] = 0;
        if (kSave && kFuse && GRP == 0 && b == 0 && q == 0) clear_sums(a.sums, h, lane);
        for (int c = 0; c < nchunk; ++c, ++it) {
            __syncthreads();
            if (kSave && GRP == 0) {
                // The state at the chunk start goes to the workspace transposed, bf16 [chunk][i][j] in the
                // first half of this pair's slice: a lane's four rows j = 16m + 4g .. +3 of its column i are
                // eight contiguous bytes there, so a chunk takes four stores per lane.  They are issued behind
                // the barrier (the state registers do not change before the end of tile 0) and queue while
                // the other waves already work on the chunk.
                char *dst = reinterpret_cast<char *>(a.ckpt + (int64_t)bh * a.slice * (kN * kN)) + (int64_t)c * (kN * kN * 2) + (16 * q + l16) * (kN * 2) + 8 * g;
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    *reinterpret_cast<uint2 *>(dst + 32 * m) = make_uint2(pack_bf16x2(S[m][0], S[m][1]), pack_bf16x2(S[m][2], S[m][3]));
            }
            // the next pair's initial state is requested one chunk visit ahead of its use
            if (kMulti && s0 != nullptr && c == nchunk - 1 && n + 1 < n_my) request_state(bh + stride);
            // Tokens past the end were prepared as r = k = 0, decay 1: their tiles leave the state alone,
            // and their y rows are not stored.
            int op_off = FwdLds::kOp + (it & 1) * FwdLds::kOpBytes, v_off = FwdLds::kRawV + (it % 3) * kTileBytes;
            const int t0 = c * CL;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                // (fresh_s: form the tile addresses per tile instead of holding them all across the chunk)
                const unsigned char *rt = smem + op_off + FwdLds::kOpRt, *kt = smem + op_off + FwdLds::kOpKt;
                const float *gv_ = reinterpret_cast<const float *>(smem + op_off + FwdLds::kOpG);
                const float *ruk = reinterpret_cast<const float *>(smem + op_off + FwdLds::kOpRuk);
                const unsigned char *vt = smem + v_off;
                const s16x4 vf = tile_frag_tok(vt, 16 * q, 16 * p, l16, g);
                const bool minep = (p & 1) == GRP && (kFuse || a.y != nullptr);   // (no y wanted: a pass that only builds the state)
                f32x4 U[4];
                bf16x8 sop0, sop1;
                if (minep) { sop0 = acc_as_operand(S[0], S[1]); sop1 = acc_as_operand(S[2], S[3]); }
                if (kFuse) {
                    // U = K~^T V in accumulators of its own, added to the state by VALU code at the end of the tile
#pragma unroll
                    for (int m = 0; m < 4; ++m) U[m] = mfma16(tile_frag_tok(kt, 16 * m, 16 * p, l16, g), vf, (f32x4){0.f, 0.f, 0.f, 0.f});
                } else {
                    // S <- diag(g) S + K^^T V: the new contributions' decay is folded into the operand, so the
                    // update is one scaling and an MFMA accumulation onto the state itself
                    const unsigned char *kgt = smem + FwdLds::kKg + (it & 1) * kTileBytes;
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const float4 gg = *reinterpret_cast<const float4 *>(&gv_[p * kN + 16 * m + 4 * g]);
                        S[m][0] *= gg.x; S[m][1] *= gg.y; S[m][2] *= gg.z; S[m][3] *= gg.w;
                    }
#pragma unroll
                    for (int m = 0; m < 4; ++m) S[m] = mfma16(tile_frag_tok(kgt, 16 * m, 16 * p, l16, g), vf, S[m]);
                }
                if (minep) {
                    const int row = 16 * p + l16;
                    const bf16x8 rf0 = tile_frag_ch(rt, row, 0, g), rf1 = tile_frag_ch(rt, row, 1, g);
                    const bf16x8 kf0 = tile_frag_ch(kt, row, 0, g), kf1 = tile_frag_ch(kt, row, 1, g);
                    const float rukv = ruk[row];
                    // A^T[s][t] = K~_s . R~_t  (accumulator rows s = 4g+r, column t = l16)
                    f32x4 AT = {0.f, 0.f, 0.f, 0.f};
                    AT = mfma32(kf0, rf0, AT);
                    AT = mfma32(kf1, rf1, AT);
                    // Y = R~ S
                    // Without the fused output stage the products are formed transposed (the operands change
                    // places): accumulator rows i = 4g + r, column t = l16, so that a lane holds four
                    // neighbouring channels of one token and writes them with one 8-byte store.
                    f32x4 Y = {0.f, 0.f, 0.f, 0.f};
                    if (kFuse) {
                        Y = mfma32(rf0, sop0, Y);
                        Y = mfma32(rf1, sop1, Y);
                    } else {
                        Y = mfma32(sop0, rf0, Y);
                        Y = mfma32(sop1, rf1, Y);
                    }
                    settle(AT);
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const int s = 4 * g + rr;
                        AT[rr] = (l16 > s) ? AT[rr] : ((l16 == s) ? rukv : 0.f);
                    }
                    // Y += A V : the masked A^T accumulator IS the operand holding A (token t = l16, k-slots s = 4g+r)
                    chain_gap(Y);
                    const s16x4 aop = make_s16x4(pack_bf16x2(AT[0], AT[1]), pack_bf16x2(AT[2], AT[3]));
                    Y = kFuse ? mfma16(aop, vf, Y) : mfma16(vf, aop, Y);
                    settle(Y);
                    if (kFuse) {
                        unsigned char *ys = const_cast<unsigned char *>(smem) + FwdLds::kYStage + (it & 1) * kTileBytes;
                        const uint32_t y01 = pack_bf16x2(Y[0], Y[1]), y23 = pack_bf16x2(Y[2], Y[3]);
                        const int tk = 16 * p + 4 * g, chn = 16 * q + l16;
                        *reinterpret_cast<uint16_t *>(ys + ystage_off(tk, chn)) = (uint16_t)y01;
                        *reinterpret_cast<uint16_t *>(ys + ystage_off(tk + 1, chn)) = (uint16_t)(y01 >> 16);
                        *reinterpret_cast<uint16_t *>(ys + ystage_off(tk + 2, chn)) = (uint16_t)y23;
                        *reinterpret_cast<uint16_t *>(ys + ystage_off(tk + 3, chn)) = (uint16_t)(y23 >> 16);
                    } else {
                        const int t = t0 + 16 * p + l16;   // channels 16q + 4g .. +3 of this token
                        if (!kRagged || t < T) store4(y_h + ((uint32_t)t * (uint32_t)C + (uint32_t)(16 * q + 4 * g)), Y[0], Y[1], Y[2], Y[3]);
                    }
                }
                if (kFuse) {
                    // S <- diag(g) (S + U)
                    settle(U[0], U[1], U[2], U[3]);
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const float4 gg = *reinterpret_cast<const float4 *>(&gv_[p * kN + 16 * m + 4 * g]);
                        S[m][0] = (S[m][0] + U[m][0]) * gg.x; S[m][1] = (S[m][1] + U[m][1]) * gg.y;
                        S[m][2] = (S[m][2] + U[m][2]) * gg.z; S[m][3] = (S[m][3] + U[m][3]) * gg.w;
                    }
                } else {
                    settle(S[0], S[1], S[2], S[3]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // (not of a pair that is redone: its initial state, which may lie in the same place, is still needed; the flag is complete, the
        // pair's last chunk was prepared in front of its barrier)
        if (a.sT != nullptr && GRP == 0 && !s_wild[n]) {
            Ts *p = reinterpret_cast<Ts *>(a.sT) + (int64_t)bh * kN * kN + 16 * q + l16;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) store1(p + (16 * m + 4 * g + rr) * kN, S[m][rr]);
        }
    }
    if (kFuse) __syncthreads();   // the producers finish the last visit's output behind this one
}

// ------------------------------------------------------------------------------------------
// Loader / producer, lane = channel: wave p <-> tile p of every chunk.
// ------------------------------------------------------------------------------------------
// kNoR: a pass that only builds states (no y wanted): r is neither loaded nor prepared
template <typename Tin, bool kSave, bool kRagged, bool kMulti, bool kFuse, bool kNoR>
__device__ __forceinline__ void fwd_producer(const FwdArgs &a, unsigned char *smem, int *s_wild, int bh0, int part, int pw, int lane)
{
    constexpr int NT = 16;   // tokens per wave and chunk
    const int T = a.T, H = a.H;
    const int p = pw;
    const int ch = lane;
    const int64_t C = (int64_t)H * kN;
    const int nchunk = (T + CL - 1) / CL;
    const int stride = (int)gridDim.x;
    const int n_my = kMulti ? (a.nitems - bh0 + stride - 1) / stride : 1;
    const int nvisit = n_my * nchunk;   // chunk visits of this workgroup, pair after pair
    const uint32_t rowbytes = (uint32_t)C * 2u;
    const uint32_t lds0 = lds_address(smem);
    // this lane's part of an 8-row block load: row (lane >> 3), 16-byte piece swizzled with the row
    const int lrow = lane >> 3;
    const uint32_t lpiece = (uint32_t)(((lane & 7) ^ lrow) << 4);
    // The load stream and the preparation stream each walk the visits in order; `ld_*` / `pp_*` are
    // the (pair, chunk) the next load / preparation belongs to.
    int ld_c = 0, ld_bh = bh0, ld_h = 0;
    const bf16_t *rb, *kb_, *vb, *wb, *gb = nullptr;   // uniform: this pair's first row (gb: gate, fused output stage)
    auto point_loads = [&]() {
        const int b = ld_bh / H, h = ld_bh - b * H;
        ld_h = h;
        const int64_t base = (int64_t)b * T * C + (int64_t)h * kN;
        rb = a.r + base; kb_ = a.k + base; vb = a.v + base; wb = a.w + base;
        if (kFuse) gb = a.gate + base;
    };
    point_loads();
    // Rows past the end of the sequence are fetched from its last row (valid memory); the operand
    // preparation turns them into r = k = 0, w = -inf (decay 1), and the v rows only ever meet zero
    // operands.  Each wave loads what it reads itself, so its own vmcnt covers its inputs; v is
    // picked up by the consumers a barrier later.
    constexpr int kLoads = 8 + (kFuse ? 2 : 0) - (kNoR ? 2 : 0);   // per chunk and wave
    constexpr int kLoads0 = kLoads + (kFuse ? 2 : 0);                  // wave 0 also brings the norm's scale and offset
    auto issue_loads = [&](int it) {   // visit `it` = the load stream's current (pair, chunk)
        const int tb = ld_c * CL + 16 * p;
        const uint32_t rkw = lds0 + FwdLds::kRawRKW + (it & 1) * 3 * kTileBytes + 16 * p * kTileRow;
        const uint32_t vv = lds0 + FwdLds::kRawV + (it % 3) * kTileBytes + 16 * p * kTileRow;
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const int t = tb + 8 * blk + lrow;
            // (back to front only where no y is wanted: asked by every load of the others, it cost a ragged prompt 4 to 8 %)
            const uint32_t o = (uint32_t)(kNoR && a.reverse ? (kRagged ? max(T - 1 - t, 0) : T - 1 - t) : kRagged ? min(t, T - 1) : t) * rowbytes + lpiece;
            load_rows8_to_lds(wb, o, rkw + 2 * kTileBytes + 8 * blk * kTileRow);
            if (!kNoR) load_rows8_to_lds(rb, o, rkw + 8 * blk * kTileRow);
            load_rows8_to_lds(kb_, o, rkw + kTileBytes + 8 * blk * kTileRow);
            load_rows8_to_lds(vb, o, vv + 8 * blk * kTileRow);
            if (kFuse) load_rows8_to_lds(gb, o, lds0 + FwdLds::kRawG + (it & 3) * kTileBytes + (16 * p + 8 * blk) * kTileRow);
        }
        if (kFuse && pw == 0 && lane < 16) {
            // scale and offset of this visit's head (64 floats each), read by all four waves' output stage
            const uint32_t tab = lds0 + FwdLds::kGnTab + (it & 3) * (2 * kN * 4);
            load_rows8_to_lds(a.gn_scale + ld_h * kN, (uint32_t)lane * 16u, tab);
            load_rows8_to_lds(a.gn_offset + ld_h * kN, (uint32_t)lane * 16u, tab + kN * 4);
        }
        if (++ld_c == nchunk && kMulti) { ld_c = 0; ld_bh += stride; if (ld_bh < a.nitems) point_loads(); }
    };
    // waits until at most `stores` + this wave's loads of one visit are in flight
    auto wait_visit_loads = [&](bool next_in_flight, bool stores_behind) {
        if (next_in_flight) {
            if (stores_behind) { if (pw == 0) wait_loads<kLoads0 + 16>(); else wait_loads<kLoads + 16>(); }
            else { if (pw == 0) wait_loads<kLoads0>(); else wait_loads<kLoads>(); }
        } else {
            if (stores_behind) wait_loads<16>(); else wait_loads<0>();
        }
    };
    // per-lane byte offsets of channel `ch` inside a tile row, for the 8 swizzle phases
    uint32_t choff[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) choff[s] = (uint32_t)((((ch >> 3) ^ s) << 4) + ((ch & 7) << 1)) + (uint32_t)(16 * p * kTileRow);
    // Fused output stage for the chunk the consumers staged during the previous visit; wave p takes
    // tile p, lane = channel:  out = ((y - mean) * rstd * gn_scale + gn_offset) * gate, mean and
    // variance over the head's 64 channels of a token (two passes, like a layer norm).
    int fl_c = 0, fl_bh = bh0;
    bf16_t *ob = nullptr, *yb = nullptr;
    float *sb = nullptr;
    constexpr bool train = kFuse && kSave;   // training: y and the norm's statistics are written too
    auto point_output = [&]() {
        const int b = fl_bh / H, h = fl_bh - b * H;
        ob = a.out + (int64_t)b * T * C + (int64_t)h * kN;
        if (train) { yb = a.y + (int64_t)b * T * C + (int64_t)h * kN; sb = a.stats + ((int64_t)b * T * H + h) * 2; }
    };
    if (kFuse) point_output();
    auto output_stage = [&](int it) {   // visit `it` = the output stream's current (pair, chunk)
        const unsigned char *ys = smem + FwdLds::kYStage + (it & 1) * kTileBytes;
        const unsigned char *gt = smem + FwdLds::kRawG + (it & 3) * kTileBytes;
        const float *tab = reinterpret_cast<const float *>(smem + FwdLds::kGnTab + (it & 3) * (2 * kN * 4));
        const float gsc = tab[ch], gof = tab[kN + ch];
        float yv[16], dv[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t bits = *reinterpret_cast<const uint16_t *>(ys + ystage_off(16 * p + e, ch));
            yv[e] = bf16_bits_to_float(bits);
            const int t = fl_c * CL + 16 * p + e;
            if (train && (!kRagged || t < T)) *reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(yb) + ((uint32_t)t * rowbytes + 2u * (uint32_t)ch)) = (uint16_t)bits;
        }
        // lane l of the reduction holds the total of token (l >> 2) & 15
        const float mu_own = transpose_reduce16(yv, lane) * (1.f / kN);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float mu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mu_own), 4 * e));
            yv[e] -= mu;
            dv[e] = yv[e] * yv[e];
        }
        const float rstd_own = __builtin_amdgcn_rsqf(transpose_reduce16(dv, lane) * (1.f / kN) + a.gn_eps);
        if (train && (lane & 3) == 0) {
            const int t = fl_c * CL + 16 * p + ((lane >> 2) & 15);
            if (!kRagged || t < T) *reinterpret_cast<float2 *>(sb + (int64_t)t * H * 2) = make_float2(mu_own, rstd_own);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float rstd = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(rstd_own), 4 * e));
            const float gate = bf16_bits_to_float(*reinterpret_cast<const uint16_t *>(gt + choff[e & 7] + e * kTileRow));
            const int t = fl_c * CL + 16 * p + e;
            const float o = fmaf(yv[e] * rstd, gsc, gof) * gate;
            if (!kRagged || t < T) st16(ob, (uint32_t)t * rowbytes + 2u * (uint32_t)ch, o);
        }
        if (++fl_c == nchunk && kMulti) { fl_c = 0; fl_bh += stride; if (fl_bh < a.nitems) point_output(); }
    };
    int pp_c = 0, pp_n = 0, pp_h = bh0 % H;
    float uc = load1(reinterpret_cast<const Tin *>(a.u) + pp_h * kN + ch);
    float dacc = 0.f;   // base-2 decay exponent summed over this wave's tiles of the current pair
    const float kLog2Log2e = 0.5287663729448977f;   // log2(log2(e)): exp(w) log2(e) = 2^(w log2(e) + this)
    auto prepare = [&](int it) {   // visit `it` = the preparation stream's current (pair, chunk)
        const unsigned char *raw = smem + FwdLds::kRawRKW + (it & 1) * 3 * kTileBytes;
        unsigned char *op = smem + FwdLds::kOp + (it & 1) * FwdLds::kOpBytes;
        const int tb = pp_c * CL + 16 * p;
        // exponents are kept in base 2 (one v_exp_f32 each, no extra scaling multiply)
        float cs2 = 0.f, pa = 1.f;
        float fr[NT], fk[NT], fw[NT];
#pragma unroll
        for (int e = 0; e < NT; ++e) {
            const uint32_t o = choff[e & 7] + e * kTileRow;
            uint32_t ra = kNoR ? 0u : *reinterpret_cast<const uint16_t *>(raw + o);
            uint32_t rk = *reinterpret_cast<const uint16_t *>(raw + kTileBytes + o);
            uint32_t rw = *reinterpret_cast<const uint16_t *>(raw + 2 * kTileBytes + o);
            if (kRagged && tb + e >= T) { ra = 0u; rk = 0u; rw = neg_inf_bits<Tin>(); }
            fr[e] = in_bits_to_float<Tin>(ra); fk[e] = in_bits_to_float<Tin>(rk); fw[e] = in_bits_to_float<Tin>(rw);
        }
        float xr[NT], xk[NT], pr[NT];
#pragma unroll
        for (int e = 0; e < NT; ++e) {
            const float ew2 = exp2_fast(fmaf(fw[e], kLog2e, kLog2Log2e));   // exp(w) * log2(e)
            xr[e] = fr[e] * pa;               // r exp(-c_t)
            cs2 += ew2;
            xk[e] = fk[e] * exp2_fast(cs2);   // k exp(+c_{t+1})
            pa *= exp2_fast(-ew2);
            pr[e] = fr[e] * uc * fk[e];
        }
#pragma unroll
        for (int e = 0; e < NT; e += 2) {
            const uint32_t pr2 = pack_bf16x2(xr[e], xr[e + 1]), pk2 = pack_bf16x2(xk[e], xk[e + 1]);
            const uint32_t o0 = choff[e & 7] + e * kTileRow, o1 = choff[(e + 1) & 7] + (e + 1) * kTileRow;
            if (!kNoR) {
                *reinterpret_cast<uint16_t *>(op + FwdLds::kOpRt + o0) = (uint16_t)pr2;
                *reinterpret_cast<uint16_t *>(op + FwdLds::kOpRt + o1) = (uint16_t)(pr2 >> 16);
            }
            *reinterpret_cast<uint16_t *>(op + FwdLds::kOpKt + o0) = (uint16_t)pk2;
            *reinterpret_cast<uint16_t *>(op + FwdLds::kOpKt + o1) = (uint16_t)(pk2 >> 16);
        }
        if (!kFuse) {
            // K^ = K~ g = k exp(-(c_16 - c_{t+1})): the state update's operand
            unsigned char *kg = smem + FwdLds::kKg + (it & 1) * kTileBytes;
#pragma unroll
            for (int e = 0; e < NT; e += 2) {
                const uint32_t pg2 = pack_bf16x2(xk[e] * pa, xk[e + 1] * pa);
                const uint32_t o0 = choff[e & 7] + e * kTileRow, o1 = choff[(e + 1) & 7] + (e + 1) * kTileRow;
                *reinterpret_cast<uint16_t *>(kg + o0) = (uint16_t)pg2;
                *reinterpret_cast<uint16_t *>(kg + o1) = (uint16_t)(pg2 >> 16);
            }
        }
        // the whole tile's decay: g, and the range check of exp(+c)
        if (__builtin_amdgcn_ballot_w64(!(cs2 <= kWildLimit * kLog2e)) != 0ull) {
            if (lane == 0) s_wild[pp_n] = 1;
        }
        dacc += cs2;
        reinterpret_cast<float *>(op + FwdLds::kOpG)[p * kN + ch] = pa;
        if (!kNoR) {
            const float tot = transpose_reduce16(pr, lane);
            if ((lane & 3) == 0) reinterpret_cast<float *>(op + FwdLds::kOpRuk)[16 * p + ((lane >> 2) & 15)] = tot;
        }
        if (!kMulti && !kFuse && pp_c + 1 == nchunk)   // the exponent of the pair's decay, this wave's tiles
            reinterpret_cast<float *>(smem + FwdLds::kDecay)[p * kN + ch] = dacc;
        if (++pp_c == nchunk && kMulti) {   // the next preparation opens the next pair: its head's u
            pp_c = 0; ++pp_n;
            if (pp_n < n_my) {
                pp_h = (bh0 + pp_n * stride) % H;
                uc = load1(reinterpret_cast<const Tin *>(a.u) + pp_h * kN + ch);
            }
        }
    };
    // visit `it` is loaded during visit it-2 (or the prologue), prepared during visit it-1
    issue_loads(0);
    if (nvisit > 1) issue_loads(1);
    wait_visit_loads(nvisit > 1, false);
    prepare(0);
    for (int it = 0; it < nvisit; ++it) {
        __syncthreads();
        // the raw r, k, w block of visit `it` (read by this wave's prepare(it) before the barrier) and the
        // raw v block of visit it-1 (read by the consumers before the barrier) are free again.
        // The output stage's 16 stores go out behind the loads and are not waited for: a wave's
        // memory operations complete in program order, and the loads waited for below are older
        // than both.  (With a ragged end the number of store instructions issued is not fixed;
        // they go first then and are waited for with the loads.)
        const bool outputs = kFuse && it > 0;
        const bool stores_first = kRagged || train;   // (training writes y and the statistics too: not the fixed 16 stores)
        if (outputs && stores_first) output_stage(it - 1);
        if (it + 2 < nvisit) issue_loads(it + 2);
        if (outputs && !stores_first) output_stage(it - 1);
        if (it + 1 < nvisit) {
            wait_visit_loads(it + 2 < nvisit, outputs && !stores_first);
            prepare(it + 1);
        }
    }
    if (kFuse) {
        __syncthreads();
        output_stage(nvisit - 1);
    }
    wait_loads<0>();
}

// kMulti: more (batch, head) pairs than workgroups -- each workgroup takes every gridDim.x-th pair and
// runs them back to back through one pipeline, so the loads of a pair's first chunks overlap the
// previous pair's last ones (a workgroup fills the CU's LDS, so nothing else would hide them).
constexpr int kMaxPairsPerWorkgroup = 32;
// The exact second pass leaves y in `out`; this turns one pair's rows into the fused output in place
// (a wave per token, lane = channel).
__device__ __forceinline__ void output_stage_in_place(const FwdArgs &a, int bh) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
    const int b = bh / a.H, h = bh - b * a.H;
    const int64_t C = (int64_t)a.H * kN;
    bf16_t *rowp = a.out + (int64_t)b * a.T * C + (int64_t)h * kN + lane;
    const bf16_t *gp = a.gate + (int64_t)b * a.T * C + (int64_t)h * kN + lane;
    const float gsc = a.gn_scale[h * kN + lane], gof = a.gn_offset[h * kN + lane];
    for (int t = wave; t < a.T; t += nwave) {
        const float y = load1(rowp + (int64_t)t * C);
        if (a.y) store1(a.y + (int64_t)b * a.T * C + (int64_t)h * kN + lane + (int64_t)t * C, y);
        float sum = y;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m);
        const float d = y - sum * (1.f / kN);
        float sq = d * d;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) sq += __shfl_xor(sq, m);
        const float rstd = __builtin_amdgcn_rsqf(sq * (1.f / kN) + a.gn_eps);
        if (a.stats && lane == 0) *reinterpret_cast<float2 *>(a.stats + (((int64_t)b * a.T + t) * a.H + h) * 2) = make_float2(sum * (1.f / kN), rstd);
        store1(rowp + (int64_t)t * C, fmaf(d * rstd, gsc, gof) * load1(gp + (int64_t)t * C));
    }
}

template <typename Tin, typename Ts, bool kSave, bool kRagged, bool kMulti, bool kFuse, bool kNoR = false>
__global__ __launch_bounds__(kFwdThreads) void chunk_fwd_kernel(FwdArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_wild[kMaxPairsPerWorkgroup];
    static_assert(sizeof(ScanFwdLds) <= FwdLds::kBytes, "the exact second pass reuses the LDS block");
    if (threadIdx.x < kMaxPairsPerWorkgroup) s_wild[threadIdx.x] = 0;
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // With fewer pairs than compute units a pair is shared by `split` workgroups: the value columns of
    // the state are independent of each other, so each workgroup carries the consumer waves of its
    // 4 / split column slices (and repeats the operand preparation, which does not depend on them).
    const int split = kMulti || kFuse ? 1 : a.split;
    const int bh0 = (int)blockIdx.x / split, part = (int)blockIdx.x - bh0 * split;
    const int nq = 4 / split;   // consumer waves per group
    if (kRagged && !kMulti && a.cut.segments) {
        const RowView rv = row_view(a.cut, bh0 / a.H, a.T);
        const int64_t n = rv.shift * a.H * kN;
        a.T = rv.tokens;
        move_rows(a.r, n); move_rows(a.k, n); move_rows(a.v, n); move_rows(a.w, n);
        a.v_orig = reinterpret_cast<const Tin *>(a.v_orig) + n;
        if (a.y) a.y = reinterpret_cast<bf16_t *>(reinterpret_cast<typename OutOf<Tin>::type *>(a.y) + n);
        if (kFuse) { move_rows(a.gate, n); move_rows(a.out, n); move_rows(a.stats, rv.shift * a.H * 2); }
    }
    if (wave < 4) {
        fwd_producer<Tin, kSave, kRagged, kMulti, kFuse, kNoR>(a, smem, s_wild, bh0, part, wave, lane);
    } else {
        const int cw = wave - 4, grp = cw / nq, q = part * nq + (cw - grp * nq);
        if (grp == 0) fwd_consumer<Tin, Ts, kSave, kRagged, kMulti, kFuse, 0>(a, smem, s_wild, bh0, q, lane);
        else fwd_consumer<Tin, Ts, kSave, kRagged, kMulti, kFuse, 1>(a, smem, s_wild, bh0, q, lane);
    }
    // exact second pass for every pair of this workgroup that had a tile leave the representable range
    // (workgroups sharing a pair all see the same flags; each leaves its own value columns, which do not depend on the others: those
    // of the initial state may have been overwritten by now)
    __threadfence_block();   // workgroup scope is enough (and a device-scope fence would write back the L2)
    __syncthreads();
    if (!kMulti && !kFuse && a.decay && part == 0 && threadIdx.x < kN) {
        const float *e = reinterpret_cast<const float *>(smem + FwdLds::kDecay) + threadIdx.x;
        a.decay[(int64_t)bh0 * kN + threadIdx.x] = exp2_fast(-((e[0] + e[kN]) + (e[2 * kN] + e[3 * kN])));
    }
    const int stride = (int)gridDim.x;
    const int n_my = kMulti ? (a.nitems - bh0 + stride - 1) / stride : 1;
    for (int n = 0; n < n_my; ++n) {
        if (!s_wild[n]) continue;   // uniform over the workgroup
        const int bh = bh0 + n * stride;
        __syncthreads();
        typedef typename OutOf<Tin>::type Tout;
        auto in = [](const void *p) { return reinterpret_cast<const Tin *>(p); };
        scan_fwd_body<Tin, Tout, Ts>(*reinterpret_cast<ScanFwdLds *>(smem), bh / a.H, bh % a.H, a.T, a.H, in(a.r), in(a.k), in(a.v_orig), in(a.w), in(a.u),
                                     reinterpret_cast<const Ts *>(a.s0), a.map, reinterpret_cast<Tout *>(kFuse ? a.out : a.y), reinterpret_cast<Ts *>(a.sT), a.reverse != 0,
                                     part * 16 * nq, (part + 1) * 16 * nq);
        if (kFuse) {
            __threadfence_block();
            __syncthreads();
            output_stage_in_place(a, bh);
        }
    }
}

// compute units of the current device (an immutable device property, looked up once per device)
int compute_units() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

template <typename Tin, typename Ts, bool kSave, bool kRagged, bool kMulti, bool kFuse, bool kNoR = false>
static hipError_t launch_fwd(hipStream_t st, const FwdArgs &a, unsigned grid) {
    constexpr auto kern = chunk_fwd_kernel<Tin, Ts, kSave, kRagged, kMulti, kFuse, kNoR>;
    const size_t lds = kFuse ? FwdLds::kBytesFused : FwdLds::kBytes;
    hipError_t e = allow_dynamic_lds<kern>((int)lds);
    if (e != hipSuccess) return e;
    const int split = kMulti || kFuse ? 1 : a.split;
    hipLaunchKernelGGL(kern, dim3(grid * split), dim3((4 + 8 / split) * 64), lds, st, a);
    return hipGetLastError();
}
template <typename Tin, typename Ts, bool kSave, bool kRagged, bool kFuse>
static hipError_t launch_fwd(hipStream_t st, const FwdArgs &a, bool multi, unsigned grid) {
    // no y wanted and fp32 states (the state-only passes of the backward and of the time segments):
    // the variant that leaves r alone
    if constexpr (!kFuse && std::is_same<Ts, float>::value && std::is_same<Tin, bf16_t>::value) {
        if (a.y == nullptr)
            return multi ? launch_fwd<Tin, Ts, kSave, kRagged, true, kFuse, true>(st, a, grid)
                         : launch_fwd<Tin, Ts, kSave, kRagged, false, kFuse, true>(st, a, grid);
    }
    return multi ? launch_fwd<Tin, Ts, kSave, kRagged, true, kFuse>(st, a, grid) : launch_fwd<Tin, Ts, kSave, kRagged, false, kFuse>(st, a, grid);
}
template <typename Ts>
static hipError_t launch_fwd(hipStream_t st, const FwdArgs &a, bool save, bool ragged, bool multi, unsigned grid) {
    if (save) return ragged ? launch_fwd<bf16_t, Ts, true, true, false>(st, a, multi, grid) : launch_fwd<bf16_t, Ts, true, false, false>(st, a, multi, grid);
    return ragged ? launch_fwd<bf16_t, Ts, false, true, false>(st, a, multi, grid) : launch_fwd<bf16_t, Ts, false, false, false>(st, a, multi, grid);
}
template <typename Ts>
static hipError_t launch_fwd_fused(hipStream_t st, const FwdArgs &a, bool ragged, bool multi, unsigned grid) {
    return ragged ? launch_fwd<bf16_t, Ts, false, true, true>(st, a, multi, grid) : launch_fwd<bf16_t, Ts, false, false, true>(st, a, multi, grid);
}

// One workgroup per pair while they all fit on the chip at once; beyond that one workgroup per
// compute unit (more only if a workgroup would otherwise get more pairs than it keeps flags for).
static unsigned forward_grid(int64_t pairs, bool *multi, int *split) {
    const int64_t cus = compute_units();
    *multi = pairs > cus;
    *split = pairs * 4 <= cus ? 4 : pairs * 2 <= cus ? 2 : 1;
    return (unsigned)(!*multi ? pairs : (pairs + cus * kMaxPairsPerWorkgroup - 1) / (cus * kMaxPairsPerWorkgroup) * cus);
}

hipError_t chunk_forward(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                         const void *r, const void *k, const void *v, const void *w, const void *u,
                         const void *s0, const int64_t *map, void *y, void *sT, void *saved_states, float *decay, bool reverse,
                         bool counters, RowCut cut, bool keep_inputs)
{
    // (rows that are segments and find their states here, not in the chain, are fewer than the block form takes: segments_in_block_form)
    if (y != nullptr && decay == nullptr && !reverse && !cut.segments && block_forward_applies(B, T, H))
        return block_forward(st, state_dtype, B, T, H, r, k, v, w, u, s0, map, y, sT, saved_states, counters, RowCut(), SegmentChain(), keep_inputs);
    FwdArgs a = {};
    a.decay = decay;
    a.reverse = reverse;
    a.cut = cut;
    a.T = (int)T; a.H = (int)H; a.nitems = (int)(B * H); a.slice = (int)((T + CL - 1) / CL);
    a.r = (const bf16_t *)r; a.k = (const bf16_t *)k; a.v = (const bf16_t *)v; a.w = (const bf16_t *)w; a.u = (const bf16_t *)u;
    a.v_orig = v;
    a.s0 = s0; a.map = map; a.y = (bf16_t *)y; a.sT = sT; a.ckpt = (float *)saved_states;
    a.arrivals = saved_states && counters ? reinterpret_cast<int *>(reinterpret_cast<char *>(saved_states) + chunk_backward_workspace_bytes(B, T, H)) : nullptr;
    bool multi;
    const unsigned grid = forward_grid(B * H, &multi, &a.split);
    if ((cut.segments || decay) && multi) return hipErrorInvalidValue;
    const bool save = saved_states != nullptr, ragged = (T % CL) != 0 || cut.segments;
    return state_dtype == kF32 ? launch_fwd<float>(st, a, save, ragged, multi, grid)
                               : launch_fwd<bf16_t>(st, a, save, ragged, multi, grid);
}

// bf16 copy of an fp16 or fp32 tensor (n a multiple of 8 elements, 16-byte aligned): what the MFMAs take as v and gy
template <typename Tsrc>
__global__ __launch_bounds__(256) void to_bf16_kernel(const Tsrc *__restrict__ src, bf16_t *__restrict__ dst, int64_t n8)
{
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
        Raw8<Tsrc> x;
        x.load(src + 8 * i);
        float f[8];
        x.to_float(f);
        *reinterpret_cast<uint4 *>(dst + 8 * i) = make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
    }
}
hipError_t convert_to_bf16(hipStream_t st, int src_dtype, const void *src, void *dst, int64_t n)
{
    const int64_t n8 = n / 8;
    const unsigned grid = (unsigned)((n8 + 255) / 256 < 16384 ? (n8 + 255) / 256 : 16384);
    if (src_dtype == kF16) hipLaunchKernelGGL(to_bf16_kernel<f16_t>, dim3(grid), dim3(256), 0, st, (const f16_t *)src, (bf16_t *)dst, n8);
    else hipLaunchKernelGGL(to_bf16_kernel<float>, dim3(grid), dim3(256), 0, st, (const float *)src, (bf16_t *)dst, n8);
    return hipGetLastError();
}

// The saving forward of the training pair for fp16 tensors (y fp32, zero initial state): r, k, w are
// read as fp16 and unpacked exactly, v_bf16 is the bf16 copy of v the MFMAs take.
hipError_t chunk_forward_save_f16(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                  const void *r, const void *k, const void *v, const void *v_bf16, const void *w, const void *u,
                                  void *y, void *saved_states)
{
    FwdArgs a = {};
    a.T = (int)T; a.H = (int)H; a.nitems = (int)(B * H); a.slice = (int)((T + CL - 1) / CL);
    a.r = (const bf16_t *)r; a.k = (const bf16_t *)k; a.v = (const bf16_t *)v_bf16; a.w = (const bf16_t *)w; a.u = (const bf16_t *)u;
    a.v_orig = v;
    a.y = (bf16_t *)y; a.ckpt = (float *)saved_states;
    a.arrivals = reinterpret_cast<int *>(reinterpret_cast<char *>(saved_states) + chunk_backward_workspace_bytes(B, T, H));
    bool multi;
    const unsigned grid = forward_grid(B * H, &multi, &a.split);
    return (T % CL) != 0 ? launch_fwd<f16_t, float, true, true, false>(st, a, multi, grid)
                         : launch_fwd<f16_t, float, true, false, false>(st, a, multi, grid);
}

hipError_t chunk_forward_fused(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                               const void *r, const void *k, const void *v, const void *w, const void *u,
                               const void *s0, const int64_t *map, const void *gate, const float *gn_scale,
                               const float *gn_offset, float gn_eps, void *out, void *sT, RowCut cut)
{
    if (!cut.segments && block_forward_applies(B, T, H))
        return block_forward_fused(st, state_dtype, B, T, H, r, k, v, w, u, s0, map, gate, gn_scale, gn_offset, gn_eps, out, nullptr, nullptr, sT, nullptr);
    FwdArgs a = {};
    a.T = (int)T; a.H = (int)H; a.nitems = (int)(B * H); a.slice = (int)((T + CL - 1) / CL);
    a.r = (const bf16_t *)r; a.k = (const bf16_t *)k; a.v = (const bf16_t *)v; a.w = (const bf16_t *)w; a.u = (const bf16_t *)u;
    a.s0 = s0; a.map = map; a.sT = sT;
    a.v_orig = v;
    a.gate = (const bf16_t *)gate; a.gn_scale = gn_scale; a.gn_offset = gn_offset; a.gn_eps = gn_eps; a.out = (bf16_t *)out;
    bool multi;
    const unsigned grid = forward_grid(B * H, &multi, &a.split);
    a.split = 1;   // the output stage needs a chunk's whole rows in one workgroup
    a.cut = cut;
    if (cut.segments && multi) return hipErrorInvalidValue;
    const bool ragged = (T % CL) != 0 || cut.segments;
    return state_dtype == kF32 ? launch_fwd_fused<float>(st, a, ragged, multi, grid)
                               : launch_fwd_fused<bf16_t>(st, a, ragged, multi, grid);
}

// Training with the fused output stage: out = (group_norm_head(y) * gn_scale + gn_offset) * gate, and for
// the backward y itself (bf16), the norm's statistics and the chunk states.  s0: null (zero initial state: what
// the caller sees), or one fp32 state per pair (a segment's incoming state).
static hipError_t fused_save_from(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                  const void *r, const void *k, const void *v, const void *w, const void *u, const float *s0,
                                  const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps,
                                  void *out, void *y, float *stats, void *saved_states, GnSums sums, RowCut cut = RowCut())
{
    if (!cut.segments && block_forward_applies(B, T, H))
        return block_forward_fused(st, kF32, B, T, H, r, k, v, w, u, s0, nullptr, gate, gn_scale, gn_offset, gn_eps, out, y, stats, nullptr, saved_states,
                                   RowCut(), SegmentChain(), sums);
    FwdArgs a = {};
    a.s0 = s0; a.sums = sums;
    a.T = (int)T; a.H = (int)H; a.nitems = (int)(B * H); a.slice = (int)((T + CL - 1) / CL);
    a.r = (const bf16_t *)r; a.k = (const bf16_t *)k; a.v = (const bf16_t *)v; a.w = (const bf16_t *)w; a.u = (const bf16_t *)u;
    a.v_orig = v;
    a.gate = (const bf16_t *)gate; a.gn_scale = gn_scale; a.gn_offset = gn_offset; a.gn_eps = gn_eps; a.out = (bf16_t *)out;
    a.y = (bf16_t *)y; a.stats = stats; a.ckpt = (float *)saved_states;
    a.arrivals = reinterpret_cast<int *>(reinterpret_cast<char *>(saved_states) + chunk_backward_workspace_bytes(B, T, H));
    bool multi;
    const unsigned grid = forward_grid(B * H, &multi, &a.split);
    a.split = 1;
    a.cut = cut;
    if (cut.segments && multi) return hipErrorInvalidValue;
    return (T % CL) != 0 || cut.segments ? launch_fwd<bf16_t, float, true, true, true>(st, a, multi, grid)
                         : launch_fwd<bf16_t, float, true, false, true>(st, a, multi, grid);
}
hipError_t chunk_forward_fused_save(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                    const void *r, const void *k, const void *v, const void *w, const void *u,
                                    const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps,
                                    void *out, void *y, float *stats, void *saved_states, GnSums sums)
{
    return fused_save_from(st, B, T, H, r, k, v, w, u, nullptr, gate, gn_scale, gn_offset, gn_eps, out, y, stats, saved_states, sums);
}

// ------------------------------------------------------------------------------------------
// Long sequences, few pairs: time cut into segments that run side by side.
//
// With fewer (batch, head) pairs than half the compute units most of the chip would idle while each
// pair walks its sequence alone.  The map from a segment's incoming state to its outgoing state is
// affine, S_out = D o S_in + U with D[j] = exp(-sum_t exp(w_t[j])) over the segment and U the state
// the segment builds from zero, so: (A) every segment runs from a zero state (block form: wkv6_state.hip; all segments at once;
// a (B,T,C) tensor cut into P equal segments IS a (B*P, T/P, C) tensor, and RowCut stands for other lengths; no y in this pass) and leaves
// U and, from the producer waves, D; (B) the P affine maps of a pair are chained, at the start of the second pass in
// the block form (chain_start), by a tiny kernel that leaves each segment's true incoming state where its U was (and the final
// state) in the others; (C) every segment runs again from its true state and writes y.  Twice the forward work on P times the
// workgroups.
// ------------------------------------------------------------------------------------------
constexpr int kMostSegments = 16;
// kReverse: the same chain walked from the last segment to the first, which is what the reverse
// state of the backward pass obeys (the gradient arriving at the end of segment p is what segment
// p + 1 sends into its incoming state: its own contribution plus D_{p+1} times what arrives at its end).
// kFactors: `decay` holds one or two factors of each segment's decay, [kFactors][pairs][64].
template <typename Ts, bool kReverse, int P, int kFactors>
__global__ __launch_bounds__(256) void segment_chain_kernel(int H, const Ts *__restrict__ s0, const int64_t *__restrict__ map,
                                                            const float *__restrict__ decay, float *__restrict__ states, Ts *__restrict__ sT)   // sT: the final state, or null
{
    // Thread: four value columns i0..i0+3 of one key row j of one (batch, head): 1024 threads per pair,
    // gridDim.x * 256 = B * H * 1024.  states[(b*P + seg), h] holds U on entry and the segment's
    // incoming state on exit.  All P loads are issued before the chain is walked (their addresses do
    // not depend on it): the kernel takes about two memory round trips instead of 2 P.  For that P has to be known to the
    // compiler: loops of up to 16 steps with a way out at a run-time P kept x and d in 272 bytes of scratch memory (a prompt of
    // B1 T4096 H8, 16 segments: 43 us), and with steps past P that change nothing it took 32 us (so: 27.5 us).
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int i0 = (e & 15) * 4, j = (e >> 4) & 63, bh = e >> 10;
    const int b = bh / H, h = bh - b * H;
    const int64_t np = (int64_t)(gridDim.x >> 2) * P;   // pairs of all segments
    auto pair_of_step = [&](int n) { return ((int64_t)b * P + (kReverse ? P - 1 - n : n)) * H + h; };   // step n of the walk
    float4 x[P];
    float d[P];
#pragma unroll
    for (int n = 0; n < P; ++n) {
        const int64_t vp = pair_of_step(n);
        x[n] = *reinterpret_cast<const float4 *>(states + (vp * kN + j) * kN + i0);
        d[n] = decay[vp * kN + j];
        if (kFactors == 2) d[n] *= decay[(np + vp) * kN + j];
    }
    float S[4] = {0.f, 0.f, 0.f, 0.f};
    if (s0) {
        const int64_t row = map ? map[b] : (int64_t)b;
        load4(s0 + ((row * H + h) * kN + j) * kN + i0, S);
    }
#pragma unroll
    for (int n = 0; n < P; ++n) {
        const float dd = d[n];
        *reinterpret_cast<float4 *>(states + (pair_of_step(n) * kN + j) * kN + i0) = make_float4(S[0], S[1], S[2], S[3]);
        S[0] = fmaf(S[0], dd, x[n].x); S[1] = fmaf(S[1], dd, x[n].y); S[2] = fmaf(S[2], dd, x[n].z); S[3] = fmaf(S[3], dd, x[n].w);
    }
    if (sT) store4(sT + (((int64_t)b * H + h) * kN + j) * kN + i0, S[0], S[1], S[2], S[3]);
}
template <typename Ts, bool kReverse, int kFactors = 1, int N = kMostSegments>
static hipError_t launch_chain(hipStream_t st, int P, int64_t B, int64_t H, const Ts *s0, const int64_t *map,
                               const float *decay, float *states, Ts *sT)
{
    if constexpr (N < 2) {
        return hipErrorInvalidValue;
    } else {
        if (P != N) return launch_chain<Ts, kReverse, kFactors, N - 1>(st, P, B, H, s0, map, decay, states, sT);
        hipLaunchKernelGGL((segment_chain_kernel<Ts, kReverse, N, kFactors>), dim3((unsigned)(B * H * 4)), dim3(256), 0, st, (int)H, s0, map, decay, states, sT);
        return hipGetLastError();
    }
}

// Segments of a sequence of T tokens when `pairs` (batch, head) pairs share the chip: as many as still fit it once, each a
// whole number of chunks and at least `least` of them; the last one ends with the sequence.  (Segments that had to
// divide the sequence left training at all other lengths to one workgroup per pair: forward and backward at H32 T8191 771 ->
// 176 us, H8 T5003 475 -> 88.  At least three chunks of a prompt and four in training, as long as the chain was a launch of its
// own, / one: training pair bf16 B1 T1400 H16 67.8 / 44.4, T1900 H8 66.8 / 44.4, fp32 B1 T1400 H8 116 / 77, prompt T1337 H8 23.2 / 19.2.)
int plan_segments(int64_t pairs, int64_t T, int64_t least, int64_t *L) {
    const int64_t chunks = (T + CL - 1) / CL, fit = compute_units() / pairs;
    const int64_t most = fit < kMostSegments ? fit : kMostSegments;
    if (most < 2) return 1;
    int64_t n = (chunks + most - 1) / most;
    if (n < least) n = least;
    *L = n * CL;
    return (int)((chunks + n - 1) / n);
}
RowCut cut_of(int P, int64_t L, int64_t T) {
    RowCut c;
    if (P * L != T) { c.segments = P; c.total = T; }
    return c;
}

// The second pass of the segments, `rows` of them: in block form from a quarter of the chip on (half of it, in one piece:
// the tile form's two workgroups to a pair save nothing that the chain at the start and whole rows do not save as well; training pair of
// B1 H8 T1000 46.6 us as tiles / 36.8, T4000 73.8 / 63.0, H4 T768 38.8 / 31.2).  Fewer rows still run the tile form, whose y is, but
// for the chain's rounding, that of a call in one piece.
bool segments_in_block_form(int64_t rows, int64_t H) { return 4 * rows * H >= compute_units(); }

// From which length a prompt of `pairs` (batch, head) pairs runs in P segments.  Two things move the line besides P and the output stage,
// which the first pass leaves out.  A prompt of whole chunks runs in one piece on kernels without the checks of a ragged end, and pays later.
// And the workgroups of a head's segments, H apart in the grid, are on one XCD, where the second pass finds the first one's states in
// the L2, only if H is a multiple of 8 (else on two, and of four or eight where H is no multiple of 4).  In one piece / in segments, us:
//   four and more     B1 H32 T200 11.2 / 10.6, B2 H32 T256 12.5 / 11.6, few pairs B2 H8 T256 9.7 / 10.4; B4 H12 T256 11.6 / 12.3, T257 13.6 / 13.1;
//                     B4 H14 T256 12.1 / 14.4, B4 H10 T384 14.3 / 15.0, T448 16.0 / 15.3, B6 H10 T448 17.3 / 17.7, but B2 H14 T384 13.7 / 13.1
//   three             B4 H20 T512 18.1 / 19.2, T576 19.8 / 19.5; B6 H14 T640 21.6 / 22.0; B3 H28 T530 20.5 / 19.4, T700 24.0 / 21.4
//   two               B2 H64 T1344 42.4 / 43.1, T1100 37.4 / 37.3; B6 H20 T1280 39.6 / 40.4, B4 H32 T1500 49.2 / 47.6
//   with the stage    four B1 H32 T200 14.6 / 11.7, B3 H20 T256 13.8 / 14.8, B4 H14 T256 13.6 / 15.8; three B3 H28 T320 16.5 / 17.5, T260 18.3 / 16.8;
//                     two B2 H64 T320 17.4 / 19.4, T330 22.5 / 19.3, B4 H30 T448 22.0 / 23.1
static bool prompt_takes(int P, int64_t T, int64_t pairs, int64_t H, bool fused) {
    struct Least { int ragged, whole; };
    static constexpr Least kLeast[3][2][3] = {   // two segments, three, four and more; without and with the output stage; H a multiple of 8, of 4, others
        {{{1281, 1408}, {1281, 1408}, {1281, 1408}}, {{321, 384}, {321, 512}, {321, 512}}},
        {{{513, 512}, {513, 576}, {513, 704}}, {{257, 320}, {257, 384}, {257, 384}}},
        {{{193, 256}, {257, 320}, {385, 512}}, {{193, 256}, {193, 320}, {257, 384}}}};
    if (P < 2) return false;
    const int heads = H % 8 == 0 ? 0 : H % 4 == 0 ? 1 : 2;
    Least l = kLeast[P >= 4 ? 2 : P - 2][fused][heads];
    if (P >= 4 && !fused && heads == 0 && pairs <= 16) l = {257, 320};
    if (P >= 4 && !fused && heads == 2 && pairs <= 32) l.whole = 384;
    return T >= (T % CL == 0 ? l.whole : l.ragged);
}
// any_length: a batch's length need not divide into the segments, either.  Without it (wkv6_forward_workspace_bytes, which promises
// no workspace then) a batch of prompts ran as segments only where 16, 8, 4 or 2 equal ones of whole chunks make its length,
// and otherwise on one or two workgroups a pair.
static int forward_segments_plan(int64_t B, int64_t T, int64_t H, bool fused, bool any_length, int64_t *L) {
    if (B == 1 || any_length) {
        int P = plan_segments(B * H, T, 1, L);
        if (P > 1 && segments_in_block_form(B * P, H)) return prompt_takes(P, T, B * H, H, fused) ? P : 1;
        P = T >= 1024 ? plan_segments(B * H, T, 3, L) : 1;
        return P >= 4 ? P : 1;
    }
    for (int P = kMostSegments; P >= 2; P >>= 1)
        if (B * H * P <= compute_units() && T % (P * CL) == 0 &&
            (segments_in_block_form(B * P, H) ? prompt_takes(P, T, B * H, H, fused) : T >= 1024 && P >= 4 && T / P >= 4 * CL)) {
            *L = T / P;
            return P;
        }
    return 1;
}
size_t chunk_forward_segments_workspace_bytes(int64_t B, int64_t T, int64_t H, bool fused, bool any_length) {
    int64_t L;
    const int P = forward_segments_plan(B, T, H, fused, any_length, &L);
    // per segment and pair two states (what it leaves alone, what it starts from) and the decay
    return P <= 1 ? 0 : (size_t)(B * P * H) * (2 * kN * kN + kN) * sizeof(float);
}

// With `gate` the second pass runs the fused output stage (y = out then).
hipError_t chunk_forward_segments_run(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                                      const void *r, const void *k, const void *v, const void *w, const void *u,
                                      const void *s0, const int64_t *map, void *y, void *sT, void *workspace, bool any_length,
                                      const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps)
{
    int64_t L = 0;
    const int P = forward_segments_plan(B, T, H, gate != nullptr, any_length, &L);
    const int64_t rows = B * P;
    const RowCut cut = cut_of(P, L, T);
    float *states = (float *)workspace, *start = states + rows * H * kN * kN, *decay = start + rows * H * kN * kN;
    if (segments_in_block_form(rows, H)) {   // the chain at the start of the second pass
        GivenStates given;
        given.states = s0; given.map = map; given.bf16 = state_dtype != kF32; given.P = P; given.start = start;
        const hipError_t e = segment_states(st, rows, L, H, k, v, w, u, states, decay, false, cut, given);
        if (e != hipSuccess) return e;
        SegmentChain c;
        c.P = P; c.alone = states; c.decay = decay; c.given = s0 != nullptr; c.last = sT; c.bf16 = state_dtype != kF32; c.start = start;
        return gate ? block_forward_fused(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, gate, gn_scale, gn_offset, gn_eps, y, nullptr, nullptr, nullptr, nullptr, cut, c)
                    : block_forward(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, y, nullptr, nullptr, true, cut, c);
    }
    hipError_t e = chunk_forward(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, nullptr, states, nullptr, decay, false, true, cut);
    if (e != hipSuccess) return e;
    e = state_dtype == kF32 ? launch_chain<float, false>(st, P, B, H, (const float *)s0, map, decay, states, (float *)sT)
                            : launch_chain<bf16_t, false>(st, P, B, H, (const bf16_t *)s0, map, decay, states, (bf16_t *)sT);
    if (e != hipSuccess) return e;
    return gate ? chunk_forward_fused(st, kF32, rows, L, H, r, k, v, w, u, states, nullptr, gate, gn_scale, gn_offset, gn_eps, y, nullptr, cut)
                : chunk_forward(st, kF32, rows, L, H, r, k, v, w, u, states, nullptr, y, nullptr, nullptr, nullptr, false, true, cut);
}

hipError_t segment_chain_reverse(hipStream_t st, int P, int64_t B, int64_t H, const float *decay, float *states,
                                 const float *arriving, float *leaving) {
    return launch_chain<float, true>(st, P, B, H, arriving, nullptr, decay, states, leaving);
}
hipError_t segment_chain_factors(hipStream_t st, int P, int64_t B, int64_t H, const float *decay, float *states, bool reverse) {
    return reverse ? launch_chain<float, true, 2>(st, P, B, H, nullptr, nullptr, decay, states, nullptr)
                   : launch_chain<float, false, 2>(st, P, B, H, nullptr, nullptr, decay, states, nullptr);
}
hipError_t segment_chain_forward(hipStream_t st, int P, int64_t B, int64_t H, const float *decay, float *states, const float *s0) {
    return launch_chain<float, false>(st, P, B, H, s0, nullptr, decay, states, nullptr);
}

// ------------------------------------------------------------------------------------------
// The same for the training pair (saving forward, backward from the saved states): the forward
// keeps every segment's incoming state and the decay over it for the backward, whose reverse state
// is chained the same way (see chunk_backward_saved_segments).
// ------------------------------------------------------------------------------------------
// The pair of kernels gains at every length, in one piece / in segments: B1 T512 H8 57.9 / 30.7 us, T768 H8 80.7 / 33.1, H40 82.1 / 43.1,
// T1000 H16 108 / 39, B2 T1000 H12 108 / 47; two segments B2 H48 T768 84.8 / 71.2, T1000 113 / 92, T1900 197 / 145.  But a step through
// the torch flavour takes 75 us of host time with the two more launches and 65 without, so below 705 tokens, where one piece takes less
// than that, a caller who waits for each step would lose: B1 T705 H8 79.4 / 73.8 us, B2 T740 H12 81.5 / 75.8, B1 T768 H32 77.5 / 78.4, T800 H16
// 86.8 / 77.3.  Two or three segments from 833 on: the backward without saved states, which takes the same plan, loses with them before
// (B5 T768 H24 75.7 / 78.3, T1000 101.8 / 97.8).
static int train_segments_plan(int64_t B, int64_t T, int64_t H, int64_t *L) {
    if (T <= 704) return 1;
    int P = plan_segments(B * H, T, 1, L);
    if (segments_in_block_form(B * P, H)) return P >= 4 || T > 832 ? P : 1;
    // (tile form: two state-only passes at 0.7 of a forward each on top of the forward and the backward, and three small kernels)
    if (T < 1024) return 1;
    P = plan_segments(B * H, T, 4, L);
    return T >= 2048 || P >= 4 ? P : 1;
}
int chunk_train_segments(int64_t B, int64_t T, int64_t H) {
    int64_t L;
    return train_segments_plan(B, T, H, &L);
}
TrainSegments train_segments_layout(int64_t B, int64_t T, int64_t H, void *extra) {
    TrainSegments s;
    s.L = T;
    s.P = train_segments_plan(B, T, H, &s.L);
    s.cut = cut_of(s.P, s.L, T);
    const size_t pairs = (size_t)(B * s.P * H);
    s.states = reinterpret_cast<float *>(extra);
    s.gstates = s.states + pairs * kN * kN;
    s.decay = s.gstates + pairs * kN * kN;
    s.gu_rows = s.decay + pairs * kN;
    s.alone = s.gu_rows + pairs * kN;
    s.bytes_unsaved = pairs * (2 * kN * kN + 2 * kN) * sizeof(float);
    s.bytes = s.bytes_unsaved + pairs * kN * kN * sizeof(float);
    return s;
}

// The second pass of the saving forward, from what the first one left in `alone` and `decay`.
static SegmentChain train_chain(const TrainSegments &s, float *start) {
    SegmentChain c;
    c.P = s.P; c.alone = s.alone; c.decay = s.decay; c.start = start;
    return c;
}
hipError_t chunk_forward_save_segments(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                       const void *r, const void *k, const void *v, const void *w, const void *u,
                                       void *y, void *saved, void *extra)
{
    const TrainSegments s = train_segments_layout(B, T, H, extra);
    const int64_t L = s.L, rows = B * s.P;
    const bool block = segments_in_block_form(rows, H);
    hipError_t e = block ? segment_states(st, rows, L, H, k, v, w, u, s.alone, s.decay, false, s.cut, GivenStates(), s.P)
        : chunk_forward(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, nullptr, s.states, nullptr, s.decay, false, true, s.cut);
    if (e != hipSuccess) return e;
    if (block) return block_forward(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, y, nullptr, saved, true, s.cut, train_chain(s, s.states));
    if ((e = segment_chain_forward(st, s.P, B, H, s.decay, s.states, nullptr)) != hipSuccess) return e;
    return chunk_forward(st, kF32, rows, L, H, r, k, v, w, u, s.states, nullptr, y, nullptr, saved, nullptr, false, true, s.cut);
}

// The same with the fused output stage in the second pass.  out, y, gate and the statistics are indexed by
// token, and the tokens of the B*P rows are those of the (B, T) rows in the same order.
hipError_t chunk_forward_fused_save_segments(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                             const void *r, const void *k, const void *v, const void *w, const void *u,
                                             const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps,
                                             void *out, void *y, float *stats, void *saved, void *extra, GnSums sums)
{
    const TrainSegments s = train_segments_layout(B, T, H, extra);
    const int64_t L = s.L, rows = B * s.P;
    const bool block = segments_in_block_form(rows, H);
    hipError_t e = block ? segment_states(st, rows, L, H, k, v, w, u, s.alone, s.decay, false, s.cut, GivenStates(), s.P)
        : chunk_forward(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, nullptr, s.states, nullptr, s.decay, false, true, s.cut);
    if (e != hipSuccess) return e;
    if (block) return block_forward_fused(st, kF32, rows, L, H, r, k, v, w, u, nullptr, nullptr, gate, gn_scale, gn_offset, gn_eps, out, y, stats, nullptr, saved, s.cut, train_chain(s, s.states), sums);
    if ((e = segment_chain_forward(st, s.P, B, H, s.decay, s.states, nullptr)) != hipSuccess) return e;
    return fused_save_from(st, rows, L, H, r, k, v, w, u, s.states, gate, gn_scale, gn_offset, gn_eps, out, y, stats, saved, sums, s.cut);
}

}  // namespace wkv6
