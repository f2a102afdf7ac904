// Backward of the full-precision chunk form (see wkv6_chunk32.h): fp32 and fp16 tensors, gradients fp32-exact
// to rounding, every product on v_mfma_f32_16x16x4_f32.
//
// Chunks of 32 tokens from the last to the first.  With S_0 the state at the chunk's start (saved by the
// forward), G = dL/dS at its end, B[t][s] = sum_j gy_t[j] v_s[j] (s < t), vgy_t = B[t][t], A as in the forward:
//   gv_s = K'_s G + sum_{t>=s} A[t][s] gy_t                       (A's diagonal holds sum_i r u k)
//   gr_t = e^{c_t} o Z_t + u k_t vgy_t ,    Z_t = gy_t S_0^T + e^{-m} o sum_{s<t} B[t][s] K~_s
//   gk_s = e^{c_32-c_{s+1}} o W_s + u r_s vgy_s ,  W_s = v_s G^T + e^{m-c_32} o sum_{t>s} B[t][s] R~_t
//   gu  += r_t k_t vgy_t
//   G   <- e^{c_32} o G + R'^T gy
//   gw_t = d_t (E_{t+1} - K'_t W_t) ,  E_t = E_{t+1} + R'_t Z_t - K'_t W_t ,  E_T = 0
// (E_t[i] = sum_j S_t[i][j] G_t[i][j]: what flows into channel i's decay at token t is the balance of what
// the later tokens read from the state and what they wrote to it.)
//
// One workgroup of twelve waves per (batch, head) pair, three roles of four waves (one wave of each role per SIMD,
// so that one role's waits are another's issue slots):
//   loading waves   tiles R', K', v, gy of the next chunk and r, k, e^{c_t}, e^{c_32-c_{t+1}}, d of the chunk in hand
//                   -> LDS (loads issued a step and a half ahead of their use)
//   value waves     wave q owns value columns 16q.. of G: gv = K' G + A^T gy, the update of G, the tiles of A
//   key waves       wave q owns key rows 16q.. of every per-channel output: Z, W, gr, gk, gw, gu, the tiles of B; S_0^T
//                   comes straight from the saved states, G^T from the value waves through LDS (a copy kept up to date by
//                   the key waves themselves cost a seventh of all matrix instructions)
// Two workgroup barriers per chunk, the matrix instructions shared out evenly between the two phases (24 and 25 products
// over 16 indices per SIMD):
//   phase 1  tiles of A and B -> LDS ; K' G ; v G^T
//   phase 2  gy S_0^T ; the three products with A and B ; gradients out (lane = token, 16 bytes each) ; G update -> LDS
#include "wkv6_chunk32.h"
#include "wkv6_kernels.h"
#include "wkv6_scan_body.h"

#include <type_traits>

namespace wkv6 {

struct C32BwdLds {
    float Rp[2][kC32][kLd], Kp[2][kC32][kLd], V[2][kC32][kLd], GY[2][kC32][kLd];   // R', K', v, gy of the chunk in hand and the next
    // what only the key waves' second phase reads: one copy, written in the first phase of the same step
    float R[kC32][kLd], K[kC32][kLd], F1[kC32][kLd], F3[kC32][kLd], D[kC32][kLd];   // r, k, e^{c_t}, e^{c_32 - c_{t+1}}, log decay
    float A[kC32][kLa], Bm[kC32][kLa];
    float G[kN][kLd];                                                             // dL/dS at the chunk's end, [value][key]
    float e_all[2][kN], e_mid[2][kN], e_rest[2][kN], inv0[2][kN], inv1[2][kN];    // e^{c_32}, e^{m}, e^{c_32-m}, e^{-m}, e^{m-c_32}
    float ruk[2][4][kC32];
    float vgy[kC32];
    int wild[4];
};
union C32BwdSmem {
    C32BwdLds chunk;
    ScanBwdALds scan_a;
    ScanBwdBLds scan_b;
};

struct C32BwdArgs {
    int T, H;
    const void *r, *k, *v, *w, *u, *gy;
    void *gr, *gk, *gv, *gw, *gu;
    float *saved;   // [pair][chunk][4096] chunk-start states as the forward leaves them (fragment order)
    // gradients through the state, [pair][key][value] fp32, all null for the stateless operator: the initial state
    // (only the per-timestep second pass reads it: the chunk states already contain it), the gradient arriving at
    // the final state, the final state itself (read where gsT is given: E_T = sum_j S_T o gsT), dL/dS_0 (out)
    const float *s0, *gsT, *sT;
    float *gs0;
    int slice;      // chunks of a pair's slice of `saved` (those of the longest row)
    RowCut cut;     // rows that are time segments
    int P;          // ... of which so many make a sequence (0: every row is a sequence)
    // Sums of gu, by the last workgroup of a head to arrive (null: not wanted): every row leaves its part, written through, at
    // parts + row * part_row + head * part_head; arrivals[head * arrival_step] counts.  Without segments both lie in the pairs'
    // slices of `saved`, in the place of the first chunk's state, which is zero and not read.
    float *parts;
    int64_t part_row, part_head;
    int *arrivals;
    int64_t arrival_step;
    void *gu_sum;     // (C) in Tg, or null
    float *gu_seq;    // with segments: (sequences, C)
};

// kOnlyG: only the reverse state is wanted (gs0): the value waves update it, everything else is left out.  (A pair that is
// redone per timestep writes its gradients too, for the pass behind this one to write again.)
// Tg: type of gr, gk, gv, gw (gu is Tout).  fp16 gradients are the fp32 ones rounded once, where they leave: what torch makes of fp32
// gradients of fp16 tensors in five kernels of its own.  Forward and backward through the torch flavour, B2 T200 H8: 100 us
// with fp32 gradients converted behind the call, 70 so; B8 T1024 H32: 375 / 291.
template <typename Tin, typename Tout, typename Tg, bool kOnlyG>
__global__ __launch_bounds__(768) void chunk32_bwd_kernel(C32BwdArgs a)
{
    extern __shared__ __align__(16) unsigned char c32_smem[];
    C32BwdLds &L = reinterpret_cast<C32BwdSmem *>(c32_smem)->chunk;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int H = a.H, pair = blockIdx.x, b = pair / H, h = pair - b * H;
    if (a.cut.segments) {
        const RowView rv = row_view(a.cut, b, a.T);
        const int64_t m = rv.shift * H * kN;
        a.T = rv.tokens;
        a.r = reinterpret_cast<const Tin *>(a.r) + m; a.k = reinterpret_cast<const Tin *>(a.k) + m;
        a.v = reinterpret_cast<const Tin *>(a.v) + m; a.w = reinterpret_cast<const Tin *>(a.w) + m;
        a.gy = reinterpret_cast<const Tout *>(a.gy) + m;
        a.gr = reinterpret_cast<Tg *>(a.gr) + m; a.gk = reinterpret_cast<Tg *>(a.gk) + m;
        a.gv = reinterpret_cast<Tg *>(a.gv) + m; a.gw = reinterpret_cast<Tg *>(a.gw) + m;
    }
    const int T = a.T;
    const int64_t C = (int64_t)H * kN;
    const int64_t base = (int64_t)b * T * C + (int64_t)h * kN;
    const int nchunk = (T + kC32 - 1) / kC32;
    const Tin *r = reinterpret_cast<const Tin *>(a.r), *k = reinterpret_cast<const Tin *>(a.k);
    const Tin *v = reinterpret_cast<const Tin *>(a.v), *w = reinterpret_cast<const Tin *>(a.w);
    const Tin *u = reinterpret_cast<const Tin *>(a.u);
    const Tout *gy = reinterpret_cast<const Tout *>(a.gy);
    float *const ck = a.saved + (int64_t)pair * a.slice * (kN * kN);
    const bool first_row = a.P ? b % a.P == 0 : a.s0 == nullptr, last_row = a.P && b % a.P == a.P - 1;
    __shared__ float s_gu[kN];   // the row's gu
    // step s handles chunk nchunk - 1 - s

    if (wave >= 8) {
        // ---------------- loading waves ----------------
        const int p = wave - 8, t16 = lane & 15, ch = 16 * p + 4 * (lane >> 4);
        float fu[4];
        load4(u + h * kN + ch, fu);
        struct Set { Raw4<Tin> r[2], k[2], v[2], w[2]; Raw4<Tout> g[2]; };   // a chunk as loaded
        Set set0, set1;
        auto fetch = [&](Set &n, int s) {
            if (s >= nchunk) return;
            const int c = nchunk - 1 - s;
            const int64_t row0 = base + (int64_t)c * kC32 * C;   // (uniform)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int o = min(16 * x + t16, T - 1 - c * kC32) * (int)C + ch;   // rows past the end read the last one
                n.r[x].load(r + row0 + o); n.w[x].load(w + row0 + o);
                if (!kOnlyG) { n.k[x].load(k + row0 + o); n.v[x].load(v + row0 + o); }
                n.g[x].load(gy + row0 + o);
            }
        };
        float f1[2][4], f3[2][4], dd[2][4];
        bool wild = false;
        auto as4 = [](const float (&f)[4]) { return (f32x4){f[0], f[1], f[2], f[3]}; };
        // operands of step s -> LDS, the scale factors stay in registers for rows()
        auto form = [&](const Set &n, int s) {
            if (s >= nchunk) return;
            const int c = nchunk - 1 - s, buf = s & 1;
            const bool valid[2] = {c * kC32 + t16 < T, c * kC32 + 16 + t16 < T};
            C32Scale sc;
            sc.wild = false;
            float fw[2][4];
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) fw[x][e] = n.w[x].at(e);
            c32_scale<0, 4>(fw, valid, sc, dd);
            wild |= sc.wild;
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int t = 16 * x + t16;
                float acc = 0.f;
                f32x4 rp, kp, fv, fg;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float fr = valid[x] ? n.r[x].at(e) : 0.f, fk = !kOnlyG && valid[x] ? n.k[x].at(e) : 0.f;
                    fv[e] = !kOnlyG && valid[x] ? n.v[x].at(e) : 0.f;
                    fg[e] = valid[x] ? n.g[x].at(e) : 0.f;
                    f1[x][e] = sc.rp[x][e];
                    f3[x][e] = sc.kp[x][e];
                    rp[e] = fr * f1[x][e];
                    kp[e] = fk * f3[x][e];
                    acc = fmaf(fr * fk, fu[e], acc);
                }
                *reinterpret_cast<f32x4 *>(&L.Rp[buf][t][ch]) = rp;
                if (kOnlyG) {
                    *reinterpret_cast<f32x4 *>(&L.GY[buf][t][ch]) = fg;
                    continue;
                }
                acc = sum_rows4(acc);
                *reinterpret_cast<f32x4 *>(&L.Kp[buf][t][ch]) = kp;
                *reinterpret_cast<f32x4 *>(&L.V[buf][t][ch]) = fv;
                *reinterpret_cast<f32x4 *>(&L.GY[buf][t][ch]) = fg;
                if (lane < 16) L.ruk[buf][p][t] = acc;
            }
            if (t16 == 0) {
                *reinterpret_cast<f32x4 *>(&L.e_all[buf][ch]) = as4(sc.all);
                *reinterpret_cast<f32x4 *>(&L.e_mid[buf][ch]) = as4(sc.mid);
                *reinterpret_cast<f32x4 *>(&L.e_rest[buf][ch]) = as4(sc.rest);
                *reinterpret_cast<f32x4 *>(&L.inv0[buf][ch]) = as4(sc.inv0);
                *reinterpret_cast<f32x4 *>(&L.inv1[buf][ch]) = as4(sc.inv1);
            }
        };
        auto rows = [&](const Set &n, int s) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int t = 16 * x + t16;
                const bool valid = (nchunk - 1 - s) * kC32 + t < T;
                f32x4 fr, fk;
#pragma unroll
                for (int e = 0; e < 4; ++e) { fr[e] = valid ? n.r[x].at(e) : 0.f; fk[e] = valid ? n.k[x].at(e) : 0.f; }
                *reinterpret_cast<f32x4 *>(&L.R[t][ch]) = fr;
                *reinterpret_cast<f32x4 *>(&L.K[t][ch]) = fk;
                *reinterpret_cast<f32x4 *>(&L.F1[t][ch]) = as4(f1[x]);
                *reinterpret_cast<f32x4 *>(&L.F3[t][ch]) = as4(f3[x]);
                *reinterpret_cast<f32x4 *>(&L.D[t][ch]) = as4(dd[x]);
            }
        };
        // Phase 1 of step s: the rows of step s to LDS, the loads of step s + 2 issued into the registers that this frees.
        // Phase 2: the operands of step s + 1 formed and published (their loads are a step and a half old).
        auto step = [&](Set &now, Set &next, int s) {
            if (!kOnlyG) rows(now, s);
            fetch(now, s + 2);
            __syncthreads();
            form(next, s + 1);
            __syncthreads();
        };
        fetch(set0, 0);
        fetch(set1, 1);
        form(set0, 0);
        __syncthreads();
        for (int s = 0; s < nchunk; s += 2) {
            step(set0, set1, s);
            if (s + 1 < nchunk) step(set1, set0, s + 1);
        }
        const bool any = __any(wild);
        if (lane == 0) L.wild[p] = any;
    } else if (wave < 4) {
        // ---------------- value waves ----------------
        const int q = wave, n = lane & 15, g = lane >> 4, col = 16 * q + n;
        Tg *gv = reinterpret_cast<Tg *>(a.gv);
        const f32x4 zero = (f32x4){0.f, 0.f, 0.f, 0.f};
        const int lane_off = n * (int)C + 16 * q + 4 * g;   // outputs: token n of a half chunk, four channels
        f32x4 G[4];   // G[ib][e] = G[16ib+4g+e][col]
#pragma unroll
        for (int i = 0; i < 4; ++i) G[i] = zero;
        if (a.gsT) {
            const float *p = a.gsT + (int64_t)pair * (kN * kN) + col;
#pragma unroll
            for (int ib = 0; ib < 4; ++ib)
#pragma unroll
                for (int e = 0; e < 4; ++e) G[ib][e] = p[(16 * ib + 4 * g + e) * kN];
        }
        auto publish = [&]() {
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) *reinterpret_cast<f32x4 *>(&L.G[col][16 * ib + 4 * g]) = G[ib];
        };
        publish();
        __syncthreads();
        for (int s = 0; s < nchunk; ++s) {
            const int c = nchunk - 1 - s, buf = s & 1;
            const bool full = (c + 1) * kC32 <= T;
            // ---- phase 1: a tile of A (wave 0: (0,0), 1: (1,1), 2: (1,0)), K' G ----
            if (!kOnlyG && q < 3) {
                const int tb = q == 0 ? 0 : 1, sb = q == 1 ? 1 : 0;
                f32x4 at = zero;
#pragma unroll
                for (int ib = 0; ib < 4; ++ib) {
                    const int i0 = 16 * ib + 4 * g;
                    const f32x4 fk = *reinterpret_cast<const f32x4 *>(&L.Kp[buf][16 * sb + n][i0]) *
                                     *reinterpret_cast<const f32x4 *>(&L.inv1[buf][i0]);
                    const f32x4 fr = *reinterpret_cast<const f32x4 *>(&L.Rp[buf][16 * tb + n][i0]) *
                                     *reinterpret_cast<const f32x4 *>(&L.inv0[buf][i0]);
                    at = mfma16(fk, fr, at);
                }
                if (tb == sb) {
                    const int t = 16 * tb + n;
                    const float diag = (L.ruk[buf][0][t] + L.ruk[buf][1][t]) + (L.ruk[buf][2][t] + L.ruk[buf][3][t]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) at[e] = (4 * g + e < n) ? at[e] : (4 * g + e == n ? diag : 0.f);
                }
                *reinterpret_cast<f32x4 *>(&L.A[16 * tb + n][16 * sb + 4 * g]) = at;
            }
            f32x4 gvt[2] = {zero, zero};
#pragma unroll
            for (int sb = 0; !kOnlyG && sb < 2; ++sb)
#pragma unroll
                for (int ib = 0; ib < 4; ++ib) {
                    const f32x4 fk = *reinterpret_cast<const f32x4 *>(&L.Kp[buf][16 * sb + n][16 * ib + 4 * g]);
                    gvt[sb] = mfma16(G[ib], fk, gvt[sb]);   // transposed: lane (n, g) gets token n, channels 4g ..
                }
            __syncthreads();
            // ---- phase 2: gv += A^T gy, out ; G <- e^{c_32} o G + R'^T gy ----
            f32x4 gyb[2];   // element e: token 16x + 4g + e, channel col
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) gyb[x][e] = L.GY[buf][16 * x + 4 * g + e][col];
#pragma unroll
            for (int sb = 0; !kOnlyG && sb < 2; ++sb)
#pragma unroll
                for (int tb = sb; tb < 2; ++tb) {
                    f32x4 fat;
#pragma unroll
                    for (int e = 0; e < 4; ++e) fat[e] = L.A[16 * tb + 4 * g + e][16 * sb + n];
                    gvt[sb] = mfma16(gyb[tb], fat, gvt[sb]);
                }
            if (!kOnlyG) {
                Tg *const out = gv + base + (int64_t)c * kC32 * C;   // (uniform; the lane's part of the address is lane_off)
                const int left = T - c * kC32 - n;                     // (token 16 x + n exists: 16 x < left)
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    if (full || 16 * x < left) store4(out + 16 * x * C + lane_off, gvt[x][0], gvt[x][1], gvt[x][2], gvt[x][3]);
            }
#pragma unroll
            for (int ib = 0; ib < 4; ++ib) {
                G[ib] *= *reinterpret_cast<const f32x4 *>(&L.e_all[buf][16 * ib + 4 * g]);
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) {
                    f32x4 fra;
#pragma unroll
                    for (int e = 0; e < 4; ++e) fra[e] = L.Rp[buf][16 * tb + 4 * g + e][16 * ib + n];
                    G[ib] = mfma16(fra, gyb[tb], G[ib]);
                }
            }
            if (!kOnlyG) publish();
            __syncthreads();
        }
        if (a.gs0) {   // what is left after the first chunk is dL/dS_0
            float *p = a.gs0 + (int64_t)pair * (kN * kN) + col;
#pragma unroll
            for (int ib = 0; ib < 4; ++ib)
#pragma unroll
                for (int e = 0; e < 4; ++e) p[(16 * ib + 4 * g + e) * kN] = G[ib][e];
        }
    } else if (kOnlyG) {
        __syncthreads();   // (the barriers of the others)
        for (int s = 0; s < nchunk; ++s) { __syncthreads(); __syncthreads(); }
    } else {
        // ---------------- key waves ----------------
        const int q = wave - 4, n = lane & 15, g = lane >> 4, col = 16 * q + n;
        Tg *gr = reinterpret_cast<Tg *>(a.gr), *gk = reinterpret_cast<Tg *>(a.gk), *gw = reinterpret_cast<Tg *>(a.gw);
        const f32x4 zero = (f32x4){0.f, 0.f, 0.f, 0.f};
        const int ch = 16 * q + 4 * g;                // outputs: token n of a half chunk, channels ch .. ch+3
        const int lane_off = n * (int)C + ch;
        f32x4 St[4];   // St[jb][e] = S_0[col][16jb+4g+e]
        f32x4 E = zero, gu_acc = zero;   // of channels ch .. ch+3 (E the same in every lane of a row)
        if (a.gsT) {   // the anchor of the decay gradient's sums: E_T = sum_j S_T o G_T over the row
            const float *pg = a.gsT + (int64_t)pair * (kN * kN) + col * kN + 4 * g;
            const float *ps = a.sT + (int64_t)pair * (kN * kN) + col * kN + 4 * g;
            float part = 0.f;
#pragma unroll
            for (int jb = 0; jb < 4; ++jb) {
                const f32x4 gv = *reinterpret_cast<const f32x4 *>(pg + 16 * jb), sv = *reinterpret_cast<const f32x4 *>(ps + 16 * jb);
                part += (sv[0] * gv[0] + sv[1] * gv[1]) + (sv[2] * gv[2] + sv[3] * gv[3]);
            }
            part = sum_rows4(part);   // row `col`; lane n of every row of lanes
#pragma unroll
            for (int e = 0; e < 4; ++e) E[e] = __shfl(part, 4 * g + e);
        }
        float fu[4];
        load4(u + h * kN + ch, fu);
        // S_0^T from the forward's fragment order: S[i][j] sits in tile (j / 16, i / 16) at lane (j % 16) + 16 ((i % 16) / 4), element i % 4
        auto load_state = [&](int c) {
            const float *p0 = ck + (int64_t)c * (kN * kN) + (q * 64 + 4 * g + 16 * (n >> 2)) * 4 + (n & 3);
#pragma unroll
            for (int jb = 0; jb < 4; ++jb)
#pragma unroll
                for (int e = 0; e < 4; ++e) St[jb][e] = p0[jb * 1024 + e * 4];
        };
        const int lowest = a.s0 ? 0 : 1;   // the state before a sequence's first token is zero where none is given
        auto next_state = [&](int c) {     // the state of chunk c - 1, where there is one
            if (c > lowest) load_state(c - 1);
            else {
#pragma unroll
                for (int jb = 0; jb < 4; ++jb) St[jb] = zero;
            }
        };
        next_state(nchunk);
        __syncthreads();
        for (int s = 0; s < nchunk; ++s) {
            const int c = nchunk - 1 - s, buf = s & 1;
            const bool full = (c + 1) * kC32 <= T;
            // ---- phase 1: a tile of B (wave 0: (0,0), 1: (1,1), 3: (1,0)), v G^T ----
            if (q != 2) {
                const int tb = q == 0 ? 0 : 1, sb = q == 1 ? 1 : 0;
                f32x4 bt = zero;
#pragma unroll
                for (int jb = 0; jb < 4; ++jb) {
                    const f32x4 fv = *reinterpret_cast<const f32x4 *>(&L.V[buf][16 * sb + n][16 * jb + 4 * g]);
                    const f32x4 fg = *reinterpret_cast<const f32x4 *>(&L.GY[buf][16 * tb + n][16 * jb + 4 * g]);
                    bt = mfma16(fv, fg, bt);
                }
                if (tb == sb) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (4 * g + e == n) L.vgy[16 * tb + n] = bt[e];
                        bt[e] = (4 * g + e < n) ? bt[e] : 0.f;
                    }
                }
                *reinterpret_cast<f32x4 *>(&L.Bm[16 * tb + n][16 * sb + 4 * g]) = bt;
            }
            f32x4 Z[2] = {zero, zero}, W[2] = {zero, zero};
#pragma unroll
            for (int jb = 0; jb < 4; ++jb) {
                f32x4 gt;   // G[col][16jb+4g+e]
#pragma unroll
                for (int e = 0; e < 4; ++e) gt[e] = L.G[16 * jb + 4 * g + e][col];
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const f32x4 fv = *reinterpret_cast<const f32x4 *>(&L.V[buf][16 * x + n][16 * jb + 4 * g]);
                    W[x] = mfma16(gt, fv, W[x]);   // transposed: lane (n, g) gets token n, channels ch ..
                }
            }
            const float inv0 = L.inv0[buf][col], inv1 = L.inv1[buf][col];
            // the products with B come scaled from the middle of the chunk: bring these to that scale, all back at the end
            const f32x4 e_mid = *reinterpret_cast<const f32x4 *>(&L.e_mid[buf][ch]), e_rest = *reinterpret_cast<const f32x4 *>(&L.e_rest[buf][ch]);
#pragma unroll
            for (int x = 0; x < 2; ++x) W[x] *= e_rest;
            __syncthreads();
            // ---- phase 2: gy S_0^T, the products with B, the gradients ----
#pragma unroll
            for (int x = 0; x < 2; ++x) {
#pragma unroll
                for (int jb = 0; jb < 4; ++jb) {
                    const f32x4 fg = *reinterpret_cast<const f32x4 *>(&L.GY[buf][16 * x + n][16 * jb + 4 * g]);
                    Z[x] = mfma16(St[jb], fg, Z[x]);
                }
                Z[x] *= e_mid;
            }
            next_state(c);
            f32x4 rp[2], kp[2];   // R', K'; element e: token 16x + 4g + e, channel col
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = 16 * x + 4 * g + e;
                    rp[x][e] = L.Rp[buf][t][col];
                    kp[x][e] = L.Kp[buf][t][col];
                }
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int sb = 0; sb <= tb; ++sb) {
                    const f32x4 fb = *reinterpret_cast<const f32x4 *>(&L.Bm[16 * tb + n][16 * sb + 4 * g]);
                    Z[tb] = mfma16(kp[sb] * inv1, fb, Z[tb]);
                }
#pragma unroll
            for (int sb = 0; sb < 2; ++sb)
#pragma unroll
                for (int tb = sb; tb < 2; ++tb) {
                    f32x4 fbt;
#pragma unroll
                    for (int e = 0; e < 4; ++e) fbt[e] = L.Bm[16 * tb + 4 * g + e][16 * sb + n];
                    W[sb] = mfma16(rp[tb] * inv0, fbt, W[sb]);
                }
            // gradients out, lane = token 16x + n, four channels: whole 16-byte pieces of the operand tiles and of the
            // gradients (with lane = channel a wave sent twelve times the store instructions, four bytes a lane)
            f32x4 zt[2], kgk[2];
            const f32x4 row0 = *reinterpret_cast<const f32x4 *>(&L.inv0[buf][ch]), row1 = *reinterpret_cast<const f32x4 *>(&L.inv1[buf][ch]);
            const int64_t out0 = base + (int64_t)c * kC32 * C;   // (uniform; the lane's part of the address is lane_off)
            const int left = T - c * kC32 - n;                   // (token 16 x + n exists: 16 x < left)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int t = 16 * x + n;
                const f32x4 rt = *reinterpret_cast<const f32x4 *>(&L.R[t][ch]), kt = *reinterpret_cast<const f32x4 *>(&L.K[t][ch]);
                const f32x4 f1 = *reinterpret_cast<const f32x4 *>(&L.F1[t][ch]), f3 = *reinterpret_cast<const f32x4 *>(&L.F3[t][ch]);
                const float vg = L.vgy[t];
                Z[x] *= row0;
                W[x] *= row1;
                f32x4 o_r, o_k;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o_r[e] = fmaf(f1[e], Z[x][e], fu[e] * kt[e] * vg);
                    o_k[e] = fmaf(f3[e], W[x][e], fu[e] * rt[e] * vg);
                    kgk[x][e] = kt[e] * f3[e] * W[x][e];
                    zt[x][e] = fmaf(rt[e] * f1[e], Z[x][e], -kgk[x][e]);
                    gu_acc[e] = fmaf(rt[e] * kt[e], vg, gu_acc[e]);
                }
                if (full || 16 * x < left) {
                    store4(gr + out0 + 16 * x * C + lane_off, o_r[0], o_r[1], o_r[2], o_r[3]);
                    store4(gk + out0 + 16 * x * C + lane_off, o_k[0], o_k[1], o_k[2], o_k[3]);
                }
            }
            // E_{t+1} = E at the chunk's end + what the later tokens of the chunk add
#pragma unroll
            for (int x = 1; x >= 0; --x) {
                const f32x4 d = *reinterpret_cast<const f32x4 *>(&L.D[16 * x + n][ch]);
                f32x4 o_w;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float from_here = row_sum_down(zt[x][e]);
                    o_w[e] = (E[e] + next_in_row(from_here) - kgk[x][e]) * d[e];
                    E[e] += first_of_row(from_here);
                }
                // (a zero initial state: the first decay reaches no output, its gradient is zero and not
                // what rounding leaves of two equal sums)
                if (x == 0 && first_row && c == 0 && n == 0) o_w = zero;
                if (last_row && c == nchunk - 1 && c * kC32 + 16 * x + n == T - 1) o_w = zero;   // (nor does the last one of a sequence in segments)
                if (full || 16 * x < left) store4(gw + out0 + 16 * x * C + lane_off, o_w[0], o_w[1], o_w[2], o_w[3]);
            }
            __syncthreads();
        }
        // gu: the lanes of a row hold the tokens n (mod 16) of every chunk
#pragma unroll
        for (int e = 0; e < 4; ++e) gu_acc[e] = row_sum16(gu_acc[e]);
        if (n < 4) {
            const float x = n == 0 ? gu_acc[0] : n == 1 ? gu_acc[1] : n == 2 ? gu_acc[2] : gu_acc[3];
            store1(reinterpret_cast<Tout *>(a.gu) + (int64_t)b * C + h * kN + ch + n, x);
            s_gu[ch + n] = x;
        }
    }
    __syncthreads();
    // a pair whose decay left the reach: once more, one timestep at a time (the pair's slice of the saved
    // states, T/32 x 64 x 64 floats, is large enough for the T x 64 workspace of that pass behind the first chunk's state,
    // whose place may hold parts and counters)
    __shared__ float s_ft[kN];
    if (L.wild[0] | L.wild[1] | L.wild[2] | L.wild[3]) {
        const int64_t so = (int64_t)pair * (kN * kN);
        const float *s0p = a.s0 && !first_row ? a.s0 + so : nullptr, *gsTp = a.gsT && !last_row ? a.gsT + so : nullptr;
        float *gs0p = a.gs0 ? a.gs0 + so : nullptr;
        float *const wsP = ck + kN * kN;
        const bool states = s0p || gsTp || gs0p;
        __syncthreads();
        scan_bwd_a_body<Tin, Tout>(reinterpret_cast<C32BwdSmem *>(c32_smem)->scan_a, b, h, T, H, r, k, v, w, u, gy,
                                   reinterpret_cast<Tg *>(a.gr), reinterpret_cast<Tout *>(a.gu), wsP, kN,
                                   s0p, gsTp, states ? s_ft : nullptr);
        __threadfence_block();
        __syncthreads();
        scan_bwd_b_body<Tin, Tout>(reinterpret_cast<C32BwdSmem *>(c32_smem)->scan_b, b, h, T, H, r, k, v, w, u, gy, wsP, kN,
                                   reinterpret_cast<Tg *>(a.gk), reinterpret_cast<Tg *>(a.gv), reinterpret_cast<Tg *>(a.gw),
                                   gsTp, states ? s_ft : nullptr, gs0p, s0p == nullptr);
        __threadfence_block();
        __syncthreads();
        if (wave == 8) s_gu[lane] = reinterpret_cast<const Tout *>(a.gu)[(int64_t)b * C + h * kN + lane];
    }
    if (kOnlyG) return;
    // (these arguments are read anew from the argument block: kept in scalar registers across the chunks they spill others that
    // the loops use)
    const C32BwdArgs __attribute__((address_space(4))) *z = (const C32BwdArgs __attribute__((address_space(4))) *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(z));
    if (z->parts == nullptr) return;
    __shared__ int s_last;
    const int rows = (int)gridDim.x / H;
    if (wave == 8) {   // (a loading wave: it has no stores of gradients to wait for)
        __hip_atomic_store(z->parts + b * z->part_row + h * z->part_head + lane, s_gu[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (written before it is counted)
        if (lane == 0) s_last = __hip_atomic_fetch_add(z->arrivals + h * z->arrival_step, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == rows - 1;
    }
    __syncthreads();
    if (!s_last) return;
    // the last workgroup of the head: rows of a sequence first (one each without segments), then the sequences
    float *part = reinterpret_cast<float *>(c32_smem), *first = z->parts + h * z->part_head;
    const int per = z->P ? z->P : rows;
    float sum = 0.f;
    for (int s = 0; s < rows / per; ++s) {
        const float one = sum_partial_rows<12>(first + (int64_t)s * per * z->part_row, z->part_row, per, part, wave, lane);
        if (z->P && tid < kN) z->gu_seq[(int64_t)s * C + h * kN + tid] = one;
        sum += one;
        __syncthreads();
    }
    if (z->gu_sum && tid < kN) store1(reinterpret_cast<Tg *>(z->gu_sum) + h * kN + tid, sum);
    if (tid == 0) __hip_atomic_store(z->arrivals + h * z->arrival_step, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // armed again
}

template <typename Tin, typename Tout, typename Tg, bool kOnlyG>
static hipError_t launch(hipStream_t st, int64_t B, const C32BwdArgs &a) {
    constexpr int lds = (int)sizeof(C32BwdSmem);
    const hipError_t e = allow_dynamic_lds<chunk32_bwd_kernel<Tin, Tout, Tg, kOnlyG>>(lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((chunk32_bwd_kernel<Tin, Tout, Tg, kOnlyG>), dim3((unsigned)(B * a.H)), dim3(768), lds, st, a);
    return hipGetLastError();
}

hipError_t chunk32_backward(hipStream_t st, int dtype, int grad_dtype, int64_t B, int64_t T, int64_t H,
                            const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                            void *gr, void *gk, void *gv, void *gw, void *gu, void *saved_states,
                            const float *s0, const float *gsT, const float *sT, float *gs0, RowCut cut, bool only_gs0, void *gu_sum,
                            const C32Segments *seg)
{
    if (grad_dtype != kF32 && (grad_dtype != kF16 || dtype != kF16)) return hipErrorInvalidValue;
    if (gsT != nullptr && sT == nullptr) return hipErrorInvalidValue;   // (the anchor of the decay gradient needs S_T)
    C32BwdArgs a = {};
    if (seg) {
        a.P = seg->P; a.parts = seg->gu_rows; a.part_row = H * kN; a.part_head = kN;
        a.arrivals = seg->arrivals; a.arrival_step = 1;
        a.gu_sum = gu_sum; a.gu_seq = (float *)gu;
        gu = seg->gu_rows;
    } else if (gu_sum) {
        if (s0 || gsT || gs0) return hipErrorInvalidValue;   // (the first chunk's state is in use)
        const int64_t slice = (T + kC32 - 1) / kC32 * (kN * kN);
        a.parts = reinterpret_cast<float *>(saved_states) + kN; a.part_row = H * slice; a.part_head = slice;
        a.arrivals = reinterpret_cast<int *>(saved_states); a.arrival_step = slice;
        a.gu_sum = gu_sum;
    }
    a.cut = cut; a.slice = (int)((T + kC32 - 1) / kC32);
    a.s0 = s0; a.gsT = gsT; a.sT = sT; a.gs0 = gs0;
    a.T = (int)T; a.H = (int)H;
    a.r = r; a.k = k; a.v = v; a.w = w; a.u = u; a.gy = gy;
    a.gr = gr; a.gk = gk; a.gv = gv; a.gw = gw; a.gu = gu;
    a.saved = reinterpret_cast<float *>(saved_states);
    auto pick = [&](auto only) -> hipError_t {
        constexpr bool kOnlyG = decltype(only)::value;
        if (dtype == kF32) return launch<float, float, float, kOnlyG>(st, B, a);
        return grad_dtype == kF16 ? launch<f16_t, float, f16_t, kOnlyG>(st, B, a) : launch<f16_t, float, float, kOnlyG>(st, B, a);
    };
    return only_gs0 ? pick(std::true_type{}) : pick(std::false_type{});
}

hipError_t chunk32_backward_saved_segments(hipStream_t st, int dtype, int grad_dtype, int64_t B, int64_t T, int64_t H,
                                           const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                                           void *gr, void *gk, void *gv, void *gw, void *gu, void *gu_sum, void *saved)
{
    const C32Segments s = chunk32_segments_layout(B, T, H, saved);
    const int64_t rows = B * s.P;
    // what each segment alone sends back into its incoming state; the chain backwards in time; every segment between its
    // true incoming state and its true arriving gradient
    hipError_t e = chunk32_backward(st, dtype, grad_dtype, rows, s.L, H, r, k, v, w, u, gy, gr, gk, gv, gw, s.gu_rows, s.chunks,
                                    s.states, nullptr, nullptr, s.gstates, s.cut, true);
    if (e != hipSuccess) return e;
    if ((e = segment_chain_factors(st, s.P, B, H, s.decay, s.gstates, true)) != hipSuccess) return e;
    return chunk32_backward(st, dtype, grad_dtype, rows, s.L, H, r, k, v, w, u, gy, gr, gk, gv, gw, gu, s.chunks,
                            s.states, s.gstates, s.ends, nullptr, s.cut, false, gu_sum, &s);
}

}  // namespace wkv6
