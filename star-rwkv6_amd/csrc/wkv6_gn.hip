// Backward of the layer's output stage  out = (group_norm_head(y) * scale + offset) * gate  (the forward
// half is fused into the chunked forward kernel, wkv6_chunk_fwd.hip).  group_norm_head is the layer
// norm over one head's 64 channels of one token (rwkv6_model.py:94-99), `* gate` is rwkv6_model.py:158-160.
//
//   z = (y - mean) rstd,  n = z scale + offset,  out = n gate
//   ggate = gout n,  gn = gout gate,  goffset += gn,  gscale += gn z,  gz = gn scale
//   gy = rstd (gz - mean_c(gz) - z mean_c(gz z))          (means over the head's 64 channels)
//
// Bound by memory: three 16-bit tensors in, two out.  A wave takes 512 neighbouring channels (8 heads) of a token at a
// time, a lane 8 of them: every access is 16 bytes per lane and 1 KiB per wave, a head's sums are folds over 8 lanes, and
// a lane's channels stay the same over all its tokens, so the sums for scale and offset stay in registers.  Four tokens'
// rows are in flight per wave.  What is not read again soon (gout, y, gate, ggate) goes past the caches, gy is the next
// kernel's input (the gate's own backward, which reads ggate next, takes as long with it in the caches: within 3 % either way from 256 to 16384
// tokens of H32).  B8 T1024 H32, 168 MB: 31 us = 5.5 TB/s behind the forward that
// wrote y, 41 us with nothing of it cached (one head per wave, 2 bytes per lane: 49 and 55 us).
// The sums are added up by one atomic operation per channel and workgroup, onto what the forward cleared (GnSums) or, without it, a kernel
// ahead of this one (2 to 5 us and a launch: forward and backward B8 T1024 H32 167.4 / 164.1, of host time at small sizes 99 / 95).
#include "wkv6_common.h"
#include "wkv6_kernels.h"

namespace wkv6 {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kGnWaves = 4, kGnTokens = 4;   // waves per workgroup (on different tokens), tokens a wave works on at once

__device__ __forceinline__ float sum_lanes8(float x) {   // over the 8 lanes that hold one head
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xF, 0xF, true));   // row_half_mirror
    return x;
}
__device__ __forceinline__ void unpack_pairs(const u32x4 &a, float (&o)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) { o[2 * i] = __uint_as_float(a[i] << 16); o[2 * i + 1] = __uint_as_float(a[i] & 0xffff0000u); }
}
__device__ __forceinline__ u32x4 pack_pairs(const float (&v)[8]) {
    return (u32x4){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}

__global__ __launch_bounds__(kGnWaves * 64) void gn_gate_bwd_kernel(int64_t n_tok, int C, int columns,
        const bf16_t *__restrict__ gout, const bf16_t *__restrict__ y, const float *__restrict__ stats,
        const bf16_t *__restrict__ gate, const float *__restrict__ scale, const float *__restrict__ offset,
        bf16_t *__restrict__ gy, bf16_t *__restrict__ ggate, float *__restrict__ gscale, float *__restrict__ goffset)
{
    __shared__ float fold[2][kGnWaves][512];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = (int)(blockIdx.x % columns) * 512 + 8 * lane, H = C / kN;
    const int64_t part = (int64_t)(blockIdx.x / columns) * kGnWaves + wave, nparts = (int64_t)(gridDim.x / columns) * kGnWaves;
    float acc_s[8], acc_o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc_s[i] = acc_o[i] = 0.f;
    if (c < C) {
        float sc[8], of[8];
        Raw8<float> v;
        v.load(scale + c); v.to_float(sc);
        v.load(offset + c); v.to_float(of);
        auto row = [](const bf16_t *p, size_t e) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p + e)); };
        for (int64_t t0 = part * kGnTokens; t0 < n_tok; t0 += nparts * kGnTokens) {
            u32x4 rg[kGnTokens], ry[kGnTokens], ra[kGnTokens];
            float2 st[kGnTokens];
#pragma unroll
            for (int j = 0; j < kGnTokens; ++j) {
                const int64_t t = t0 + j < n_tok ? t0 + j : n_tok - 1;
                const size_t e = (size_t)t * C + c;
                rg[j] = row(gout, e); ry[j] = row(y, e); ra[j] = row(gate, e);
                st[j] = *reinterpret_cast<const float2 *>(stats + ((size_t)t * H + c / kN) * 2);
            }
#pragma unroll
            for (int j = 0; j < kGnTokens; ++j) {
                if (t0 + j >= n_tok) break;
                const size_t e = (size_t)(t0 + j) * C + c;
                float go[8], z[8], ga[8], n[8];
                unpack_pairs(rg[j], go); unpack_pairs(ry[j], z); unpack_pairs(ra[j], ga);
                float m1 = 0.f, m2 = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    z[i] = (z[i] - st[j].x) * st[j].y;
                    n[i] = go[i] * fmaf(z[i], sc[i], of[i]);
                    const float gn = go[i] * ga[i];
                    acc_o[i] += gn;
                    acc_s[i] = fmaf(gn, z[i], acc_s[i]);
                    ga[i] = gn * sc[i];                 // gz
                    m1 += ga[i];
                    m2 = fmaf(ga[i], z[i], m2);
                }
                __builtin_nontemporal_store(pack_pairs(n), reinterpret_cast<u32x4 *>(ggate + e));
                m1 = sum_lanes8(m1) * (1.f / kN);
                m2 = sum_lanes8(m2) * (1.f / kN);
#pragma unroll
                for (int i = 0; i < 8; ++i) n[i] = st[j].y * (ga[i] - m1 - z[i] * m2);
                *reinterpret_cast<u32x4 *>(gy + e) = pack_pairs(n);
            }
        }
    }
    // one addition per channel and workgroup
#pragma unroll
    for (int i = 0; i < 8; ++i) { fold[0][wave][8 * lane + i] = acc_s[i]; fold[1][wave][8 * lane + i] = acc_o[i]; }
    __syncthreads();
    for (int i = threadIdx.x; i < 1024; i += kGnWaves * 64) {
        const int which = i >> 9, ch = (int)(blockIdx.x % columns) * 512 + (i & 511);
        if (ch >= C) continue;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < kGnWaves; ++w) s += fold[which][w][i & 511];
        atomicAdd((which ? goffset : gscale) + ch, s);
    }
}

__global__ void zero2_kernel(int n, float *a, float *b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { a[i] = 0.f; b[i] = 0.f; }
}

hipError_t gn_gate_backward(hipStream_t st, int64_t B, int64_t T, int64_t H,
                            const void *gout, const void *y, const float *stats, const void *gate,
                            const float *scale, const float *offset, void *gy, void *ggate, float *gscale, float *goffset, bool cleared)
{
    const int C = (int)(H * kN);
    // (a fill kernel rather than a memset node: the call may be captured in a HIP graph)
    if (!cleared) hipLaunchKernelGGL(zero2_kernel, dim3((unsigned)((C + 255) / 256)), dim3(256), 0, st, C, gscale, goffset);
    const int64_t n = B * T;
    const int columns = (C + 511) / 512;
    // as many workgroups as the chip holds at once (four of four waves per compute unit; two or eight: the same time), fewer where tokens run out
    int64_t parts = (n + kGnWaves * kGnTokens - 1) / (kGnWaves * kGnTokens);
    const int64_t cap = ((int64_t)compute_units() * 4 + columns - 1) / columns;
    if (parts > cap) parts = cap;
    hipLaunchKernelGGL(gn_gate_bwd_kernel, dim3((unsigned)(columns * parts)), dim3(kGnWaves * 64), 0, st, n, C, columns,
                       (const bf16_t *)gout, (const bf16_t *)y, stats, (const bf16_t *)gate, scale, offset,
                       (bf16_t *)gy, (bf16_t *)ggate, gscale, goffset);
    return hipGetLastError();
}

}  // namespace wkv6
