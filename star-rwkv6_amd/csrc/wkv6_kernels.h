// Host-side launchers of the WKV6 kernels (internal to the library; the public ABI is include/wkv6.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

namespace wkv6 {

// Raises kernel Kern's dynamic-LDS limit to `bytes`, once per device (the setting is idempotent and
// per device; the flags below only save the runtime call on later launches).
template <auto Kern>
inline hipError_t allow_dynamic_lds(int bytes) {
    static std::atomic<bool> done[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const bool known = dev >= 0 && dev < 64;
    if (known && done[dev].load(std::memory_order_acquire)) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && known) done[dev].store(true, std::memory_order_release);
    return e;
}

enum { kBF16 = 0, kF16 = 1, kF32 = 2 };  // same numbering as the public header

// compute units of the current device (an immutable device property, looked up once per device)
int compute_units();

// --- per-timestep recurrence (wkv6_scan.hip) ---
hipError_t scan_forward(hipStream_t st, int dtype, int state_dtype, int64_t B, int64_t T, int64_t H,
                        const void *r, const void *k, const void *v, const void *w, const void *u,
                        const void *s0, const int64_t *map, void *y, void *sT);
size_t scan_backward_workspace_bytes(int64_t B, int64_t T, int64_t C);
hipError_t scan_backward(hipStream_t st, int dtype, int64_t B, int64_t T, int64_t H,
                         const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                         void *gr, void *gk, void *gv, void *gw, void *gu, void *workspace);

// --- head sizes other than 64, multiples of 4 up to 128 (wkv6_generic.hip): the per-timestep recurrence, one thread per channel; every
// dtype, states (B,H,N,N), state_map, gradients through the state (s0 / gsT / gs0 fp32, may be null)
bool generic_head_size(int64_t N);
hipError_t generic_forward(hipStream_t st, int dtype, int state_dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                           const void *r, const void *k, const void *v, const void *w, const void *u,
                           const void *s0, const int64_t *map, void *y, void *sT);
size_t generic_backward_workspace_bytes(int64_t B, int64_t T, int64_t C);
hipError_t generic_backward(hipStream_t st, int dtype, int64_t B, int64_t T, int64_t H, int64_t N,
                            const void *r, const void *k, const void *v, const void *w, const void *u,
                            const float *s0, const void *gy, const float *gsT,
                            void *gr, void *gk, void *gv, void *gw, void *gu, float *gs0, void *workspace);

// one timestep (T = 1) with the layer's output stage fused in (bf16 tensors), see chunk_forward_fused
hipError_t step_forward_fused(hipStream_t st, int state_dtype, int64_t B, int64_t H,
                              const void *r, const void *k, const void *v, const void *w, const void *u,
                              const void *s0, const int64_t *map, const void *gate, const float *gn_scale,
                              const float *gn_offset, float gn_eps, void *out, void *sT);

// with gradients through the state: S_0 = s0 (null = 0), G_T = gsT (null = 0), gs0 = dL/dS_0 (may be null);
// states are fp32 (B,H,64,64) [key][value]
size_t scan_backward_state_workspace_bytes(int64_t B, int64_t T, int64_t C);
hipError_t scan_backward_state(hipStream_t st, int dtype, int64_t B, int64_t T, int64_t H,
                               const void *r, const void *k, const void *v, const void *w, const void *u,
                               const float *s0, const void *gy, const float *gsT,
                               void *gr, void *gk, void *gv, void *gw, void *gu, float *gs0, void *workspace);

// Time segments as rows of a (B * segments, L, C) view.  Segments that do not divide the sequence evenly start at
// (row / segments) * total + (row % segments) * L and the last one of a sequence ends with it: `total` tokens,
// `segments` per sequence.  Zero segments: the rows are sequences of their own (or the segments divide evenly, which
// is the same thing).
struct RowCut {
    int segments = 0;
    int64_t total = 0;
};
// What a workgroup of one row makes of it at its start: its own number of tokens and the tokens its pointers move by, so that
// everything behind addresses row `row` of `tokens` tokens as ever (all of the workgroup's pairs lie in this row).
struct RowView {
    int tokens;
    int64_t shift;
};
__device__ __forceinline__ RowView row_view(const RowCut &cut, int row, int L) {
    const int b = row / cut.segments, s = row - b * cut.segments;
    const int64_t first = (int64_t)s * L, left = cut.total - first;
    const int tokens = left < L ? (int)left : L;
    return {tokens, b * cut.total + first - (int64_t)row * tokens};
}
template <typename P> __device__ __forceinline__ void move_rows(P *&p, int64_t elements) {
    if (p) p += elements;
}

// How the rows of a launch, the P segments of each sequence, come by the state they start from (the block-form kernels; the
// tile form and the full-precision form are handed the states by segment_chain_kernel): from what every segment leaves alone,
// started from zero, and the decay over it.
struct SegmentChain {
    int P = 0;                        // segments of a sequence (0: every row is a sequence of its own)
    const float *alone = nullptr;     // [rows][H][64][64] (fp32, [key][value])
    const float *decay = nullptr;     // [rows][H][64]
    bool given = false;               // forward: `start` of every sequence's first segment holds the state it starts from (otherwise zero)
    void *last = nullptr;             // forward: the sequences' final states [B][H][64][64], or null
    bool bf16 = false;                // `last` is bf16 (otherwise fp32)
    float *start = nullptr;           // [rows][H][64][64]: receives what every segment starts from
};

// The states the sequences start from, which the first pass leaves as fp32 in the place of the first segments' `start`: the second
// pass stores the final states, and a caller's final states may lie where the given ones do.
struct GivenStates {
    const void *states = nullptr;     // (n_state, H, 64, 64), or null: zero
    const int64_t *map = nullptr;     // batch row -> row of `states`, or null: the same
    bool bf16 = false;                // otherwise fp32
    int P = 1;                        // segments of a sequence
    float *start = nullptr;           // as in SegmentChain
};
// First pass over the segments (wkv6_state.hip, bf16): the state each row of at most L tokens builds from zero and the decay over it
// (may be null); reverse: the rows read back to front
hipError_t segment_states(hipStream_t st, int64_t rows, int64_t L, int64_t H, const void *k, const void *v, const void *w, const void *u,
                          float *states, float *decay, bool reverse, RowCut cut, const GivenStates &given = GivenStates(),
                          int P = 0);   // P: segments of a sequence, of which the last (reverse: the first) is not wanted (its decay is left as zero)

// --- chunk-parallel MFMA form, bf16 tensors only (wkv6_chunk.hip) ---
hipError_t chunk_forward(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                         const void *r, const void *k, const void *v, const void *w, const void *u,
                         const void *s0, const int64_t *map, void *y, void *sT, void *saved_states,
                         float *decay = nullptr,   // see FwdArgs
                         bool reverse = false,     // the time axis read back to front (no y)
                         bool counters = true,     // saved_states ends with the per-head counters of the fused gu sum (zeroed here)
                         RowCut cut = RowCut(), bool keep_inputs = false);   // keep_inputs: a backward will read them again

// --- block form (wkv6_block_fwd.hip, wkv6_block_bwd.hip): a 64-token chunk as one block of the
// recurrence; bf16 tensors, T a multiple of 64, between half a pair and one pair per compute unit.
// Same arguments and the same saved-state layout as the tile form above, which takes every other case.
// workgroups of a block-form launch (0: the shape is not taken)
int64_t block_grid(int64_t B, int64_t H);
bool block_forward_applies(int64_t B, int64_t T, int64_t H);
hipError_t block_forward(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                         const void *r, const void *k, const void *v, const void *w, const void *u,
                         const void *s0, const int64_t *map, void *y, void *sT, void *saved_states, bool counters,
                         RowCut cut = RowCut(), SegmentChain chain = SegmentChain(),   // (rows that are segments: cut and chain, s0 = map = sT = null)
                         bool keep_inputs = false);   // a backward will read them again

// The sums over tokens that the norm's backward will add up, (H, 64) each (null: none): the saving fused forward clears them, where the
// backward would need a launch of its own for it.
struct GnSums {
    float *scale = nullptr, *offset = nullptr;
};
// by the 64 lanes of one wave per head
__device__ __forceinline__ void clear_sums(const GnSums &s, int h, int lane) {
    if (s.scale) { s.scale[h * 64 + lane] = 0.f; s.offset[h * 64 + lane] = 0.f; }
}

// the block-form forward with the layer's output stage fused in (see chunk_forward_fused / chunk_forward_fused_save):
// y and stats may be null (inference), saved_states null without a backward to follow
hipError_t block_forward_fused(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                               const void *r, const void *k, const void *v, const void *w, const void *u,
                               const void *s0, const int64_t *map, const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps,
                               void *out, void *y, float *stats, void *sT, void *saved_states,
                               RowCut cut = RowCut(), SegmentChain chain = SegmentChain(), GnSums sums = GnSums());
bool block_backward_applies(int64_t B, int64_t T, int64_t H);
// workspace: the chunk-start states as a forward pass leaves them, followed by the per-head counters; gu_sum may be null
hipError_t block_backward(hipStream_t st, int64_t B, int64_t T, int64_t H,
                          const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                          void *gr, void *gk, void *gv, void *gw, void *gu, void *workspace, void *gu_sum,
                          const float *s0 = nullptr, const float *gsT = nullptr, float *gs0 = nullptr, RowCut cut = RowCut(),
                          float *gu_rows = nullptr,    // gu_rows: see chunk_backward; one pair per workgroup
                          // rows that are segments: gu (sequences, C) and gu_sum from all of them, gu_rows as scratch, gw zero at the
                          // ends of the sequences; s0 = what the forward's segments started from, gsT = gs0 = null
                          SegmentChain chain = SegmentChain());

// --- full-precision chunk form (wkv6_chunk32_fwd.hip, wkv6_chunk32_bwd.hip): fp32 and fp16 tensors on the
// fp32 matrix instructions, chunks of 32 tokens, fp32 states; any T (the last chunk may be short).
bool chunk32_forward_applies(int dtype, int64_t B, int64_t T, int64_t H);
size_t chunk32_saved_bytes(int64_t B, int64_t T, int64_t H);   // one fp32 state per chunk and pair
// saved_states (may be null): receives the chunk-start states for chunk32_backward; y may be null then
hipError_t chunk32_forward(hipStream_t st, int dtype, int state_dtype, int64_t B, int64_t T, int64_t H,
                           const void *r, const void *k, const void *v, const void *w, const void *u,
                           const void *s0, const int64_t *map, void *y, void *sT, void *saved_states,
                           float *decay = nullptr,   // [2][pair][64]: two factors of each row's decay
                           RowCut cut = RowCut(), int *arrivals = nullptr);   // arrivals: see C32FwdArgs

struct C32Segments;
// saved_states: what chunk32_forward left (the pair's slice also serves the per-timestep pass of a pair
// whose decay left the chunk form's reach); gu (B, C)
// grad_dtype: type of gr, gk, gv, gw: kF32, or kF16 for fp16 tensors
hipError_t chunk32_backward(hipStream_t st, int dtype, int grad_dtype, int64_t B, int64_t T, int64_t H,
                            const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                            void *gr, void *gk, void *gv, void *gw, void *gu, void *saved_states,
                            // gradients through the state ((B,H,64,64) fp32 [key][value]; sT = the forward's final state,
                            // needed with gsT); the saved states come from a forward that started from s0
                            const float *s0 = nullptr, const float *gsT = nullptr, const float *sT = nullptr, float *gs0 = nullptr,
                            RowCut cut = RowCut(), bool only_gs0 = false,   // only_gs0: nothing but gs0 is wanted
                            // gu_sum (may be null; without states): (C) in grad_dtype, the sum of gu over the batch
                            // seg: the rows are segments: gu (sequences, C) and gu_sum from all of them, gw zero at the sequences' ends
                            void *gu_sum = nullptr, const C32Segments *seg = nullptr);

// The training pair in time segments; what the forward leaves for the backward in `saved` (the first part as chunk32_forward).
struct C32Segments {
    int P;             // segments per sequence (1: does not apply)
    int64_t L;         // tokens of a segment (the last one of a sequence may be shorter)
    RowCut cut;
    float *chunks;     // chunk states of the segments
    float *states, *ends, *gstates;   // [B*P][H][64][64]: state entering and leaving each segment, gradient arriving at its end
    float *decay;      // [2][B*P][H][64]
    float *gu_rows;    // [B*P][C]
    int *arrivals;     // [H]
    size_t bytes;
};
int chunk32_train_segments(int64_t B, int64_t T, int64_t H, int64_t *L);
C32Segments chunk32_segments_layout(int64_t B, int64_t T, int64_t H, void *saved);
hipError_t chunk32_forward_save_segments(hipStream_t st, int dtype, int64_t B, int64_t T, int64_t H,
                                         const void *r, const void *k, const void *v, const void *w, const void *u,
                                         void *y, void *saved);
hipError_t chunk32_backward_saved_segments(hipStream_t st, int dtype, int grad_dtype, int64_t B, int64_t T, int64_t H,
                                           const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                                           void *gr, void *gk, void *gv, void *gw, void *gu, void *gu_sum, void *saved);

// fp16 tensors on the chunked kernels (training pair only: y and the gradients are fp32).  r, k, w stay
// fp16 (the kernels unpack them exactly); v and gy are consumed as bf16 MFMA operands, so the caller
// keeps bf16 copies of them (convert_to_bf16) next to the saved states.
hipError_t convert_to_bf16(hipStream_t st, int src_dtype, const void *src, void *dst, int64_t n);
hipError_t chunk_forward_save_f16(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                  const void *r, const void *k, const void *v, const void *v_bf16, const void *w, const void *u,
                                  void *y, void *saved_states);

// Few pairs, long sequence: the forward as P time segments side by side (two passes joined by the
// affine map of a segment's state).  The workspace's size is 0 where that does not apply to the shape.
// fused: with the output stage; any_length: batches of a length that does not divide evenly, too
size_t chunk_forward_segments_workspace_bytes(int64_t B, int64_t T, int64_t H, bool fused, bool any_length);
hipError_t chunk_forward_segments_run(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                                      const void *r, const void *k, const void *v, const void *w, const void *u,
                                      const void *s0, const int64_t *map, void *y, void *sT, void *workspace, bool any_length,
                                      const void *gate = nullptr, const float *gn_scale = nullptr,
                                      const float *gn_offset = nullptr, float gn_eps = 0.f);

// The training pair of a long sequence of few pairs as P time segments side by side.  The saving
// forward leaves, behind the saved chunk states (`extra`), every segment's incoming state and decay
// exponents; the backward chains its reverse state through the same affine maps (two passes each).
struct TrainSegments {
    int P;              // segments per sequence (1: does not apply)
    int64_t L;          // tokens of a segment (the last one of a sequence may be shorter)
    RowCut cut;         // how the kernels find them
    float *states;      // [B*P][H][64][64] state entering each segment
    float *decay;       // [B*P][H][64] decay over each segment
    float *gstates;     // [B*P][H][64][64] gradient arriving at the end of each segment
    float *gu_rows;     // [B*P][C] gu of each segment
    float *alone;       // [B*P][H][64][64] (training pair in block form) what each segment leaves alone, forward or backward in time
    size_t bytes_unsaved;   // size of the block without `alone` (a backward without saved states)
    size_t bytes;       // size of the block
};
int chunk_train_segments(int64_t B, int64_t T, int64_t H);
TrainSegments train_segments_layout(int64_t B, int64_t T, int64_t H, void *extra);
// states[(b*P + seg), h]: on entry what each segment builds alone, on exit what enters it (forward: the
// state, from s0 or zero; reverse: the gradient arriving at its end, from `arriving` or zero, and
// `leaving` receives what leaves the first segment, dL/dS_0).
hipError_t segment_chain_forward(hipStream_t st, int P, int64_t B, int64_t H, const float *decay, float *states, const float *s0);
// the same with the segments' decays as two factors each, [2][B*P][H][64]
hipError_t segment_chain_factors(hipStream_t st, int P, int64_t B, int64_t H, const float *decay, float *states, bool reverse);
int plan_segments(int64_t pairs, int64_t T, int64_t least, int64_t *L);
bool segments_in_block_form(int64_t rows, int64_t H);   // the form of the second pass of the bf16 pair and of prompts
RowCut cut_of(int P, int64_t L, int64_t T);
hipError_t segment_chain_reverse(hipStream_t st, int P, int64_t B, int64_t H, const float *decay, float *states,
                                 const float *arriving = nullptr, float *leaving = nullptr);
hipError_t chunk_backward_state_segments(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                         const void *r, const void *k, const void *v, const void *w, const void *u,
                                         const float *s0, const void *gy, const float *gsT,
                                         void *gr, void *gk, void *gv, void *gw, void *gu, float *gs0,
                                         void *saved, void *extra);
hipError_t chunk_forward_save_segments(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                       const void *r, const void *k, const void *v, const void *w, const void *u,
                                       void *y, void *saved, void *extra);
hipError_t chunk_backward_saved_segments(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                         const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                                         void *gr, void *gk, void *gv, void *gw, void *gu, void *gu_sum,
                                         void *saved, void *extra);

// forward with the layer's output stage fused in: out = (group_norm_head(y) * gn_scale + gn_offset) * gate
hipError_t chunk_forward_fused(hipStream_t st, int state_dtype, int64_t B, int64_t T, int64_t H,
                               const void *r, const void *k, const void *v, const void *w, const void *u,
                               const void *s0, const int64_t *map, const void *gate, const float *gn_scale,
                               const float *gn_offset, float gn_eps, void *out, void *sT, RowCut cut = RowCut());

// The same for training: also writes y (bf16), the norm's statistics (B,T,H,2: mean, rstd) and the chunk states
hipError_t chunk_forward_fused_save(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                    const void *r, const void *k, const void *v, const void *w, const void *u,
                                    const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps,
                                    void *out, void *y, float *stats, void *saved_states, GnSums sums);
// ... of a shape whose training pair runs in time segments (saved / extra as in chunk_forward_save_segments)
hipError_t chunk_forward_fused_save_segments(hipStream_t st, int64_t B, int64_t T, int64_t H,
                                             const void *r, const void *k, const void *v, const void *w, const void *u,
                                             const void *gate, const float *gn_scale, const float *gn_offset, float gn_eps,
                                             void *out, void *y, float *stats, void *saved, void *extra, GnSums sums);
// backward of the output stage (wkv6_gn.hip): bf16 tensors, gscale / goffset fp32 (C), zeroed inside unless they are `cleared`
hipError_t gn_gate_backward(hipStream_t st, int64_t B, int64_t T, int64_t H,
                            const void *gout, const void *y, const float *stats, const void *gate,
                            const float *scale, const float *offset, void *gy, void *ggate, float *gscale, float *goffset, bool cleared);

// input side of the time-mix layer (wkv6_mix.hip): token shift and the five low-rank mixers, bf16 tensors,
// rank R in {32, 64}.  h (B,T,5,R), w2t (5,C,R), bias (5,C) and mix_x (C) fp32.
bool shift_mix_supported(int64_t C, int64_t R);
hipError_t shift_mix_x(hipStream_t st, int64_t B, int64_t T, int64_t C, const void *x, const float *mix_x, void *x_mix);
hipError_t shift_mix_five(hipStream_t st, int64_t B, int64_t T, int64_t C, int64_t R, const void *x, const void *h,
                          const void *w2t, const float *bias, void *const out[5]);
// gcoef: five (B,T,C) planes gcoef_stride elements apart; gp and gxx (B,T,C)
hipError_t shift_mix_five_backward(hipStream_t st, int64_t B, int64_t T, int64_t C, int64_t R, const void *x, const void *h,
                                   const void *w2t, const float *bias, const void *const gout[5], void *gcoef, int64_t gcoef_stride,
                                   void *gp, void *gxx);
// gx (B,T,C), gmix_x (C) fp32, zeroed inside
hipError_t shift_mix_x_backward(hipStream_t st, int64_t B, int64_t T, int64_t C, const void *x, const float *mix_x,
                                const void *gp, const void *gxx, const void *gxm, void *gx, float *gmix_x);

// the whole input side with its products (wkv6_mix_train.hip); a (5R,C), w2t (5,C,R) and their gradients in weight_dtype
// (kBF16 or kF32); `weights` receives the forms the kernels read and is handed to the backward with h
size_t shift_mix_weights_bytes(int64_t C, int64_t R);
hipError_t shift_mix_forward(hipStream_t st, int weight_dtype, int64_t B, int64_t T, int64_t C, int64_t R, const void *x, const float *mix_x,
                             const void *a, const void *w2t, const float *bias, void *weights, void *h, void *const out[5]);
size_t shift_mix_backward_workspace_bytes(int64_t B, int64_t T, int64_t C, int64_t R);
hipError_t shift_mix_backward(hipStream_t st, int weight_dtype, int64_t B, int64_t T, int64_t C, int64_t R, const void *x, const float *mix_x,
                              const float *bias, const void *weights, const void *h, const void *const gout[5],
                              void *gx, float *gmix_x, void *ga, void *gw2t, float *gbias, void *workspace);

size_t chunk_backward_workspace_bytes(int64_t B, int64_t T, int64_t H);
// bytes of a forward -> backward hand-over buffer: the workspace plus one arrival counter per head
// (zeroed by the saving forward, used by the backward's fused batch sum of gu)
size_t chunk_saved_bytes(int64_t B, int64_t T, int64_t H);
// states_ready: the workspace already holds the chunk-start states (written by a forward pass).
// gu_sum (may be null; needs states_ready and a buffer of chunk_saved_bytes): also write sum_b gu[b].
hipError_t chunk_backward(hipStream_t st, int64_t B, int64_t T, int64_t H,
                          const void *r, const void *k, const void *v, const void *w, const void *u, const void *gy,
                          void *gr, void *gk, void *gv, void *gw, void *gu, void *workspace, bool states_ready,
                          void *gu_sum, const float *s0 = nullptr, const float *gsT = nullptr, float *gs0 = nullptr,
                          int in_dtype = kBF16, const void *v_orig = nullptr, const void *gy_orig = nullptr, RowCut cut = RowCut(),
                          float *gu_rows = nullptr);   // (B, C): takes every row's gu unrounded, in the place of gu
// s0 / gsT / gs0: gradients through the state, as in scan_backward_state (with states_ready = false)
// in_dtype kF16 (needs states_ready): r, k, w, u fp16, v and gy their bf16 copies, v_orig / gy_orig the
// caller's fp16 v and fp32 gy, gradients fp32

// sum over the batch of (B, C) partials -> (C), both in the output type (for the paths without a fused sum)
hipError_t sum_over_batch(hipStream_t st, int out_dtype, int64_t B, int64_t C, const void *partials, void *sum);

}  // namespace wkv6
