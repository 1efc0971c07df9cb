// wm_prefill.h -- arguments of the batched prefill kernels (wm_prefill.hip).
// Internal; not part of the public ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wm_format.h"

namespace wm {

// A (token, slot) pair p = t * K + k is one routed use of an expert; pair
// T * K + t is token t's use of the shared expert.
struct PrefillArgs {
    int32_t H, I, Is, E, K, T, has_shared;      // Is: 0 without a shared expert
    int32_t gt, dt, sgt, sdt;   // weight formats: routed gate = up, down; shared gate = up, down
    const uint16_t* x;          // bf16 [T][H]
    const float* router;        // fp32 [E][H]
    const uint8_t* gate;
    const uint8_t* up;
    const uint8_t* down;
    int64_t gstride, ustride, dstride;
    const uint8_t* sh_gate;
    const uint8_t* sh_up;
    const uint8_t* sh_down;
    const float* sh_gate_inp;   // fp32 [H] or NULL
    int32_t* ids;               // [T][K]
    float* w;                   // [T][K]
    float* logits;              // [T][E]
    uint32_t* hits;             // [E]
    int32_t* status;
    int32_t* sorted;            // [T * K + T] pair indices grouped by expert (batches that outgrow k_pf_group's LDS)
    int32_t* passes;            // [prefill_max_passes][64] pass records (up to pass_m pairs of one expert)
    int32_t* pass_count;        // [2]: routed passes, shared passes
    uint16_t* x16;              // fp16 [T][H]: x * 2^-e per token
    int32_t* xexp;              // [T]: e
    uint16_t* act_hi;           // fp16 [pairs][act_stride]: SwiGLU output = (hi + lo) * 2^e per (pair, 128 rows)
    uint16_t* act_lo;
    float* act_sc;              // [pairs][act_stride / 128]: 2^e
    int64_t act_stride;
    float* y;                   // [pairs][H] expert outputs
    float* sg;                  // [T] shared-expert gate
    float* out;                 // [T][H]
    int32_t n_wg;               // workgroups of the persistent expert GEMMs (one per CU)
    int32_t pass_m;             // pairs per pass: 16 or 32 (prefill_pass_size)
};

// Pass records a prefill of T tokens may need (passes of 16 pairs or more).
inline int64_t prefill_max_passes(int64_t T, int64_t K, int64_t E) { return (T * K + 15) / 16 + E + (T + 15) / 16 + 1; }

// Pairs per pass: 16 when the batch averages at most 10 pairs per routed
// expert, else 32.  A pass of 32 streams and decodes a busy expert's rows half
// as often and leaves its second row tile out where it is not needed, but its
// partial sums and staging take LDS from the ring (a slot, in some instances),
// and a small batch has fewer items to share out.  us per batch with skewed
// routing, passes of 16 / 32, at 4, 8, 12, 16, 20 pairs per expert:
//   Q8_0, 512 experts, H 4096, I 1024    1199/1209 1299/1271 1373/1399 1526/1418 1746/1485
//   Q8_0, 128 experts, H 2048, I 512      106/114   128/137   130/143   138/150   160/159
//   Q4_K, Q6_K, 512 experts, H 4096      1052/1096 1272/1280 1469/1371 1741/1579 2033/1765
//   Q2_K, Q3_K, 128 experts, H 4096       239/257   292/296   300/328   360/362   405/397
//   Q6_K, Q8_0, 256 experts, I 512        355/385   400/419   434/465   502/500   570/512
// and with rows of down above 2048 columns (prefill_wide: only gate/up takes
// passes of 32, the pairs are grouped twice), 64 experts, I 4096, at 3, 9, 12, 20, 40:
//   Q4_K, Q6_K, H 4096    513/518 586/600 643/618 885/844 1427/1283
//   Q8_0, H 2048          372/372 393/389 416/414 548/485  925/752
inline bool prefill_wide(int64_t I, int64_t Is) { return I > 2048 || Is > 2048; }
inline int prefill_pass_size(int64_t T, int64_t K, int64_t E) { return T * K <= 10 * E ? 16 : 32; }

// Weight formats the expert GEMMs read: gate and up (one format for both) and down.
inline bool prefill_type(int t) { return t == Q8_0 || t == Q2_K || t == Q3_K || t == Q4_K || t == Q5_K || t == Q6_K; }

// The phases of a prefill, stream-ordered (the caller checks types: gate and
// up of one format, formats the GEMMs read, H, I, Is powers of two from 256 to
// 4096, expert strides multiples of 16):
//   routing: router + top-K, or the caller's ids / weights; grouping; shared
//   gate; fp16 copy of x
//   gate/up + SwiGLU, down projection, combine.
int launch_prefill_route(const PrefillArgs& a, const int32_t* forced_ids, const float* forced_w, hipStream_t s);
int launch_prefill_gateup(const PrefillArgs& a, hipStream_t s);
int launch_prefill_down(const PrefillArgs& a, hipStream_t s);
int launch_prefill_combine(const PrefillArgs& a, hipStream_t s);

}  // namespace wm
