// wm_prefill.hip -- batched prefill of T tokens through the MoE block.
//
// The reference has no batched path: prompt tokens go one at a time through
// the decode loop (winmoe_inference.c:1079,2286-2288).  Here the T x K
// (token, slot) pairs are grouped by expert and every expert's matrices are
// streamed once for all of its tokens:
//
//   k_pf_router_m  reference-order fp32 logits of all tokens on fp32 MFMA
//   k_pf_router    the same for other widths and alignments (tiles of 16
//                  tokens x 16 experts, each lane one of the 16 FMA chains of
//                  4 x 4 (token, expert) pairs)
//   k_pf_tokens    per token: K-pass arg-max + softmax (or the caller's
//                  routing), x as fp16 times a power of two, the shared
//                  expert's gate
//   k_pf_group     counting sort of the pairs by expert; passes of <= 16
//                  or 32 pairs of one expert (prefill_pass_size)
//   k_pf_gemm      gate and up + SwiGLU on fp16 MFMA, persistent: one
//                  workgroup of 8 waves or two of 4 per CU work through
//                  (pass, 128-row block) items, every wave streaming its
//                  columns of the rows through an LDS-DMA ring of its own; the
//                  SwiGLU output is stored as fp16 hi + lo times a power of
//                  two per (pair, 128 rows); then the down projection of the
//                  same form (hi and lo: two MFMAs) (both in wm_pf_gemm.h, one
//                  instance per weight format)
//   k_pf_gemm2     routed K-quant passes and a few shared Q8_0 ones in one
//                  launch (shared experts of another format or width else
//                  take a launch of their own)
//   k_pf_combine   per token: sum_k w_k y_k in k order + gate * y_shared
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "../../include/winmoe_hip.h"
#include "wm_device.h"
#include "wm_format.h"
#include "wm_pf_gemm.h"
#include "wm_prefill.h"
#include "wm_wave.h"

namespace wm {

WM_DEV float bf16f(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

// ------------------------------------------------------------------ router

constexpr int PR_T = 16, PR_E = 16, PR_CH = 256, PR_LD = PR_CH + 4;

// Logits[t][e] in the reference order (transformer.h:172-191): for each
// (t, e), lane l keeps the fp32 FMA chain over columns l, l+16, ...; the 16
// lanes reduce with the xor tree 8, 4, 2, 1, then lane 0 adds the tail.
// Thread (chain l, sub-block sb) runs the chains of tokens 4*(sb/4)+i and
// experts 4*(sb%4)+j of the tile.
__global__ __launch_bounds__(256) void k_pf_router(const uint16_t* __restrict__ x, const float* __restrict__ W, int H,
                                                   int T, int E, float* __restrict__ logits) {
    __shared__ float xs[PR_T * PR_LD];
    __shared__ float wsh[PR_E * PR_LD];
    const int t0 = blockIdx.x * PR_T, e0 = blockIdx.y * PR_E;
    const int tid = threadIdx.x, l = tid & 15, sb = tid >> 4, tq = sb >> 2, eq = sb & 3;
    const int H16 = H - (H & 15);
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.0f;
    for (int c0 = 0; c0 < H16; c0 += PR_CH) {
        const int cn = min(PR_CH, H16 - c0);
        for (int i = tid; i < PR_T * PR_CH; i += 256) {
            const int r = i / PR_CH, c = i % PR_CH;
            xs[r * PR_LD + c] = (t0 + r < T && c < cn) ? bf16f(x[(int64_t)(t0 + r) * H + c0 + c]) : 0.0f;
        }
        for (int i = tid; i < PR_E * PR_CH; i += 256) {
            const int r = i / PR_CH, c = i % PR_CH;
            wsh[r * PR_LD + c] = (e0 + r < E && c < cn) ? W[(int64_t)(e0 + r) * H + c0 + c] : 0.0f;
        }
        __syncthreads();
        for (int s = 0; s < cn / 16; s++) {
            float xv[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                xv[i] = xs[(4 * tq + i) * PR_LD + l + 16 * s];
                wv[i] = wsh[(4 * eq + i) * PR_LD + l + 16 * s];
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(wv[j], xv[i], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // xor tree 8, 4, 2, 1 as row rotations (the partial sums repeat
            // with the period of the finished step)
            float v = acc[i][j];
            v += dpp_f32<DPP_ROR8>(v);
            v += dpp_f32<DPP_ROR4>(v);
            v += dpp_f32<DPP_ROR2>(v);
            v += dpp_f32<DPP_ROR1>(v);
            const int t = t0 + 4 * tq + i, e = e0 + 4 * eq + j;
            if (l == 0 && t < T && e < E) {
                for (int c = H16; c < H; c++) v = fmaf(W[(int64_t)e * H + c], bf16f(x[(int64_t)t * H + c]), v);
                logits[(int64_t)t * E + e] = v;
            }
        }
}

// The same logits on the matrix cores, for H a multiple of 128 and 16-byte
// aligned x rows and router rows.  v_mfma_f32_16x16x1_4b_f32 adds one product
// to each of 4 x 256 accumulators with a single rounding, the same bits as
// fmaf (compared over normal and subnormal operands), so its 4 blocks are 4
// of the 16 chains of a 16 x 16 (token, expert) tile: wave a runs the chains
// a, a + 4, a + 8, a + 12, block b the chain of column residue a + 4 b, and
// every chain adds its columns in the order above.  The xor tree's first two
// levels add the blocks of a wave, its last two the four waves.
//
// A workgroup takes MT x ET such tiles.  The columns come in chunks of 128,
// staged in LDS twice over with the loads of the next two chunks in flight.
// A staging thread loads 4 columns (one for each wave) of 4 consecutive steps
// of 16 columns and stores, per wave, the 4 steps as one 16-byte vector: the
// operands of 4 MFMAs are then one 16-byte read.  LDS rows are 132 floats, so
// the 16 rows of an operand read 16 different groups of 4 banks, and the
// staging puts rows 8 apart next to each other for the same reason.
//
// Tiles of 32 x 32 read each row half as often as those of 16 x 16, which
// spread a small batch over four times the workgroups: 32 x 32 from PQ_TILES
// of them on.  Routing phase less a caller-routed one, us, 16 x 16 / 32 x 32:
// 23 tokens, 512 experts, H 4096 (16 tiles of 32 x 32) 30.5 / 38.5; 100
// tokens (64) 33.3 / 38.7; 1500 tokens, 96 experts (141) 66.0 / 51.4; 2000
// tokens, 512 experts (1008) 255.6 / 149.1.  The kernel this replaced (16
// FMA chains per thread on the vector units) took 49, 72 and 270 us alone
// for 23, 512 and 2000 tokens, 512 experts.
constexpr int PQ_CH = 128, PQ_LD = PQ_CH + 4, PQ_TILES = 128;
typedef float f32x16 __attribute__((ext_vector_type(16)));
template <int MT, int ET>
__global__ __launch_bounds__(256) void k_pf_router_m(const uint16_t* __restrict__ x, const float* __restrict__ W, int H,
                                                     int T, int E, float* __restrict__ logits) {
    constexpr int XN = (16 * MT * 8 + 255) / 256, WN = (16 * ET * 8 + 255) / 256;      // staging units per thread
    __shared__ __attribute__((aligned(16))) float xs[2][16 * MT * PQ_LD];
    __shared__ __attribute__((aligned(16))) float wsh[2][16 * ET * PQ_LD];
    const int t0 = blockIdx.x * 16 * MT, e0 = blockIdx.y * 16 * ET;
    const int tid = threadIdx.x, lane = tid & 63, a = __builtin_amdgcn_readfirstlane(tid >> 6), b = lane >> 4, i = lane & 15;
    // staging unit u: steps 4 (u & 1) .. + 3 of the chunk, columns 4 bb .. + 3 of each step, of row `row`
    auto unit = [&](int u, int& row, int& col, int& dst) __attribute__((always_inline)) {
        const int kk = u & 1, bb = (u >> 1) & 3, r = u >> 3;
        row = (r & ~15) + 8 * (r & 1) + ((r >> 1) & 7);
        col = 64 * kk + 4 * bb;
        dst = row * PQ_LD + 8 * bb + 4 * kk;
    };
    const uint16_t* xsrc[XN];
    const float* wsrc[WN];
    int xdst[XN], wdst[WN];
#pragma unroll
    for (int q = 0; q < XN; q++) {
        int row, col;
        unit((tid + 256 * q) % (128 * MT), row, col, xdst[q]);
        xsrc[q] = x + (int64_t)min(t0 + row, T - 1) * H + col;         // rows past the last repeat it (not stored)
    }
#pragma unroll
    for (int q = 0; q < WN; q++) {
        int row, col;
        unit((tid + 256 * q) % (128 * ET), row, col, wdst[q]);
        wsrc[q] = W + (int64_t)min(e0 + row, E - 1) * H + col;
    }
    struct Chunk {
        uint2 x[XN][4];
        f32x4 w[WN][4];
    };
    Chunk ca, cb;
    auto gload = [&](Chunk& c, int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < WN; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) c.w[q][j] = *(const f32x4*)(wsrc[q] + c0 + 16 * j);
#pragma unroll
        for (int q = 0; q < XN; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) c.x[q][j] = *(const uint2*)(xsrc[q] + c0 + 16 * j);
    };
    auto lstore = [&](const Chunk& c, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < WN; q++)
            if (128 * ET >= 256 || tid < 128 * ET)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    *(f32x4*)&wsh[buf][wdst[q] + 32 * k] = (f32x4){c.w[q][0][k], c.w[q][1][k], c.w[q][2][k], c.w[q][3][k]};
#pragma unroll
        for (int q = 0; q < XN; q++)
            if (128 * MT >= 256 || tid < 128 * MT)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    f32x4 v;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t p = k < 2 ? c.x[q][j].x : c.x[q][j].y;
                        v[j] = __builtin_bit_cast(float, (k & 1) ? p & 0xFFFF0000u : p << 16);
                    }
                    *(f32x4*)&xs[buf][xdst[q] + 32 * k] = v;
                }
    };
    f32x16 acc[MT][ET];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < ET; e++) acc[m][e] = (f32x16)0.0f;
    auto sums = [&](int buf) __attribute__((always_inline)) {
        const float* xb = &xs[buf][i * PQ_LD + 32 * a + 8 * b];
        const float* wb = &wsh[buf][i * PQ_LD + 32 * a + 8 * b];
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            f32x4 xv[MT], wv[ET];
#pragma unroll
            for (int m = 0; m < MT; m++) xv[m] = *(const f32x4*)(xb + 16 * m * PQ_LD + 4 * kk);
#pragma unroll
            for (int e = 0; e < ET; e++) wv[e] = *(const f32x4*)(wb + 16 * e * PQ_LD + 4 * kk);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int e = 0; e < ET; e++)
                        acc[m][e] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[m][j], wv[e][j], acc[m][e], 0, 0, 0);
        }
    };
    const int nch = H / PQ_CH;
    gload(ca, 0);
    if (nch > 1) gload(cb, PQ_CH);
    lstore(ca, 0);
    __syncthreads();
    for (int c = 0; c < nch; c += 2) {
        // chunk c is in buffer 0, c + 1 in flight in cb; c + 2 goes out now
        // (a buffer was last read before the barrier ahead of its store)
        if (c + 2 < nch) gload(ca, (c + 2) * PQ_CH);
        sums(0);
        if (c + 1 == nch) break;
        lstore(cb, 1);
        __syncthreads();
        if (c + 3 < nch) gload(cb, (c + 3) * PQ_CH);
        sums(1);
        if (c + 2 < nch) lstore(ca, 0);
        __syncthreads();
    }
    // s[a] = (chain a + chain a + 8) + (chain a + 4 + chain a + 12); the logit is (s[0] + s[2]) + (s[1] + s[3])
    __syncthreads();
    float(*red)[MT * ET * 256] = (float(*)[MT * ET * 256])&xs[0][0];
    static_assert(4 * MT * ET * 256 <= 2 * 16 * MT * PQ_LD, "the partial sums take the x buffers' place");
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < ET; e++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                red[a][(m * ET + e) * 256 + 64 * r + lane] =
                    (acc[m][e][r] + acc[m][e][8 + r]) + (acc[m][e][4 + r] + acc[m][e][12 + r]);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int e = 0; e < ET; e++) {
            const int at = (m * ET + e) * 256 + tid;
            const float v = (red[0][at] + red[2][at]) + (red[1][at] + red[3][at]);
            const int t = t0 + 16 * m + 4 * b + (tid >> 6), ex = e0 + 16 * e + i;       // accumulator row 4 b + r, column i
            if (t < T && ex < E) logits[(int64_t)t * E + ex] = v;
        }
}

// ------------------------------------------------------------------ top-K, forced routing, grouping

// Exclusive prefix sums of (a, b) over the 1024 threads of a workgroup; the
// totals go to *tot.  wsum: 16 x 2 ints of LDS.
WM_DEV int2 block_excl_scan2(int2 v, int* wsum, int2* tot) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int2 inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int ux = __shfl_up(inc.x, d), uy = __shfl_up(inc.y, d);
        if (lane >= d) {
            inc.x += ux;
            inc.y += uy;
        }
    }
    if (lane == 63) {
        wsum[2 * wave] = inc.x;
        wsum[2 * wave + 1] = inc.y;
    }
    __syncthreads();
    int2 before = make_int2(0, 0), all = make_int2(0, 0);
    for (int w = 0; w < 16; w++) {
        const int2 ws = make_int2(wsum[2 * w], wsum[2 * w + 1]);
        if (w < wave) {
            before.x += ws.x;
            before.y += ws.y;
        }
        all.x += ws.x;
        all.y += ws.y;
    }
    __syncthreads();
    *tot = all;
    return make_int2(before.x + inc.x - v.x, before.y + inc.y - v.y);
}

// Sizes for which k_pf_group keeps its data on chip: the pairs' expert ids
// in registers (up to PG_REG per thread), the sorted pair list (16-bit
// entries) and the tokens' exponents (a byte each) in LDS, and the experts of
// the passes; larger batches read them from global memory, or search.
constexpr int PG_REG = 8, PG_SORT = 45056, PG_XEXP = 8192, PG_MAP = 4096;

// One workgroup: pairs grouped by expert (order inside an expert is free:
// every pair's output row is computed independently of the others), then
// cut into pass records of at most pm pairs (16 or 32): routed passes first,
// in expert order, then the shared expert's; pass_count = {routed passes,
// shared passes}.  A record also carries the x scale of each pair's token.
// The experts' hit counters are raised here (hits not NULL), one add per
// expert: with an atomic add per pair the top-K launch of 1001 tokens over 64
// experts took 17 us, the launch that holds its work now 7.
//
// Bound by latency: one workgroup, so the records are written by 8 threads
// each (16-byte pieces of a pass side by side), a pair's token is a multiply
// by kmul = ceil(2^32 / K) instead of a division, and ids are read PG_REG to
// a thread at a time: 512 tokens top-10 23 -> 11 us, 4096 tokens 114 -> 27.
__global__ __launch_bounds__(1024) void k_pf_group(const int32_t* __restrict__ ids, int T, int K, uint32_t kmul, int E,
                                                   int has_shared, int pm, int32_t* __restrict__ sorted,
                                                   int32_t* __restrict__ passes, int32_t* __restrict__ pass_count,
                                                   const int32_t* __restrict__ xexp, uint32_t* __restrict__ hits) {
    __shared__ int cnt[1025];
    __shared__ int off[1026];
    __shared__ int pbase[1026];
    __shared__ int wsum[32];
    __shared__ uint16_t srt[PG_SORT];
    __shared__ uint16_t pexp[PG_MAP];
    __shared__ uint8_t xe[PG_XEXP];
    const int tid = threadIdx.x, P = T * K, G = E + 1;      // group E: the shared expert (empty without one)
    const bool reg = P <= 1024 * PG_REG, lsort = P + (has_shared ? T : 0) <= PG_SORT, lxe = T <= PG_XEXP;
    // the ids and exponents are read once, together (more than PG_REG ids to a thread: again for the scatter)
    int ev[PG_REG];
    auto load_ids = [&](int base) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PG_REG; i++) {
            const int p = base + tid + 1024 * i;
            ev[i] = p < P ? ids[p] : -1;
            if (ev[i] >= E) ev[i] = -1;
        }
    };
    load_ids(0);
    if (lxe)
        for (int t = tid; t < T; t += 1024) xe[t] = (uint8_t)xexp[t];
    for (int e = tid; e < E; e += 1024) cnt[e] = 0;
    if (tid == 0) cnt[E] = has_shared ? T : 0;
    __syncthreads();
    for (int base = 0; base < P; base += 1024 * PG_REG) {
        if (base) load_ids(base);
#pragma unroll
        for (int i = 0; i < PG_REG; i++)
            if (ev[i] >= 0) atomicAdd(&cnt[ev[i]], 1);
    }
    __syncthreads();
    // pair offsets and pass bases of the groups, 1024 groups per round
    int2 carry = make_int2(0, 0);
    for (int base = 0; base < G; base += 1024) {
        const int e = base + tid;
        const int n = e < G ? cnt[e] : 0;
        if (e < E && n && hits) hits[e] += (uint32_t)n;
        int2 tot;
        const int2 ex = block_excl_scan2(make_int2(n, (n + pm - 1) / pm), wsum, &tot);
        if (e < G) {
            off[e] = carry.x + ex.x;
            pbase[e] = carry.y + ex.y;
            cnt[e] = carry.x + ex.x;          // scatter cursor
        }
        carry.x += tot.x;
        carry.y += tot.y;
    }
    if (tid == 0) {
        off[G] = carry.x;
        pbase[G] = carry.y;
    }
    __syncthreads();
    if (tid == 0) {
        pass_count[0] = pbase[E];
        pass_count[1] = pbase[G] - pbase[E];
    }
    const int npass = pbase[G], nrouted = pbase[E];
    const bool map = nrouted <= PG_MAP;
    if (map)
        for (int e = tid; e < E; e += 1024)
            for (int q = pbase[e]; q < pbase[e + 1]; q++) pexp[q] = (uint16_t)e;
    // the sorted list: in LDS when it fits, else in global memory
    auto put = [&](int pos, int p) __attribute__((always_inline)) {
        if (lsort) srt[pos] = (uint16_t)p;
        else sorted[pos] = p;
    };
    for (int base = 0; base < P; base += 1024 * PG_REG) {
        if (!reg) load_ids(base);
#pragma unroll
        for (int i = 0; i < PG_REG; i++)
            if (ev[i] >= 0) put(atomicAdd(&cnt[ev[i]], 1), base + tid + 1024 * i);
    }
    if (has_shared)
        for (int t = tid; t < T; t += 1024) put(off[E] + t, P + t);
    __syncthreads();
    // thread: 4 pairs of a pass
    for (int it = tid; it < 8 * npass; it += 1024) {
        const int q = it >> 3, m4 = it & 7;
        int e = E;
        if (q < nrouted) {
            if (map) e = pexp[q];
            else {
                int lo = 0, hi = E - 1;          // largest e with pbase[e] <= q
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (pbase[mid] <= q) lo = mid;
                    else hi = mid - 1;
                }
                e = lo;
            }
        }
        const int first = off[e] + (q - pbase[e]) * pm;
        const int mn = min(pm, off[e + 1] - first);
        int32_t* rec = passes + (int64_t)q * GM_REC;
        int prs[4];
        uint32_t ex = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int at = first + min(4 * m4 + j, mn - 1);
            prs[j] = lsort ? (int)srt[at] : sorted[at];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int pr = prs[j];
            const int tok = pr >= P ? pr - P : K == 1 ? pr : (int)__umulhi((uint32_t)pr, kmul);
            ex |= (uint32_t)((lxe ? (int)xe[tok] : xexp[tok]) & 0xFF) << (8 * j);
        }
        if (m4 == 0) *(int4*)rec = make_int4(e, mn, 0, 0);
        *(int4*)(rec + 4 + 4 * m4) = make_int4(prs[0], prs[1], prs[2], prs[3]);
        rec[4 + GM_M + m4] = (int32_t)ex;
    }
}

// What a batch needs of each token ahead of the expert GEMMs, one workgroup
// per token, one launch (each was a launch of its own, 5 us apiece):
//   * its experts and weights: arg-max and softmax of its logits (wave 0), or
//     the caller's (logits NULL);
//   * x bf16 [H] -> x16 = fp16(x * 2^-e) with e per token (pf_exp of the
//     token's largest |x|), xexp[t] = e.  bf16 values are exact in fp16 at
//     that scale (8 significant bits, normal range down to 2^-29 of the
//     maximum);
//   * the shared expert's gate (g not NULL): sigmoid_stable((float) sum_h
//     g[h] x[h]) with the dot in fp64 (winmoe_inference.c:2005-2009),
//     fixed-order tree.
__global__ __launch_bounds__(256) void k_pf_tokens(const uint16_t* __restrict__ x, int H, uint16_t* __restrict__ x16,
                                                   int32_t* __restrict__ xexp, const float* __restrict__ g,
                                                   float* __restrict__ sg, const float* __restrict__ logits,
                                                   const int32_t* __restrict__ fids, const float* __restrict__ fw, int E,
                                                   int K, int32_t* __restrict__ ids, float* __restrict__ w,
                                                   int32_t* __restrict__ status) {
    __shared__ float wmax[WAVES];
    __shared__ double part[256];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint16_t* xr = x + (int64_t)t * H;
    if (logits) {
        if (wave == 0)
            wave_topk<false>(logits + (int64_t)t * E, E, K, ids + (int64_t)t * K, w + (int64_t)t * K, nullptr, status, lane);
    } else if ((int)threadIdx.x < K) {
        const int64_t p = (int64_t)t * K + threadIdx.x;
        const int e = fids[p];
        ids[p] = e;
        w[p] = fw[p];
        if (e < 0 || e >= E) atomicOr(status, WM_STATUS_BAD_EXPERT_ID);
    }
    float m = 0.0f;
    for (int c0 = threadIdx.x * 8; c0 < H; c0 += 256 * 8) {
        const u32x4 v = *(const u32x4*)(xr + c0);
#pragma unroll
        for (int i = 0; i < 4; i++)
            m = fmaxf(m, fmaxf(fabsf(__builtin_bit_cast(float, v[i] << 16)),
                               fabsf(__builtin_bit_cast(float, v[i] & 0xFFFF0000u))));
    }
    m = fmaxf(m, dpp_f32<DPP_XOR1>(m));
    m = fmaxf(m, dpp_f32<DPP_XOR2>(m));
    m = fmaxf(m, dpp_f32<DPP_HALF_MIRROR>(m));
    m = fmaxf(m, dpp_f32<DPP_MIRROR>(m));       // max of the 16 lanes of each row
    float r = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 0));
    r = fmaxf(r, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 16)));
    r = fmaxf(r, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 32)));
    r = fmaxf(r, __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 48)));
    if (lane == 0) wmax[wave] = r;
    if (g) {
        double acc = 0.0;
        for (int base = 0; base < H; base += 256 * 16) {
            float gv[16], xv[16];
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int h = min(base + (int)threadIdx.x + 256 * i, H - 1);
                gv[i] = g[h];
                xv[i] = bf16f(xr[h]);
            }
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (base + (int)threadIdx.x + 256 * i < H) acc += (double)gv[i] * (double)xv[i];
        }
        part[threadIdx.x] = acc;
    }
    __syncthreads();
    const float M = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int e = pf_exp(M);
    const float inv = ldexpf(1.0f, -e);
    for (int c0 = threadIdx.x * 8; c0 < H; c0 += 256 * 8) {
        const u32x4 v = *(const u32x4*)(xr + c0);
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = __builtin_bit_cast(uint16_t, (_Float16)(__builtin_bit_cast(float, v[i] << 16) * inv));
            const uint32_t hi =
                __builtin_bit_cast(uint16_t, (_Float16)(__builtin_bit_cast(float, v[i] & 0xFFFF0000u) * inv));
            o[i] = lo | (hi << 16);
        }
        *(u32x4*)(x16 + (int64_t)t * H + c0) = o;
    }
    if (threadIdx.x == 0) xexp[t] = e;
    if (!g) return;
    for (int d = 128; d >= 64; d >>= 1) {
        if ((int)threadIdx.x < d) part[threadIdx.x] += part[threadIdx.x + d];
        __syncthreads();
    }
    if (wave == 0) {
        double v = part[lane];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_down(v, d);
        if (lane == 0) sg[t] = sigmoid_stable((float)v);
    }
}

// out[t][h] = sum_k w[t][k] y[t*K + k][h] (k order, invalid ids skipped) + gate(t) * y_shared[t][h];
// 4 consecutive h per thread.
__global__ __launch_bounds__(256) void k_pf_combine(PrefillArgs a) {
    const int t = blockIdx.y, h4 = blockIdx.x * 256 + threadIdx.x;
    if (4 * h4 >= a.H) return;
    const int H4 = a.H / 4;
    const f32x4* y4 = (const f32x4*)a.y;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k = 0; k < a.K; k++) {
        const int e = a.ids[(int64_t)t * a.K + k];
        if (e < 0 || e >= a.E) continue;
        const float wk = a.w[(int64_t)t * a.K + k];
        const f32x4 v = y4[((int64_t)t * a.K + k) * H4 + h4];
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = fmaf(wk, v[i], acc[i]);
    }
    if (a.has_shared) {
        f32x4 ys = y4[((int64_t)a.T * a.K + t) * H4 + h4];
        if (a.sh_gate_inp) {
            const float gt = a.sg[t];
#pragma unroll
            for (int i = 0; i < 4; i++) ys[i] *= gt;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = acc[i] + ys[i];
    }
    ((f32x4*)a.out)[(int64_t)t * H4 + h4] = acc;
}

// ------------------------------------------------------------------ launcher

static void launch_group(const PrefillArgs& a, uint32_t* hits, hipStream_t s) {
    const uint32_t kmul = (uint32_t)(((1ull << 32) + a.K - 1) / a.K);       // (0 for K = 1)
    hipLaunchKernelGGL(k_pf_group, dim3(1), dim3(1024), 0, s, a.ids, a.T, a.K, kmul, a.E, a.has_shared, a.pass_m, a.sorted,
                       a.passes, a.pass_count, a.xexp, hits);
}

int launch_prefill_route(const PrefillArgs& a, const int32_t* forced_ids, const float* forced_w, hipStream_t s) {
    if (!forced_ids) {
        if (a.H % PQ_CH == 0 && ((uintptr_t)a.x & 15) == 0 && ((uintptr_t)a.router & 15) == 0) {
            const int64_t tiles = (int64_t)((a.T + 31) / 32) * ((a.E + 31) / 32);
            if (tiles >= PQ_TILES)
                hipLaunchKernelGGL((k_pf_router_m<2, 2>), dim3((a.T + 31) / 32, (a.E + 31) / 32), dim3(256), 0, s, a.x,
                                   a.router, a.H, a.T, a.E, a.logits);
            else
                hipLaunchKernelGGL((k_pf_router_m<1, 1>), dim3((a.T + 15) / 16, (a.E + 15) / 16), dim3(256), 0, s, a.x,
                                   a.router, a.H, a.T, a.E, a.logits);
        } else
            hipLaunchKernelGGL(k_pf_router, dim3((a.T + PR_T - 1) / PR_T, (a.E + PR_E - 1) / PR_E), dim3(256), 0, s, a.x,
                               a.router, a.H, a.T, a.E, a.logits);
    }
    hipLaunchKernelGGL(k_pf_tokens, dim3(a.T), dim3(256), 0, s, a.x, a.H, a.x16, a.xexp,
                       a.has_shared ? a.sh_gate_inp : nullptr, a.sg, forced_ids ? nullptr : a.logits, forced_ids, forced_w,
                       a.E, a.K, a.ids, a.w, a.status);
    launch_group(a, a.hits, s);
    return (int)hipGetLastError();
}

// One gate/up or down GEMM launch of format wt over the passes sel selects,
// for passes of m pairs.
template <int M> static int launch_q8(bool gateup, const PfGemm& g, int n_wg, hipStream_t s) {
    return gateup ? launch_pf_gemm<1, Q8_0, M>(g, n_wg, s) : launch_pf_gemm<2, Q8_0, M>(g, n_wg, s);
}
static int launch_fmt(int m, bool gateup, int wt, const PfGemm& g, int n_wg, hipStream_t s) {
    if (wt != Q8_0) return launch_pf_gemm_kq(m, gateup, wt, g, n_wg, s);
    return m == 16 ? launch_q8<16>(gateup, g, n_wg, s) : launch_q8<32>(gateup, g, n_wg, s);
}

// Routed and shared passes in one launch when their formats and row lengths
// agree, or when the routed ones are K-quants and the shared ones few and
// Q8_0; else in two.
struct PfShape {
    int wt, ncol;
};
static int launch_split(int m, bool gateup, PfShape r, PfShape sh, bool has_shared, PfGemm& g, int n_wg, hipStream_t s) {
    const bool one = !has_shared || (r.wt == sh.wt && r.ncol == sh.ncol);
    g.sel = one ? 0 : 1;
    g.ncol = r.ncol;
    g.rb = (int32_t)matrix_bytes(r.wt, 1, r.ncol);
    if (one) return launch_fmt(m, gateup, r.wt, g, n_wg, s);
    PfGemm h = g;
    h.sel = 2;
    h.ncol = sh.ncol;
    h.rb = (int32_t)matrix_bytes(sh.wt, 1, sh.ncol);
    // One launch when the shared items are less than half a round of the
    // workgroups; from there a launch of their own fills the chip, and the two
    // kernels keep their registers (two launches / one, us per batch: 23 tokens
    // 231 / 208, 512 tokens 952 / 965, 2000 tokens level).
    const int grid = n_wg * (8 / gm_waves(gateup, r.ncol)), items = (g.T + m - 1) / m * g.nrb_s;
    if (r.wt != Q8_0 && sh.wt == Q8_0 && (gateup || m == 16) && 2 * items < grid)
        return launch_pf_gemm_kq_q8(m, gateup, r.wt, g, h, n_wg, s);
    if (int rc = launch_fmt(m, gateup, r.wt, g, n_wg, s)) return rc;
    return launch_fmt(m, gateup, sh.wt, h, n_wg, s);
}

int launch_prefill_gateup(const PrefillArgs& a, hipStream_t s) {
    PfGemm g = {};
    g.w0 = a.gate; g.w1 = a.up; g.st0 = a.gstride; g.st1 = a.ustride;
    g.s0 = a.sh_gate; g.s1 = a.sh_up;
    g.mb_r = (int32_t)matrix_bytes(a.gt, a.I, a.H);
    g.mb_s = a.has_shared ? (int32_t)matrix_bytes(a.sgt, a.Is, a.H) : g.mb_r;
    g.a_hi = a.x16; g.a_lo = a.x16; g.a_ld = a.H; g.a_sc = nullptr; g.sc_ld = 0;
    g.T = a.T; g.K = a.K;
    g.rows_item = GM_ROWS;
    g.nrb_r = a.I / GM_ROWS; g.nrb_s = a.has_shared ? a.Is / GM_ROWS : 1;
    g.recs = a.passes; g.npass = a.pass_count;
    g.o_hi = a.act_hi; g.o_lo = a.act_lo; g.o_sc = a.act_sc; g.o_ld = a.act_stride; g.osc_ld = a.act_stride / 128;
    return launch_split(a.pass_m, true, {a.gt, a.H}, {a.sgt, a.H}, a.has_shared, g, a.n_wg, s);
}

// Rows of a down item: 512 read a pass's activations least often; a batch
// whose items are then fewer than two rounds of the workgroups (two per CU)
// takes 256, and 128 below half a round, so that the rounds come out even.
// us per batch, 512 / 256 / 128 rows: 8 tokens, 64 experts, H 2048 (0.3
// rounds) 77 / 70 / 69; 1001 tokens, 64 experts, H 2048 (1.5) 179 / 174 /
// 190; 300 tokens, 128 experts, H 2048 (1.6) 159 / 153 / 153; 512 tokens Q4_K,
// Q6_K, 512 experts, H 4096 (10) 956 / 966 / 983; 4096 tokens Q8_0 3627 / 3781
// / 4112.
static int down_rows(const PrefillArgs& a) {
    const int64_t pairs = (int64_t)a.T * a.K, m = a.pass_m;
    const int64_t passes = std::min<int64_t>(pairs, a.E) + pairs / m + (a.has_shared ? a.T / m : 0);
    const int64_t items = passes * a.H / 512, grid = 2 * (int64_t)a.n_wg;
    return a.H % 512 || items < 2 * grid ? (2 * items < grid ? 128 : 256) : 512;
}

// Down of rows longer than 2048 columns (slices of 512, hi and lo) has
// registers for 16 pairs only: after gate/up in passes of 32 the pairs are
// grouped again.  That launch is 10 us; gate/up in passes of 16 as well cost a
// busy expert more: 1500 tokens top-2 of 8 experts, H and I 4096, Q8_0, gate/up
// 925 us in passes of 16, 721 in passes of 32.
int launch_prefill_down(const PrefillArgs& args, hipStream_t s) {
    PrefillArgs a = args;
    if (a.pass_m > 16 && prefill_wide(a.I, a.Is)) {
        a.pass_m = 16;
        launch_group(a, nullptr, s);
    }
    PfGemm g = {};
    g.w0 = a.down; g.w1 = a.down; g.st0 = g.st1 = a.dstride;
    g.s0 = g.s1 = a.sh_down;
    g.mb_r = (int32_t)matrix_bytes(a.dt, a.H, a.I);
    g.mb_s = a.has_shared ? (int32_t)matrix_bytes(a.sdt, a.H, a.Is) : g.mb_r;
    g.a_hi = a.act_hi; g.a_lo = a.act_lo; g.a_ld = a.act_stride; g.a_sc = a.act_sc; g.sc_ld = a.act_stride / 128;
    g.T = a.T; g.K = a.K;
    g.rows_item = down_rows(a);
    g.nrb_r = g.nrb_s = a.H / g.rows_item;
    g.recs = a.passes; g.npass = a.pass_count;
    g.y = a.y; g.y_ld = a.H;
    return launch_split(a.pass_m, false, {a.dt, a.I}, {a.sdt, a.Is}, a.has_shared, g, a.n_wg, s);
}

int launch_prefill_combine(const PrefillArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_combine, dim3((a.H / 4 + 255) / 256, a.T), dim3(256), 0, s, a);
    return (int)hipGetLastError();
}

}  // namespace wm
