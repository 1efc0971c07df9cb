// wm_pf_gemm.h -- the grouped expert GEMMs of the batched prefill (fp16 MFMA),
// for every supported weight format.  Included by wm_prefill.hip (Q8_0
// instances, the prefill launcher) and wm_prefill_kq.hip (K-quant instances).
// Internal; not part of the public ABI.
//
// One workgroup of 8 waves per CU, or two of 4 (gm_waves), work through a
// static list of items: item j of a launch is (pass, block of matrix rows),
// and workgroup b takes one of every round of `grid` items: pf_item_slot (the
// row blocks of a pass on workgroups of one XCD), pf_item_slot_full.
//
// The matrix columns are cut into slices, one per wave (groups of waves when
// there are fewer slices than waves: each group then takes its own 16-row tiles).
// A wave keeps the activations of its slice, for all pairs of the pass, in
// registers as MFMA operands for the whole item, and streams its slice of
// every row tile: 16 rows x KC columns of raw blocks per ring slot, filled by
// LDS-DMA of its own, read into registers and refilled at once, so a wave
// waits for its own loads only and nearly the whole ring is always in flight.
// The waves together read 16 whole rows, a contiguous piece of memory.  The
// waves' partial sums of a tile meet in LDS (one barrier per tile), are added
// in slice order and leave as the item's outputs.
//
// A ring slot holds, for each of its 16 rows, GR granules of 16 B from the
// 16-byte boundary at or before the row start plus the one at or before the
// chunk's offset in the row (Q8_0 272 B, Q4_K 144 B and Q5_K 176 B start
// aligned; Q2_K 84 B, Q3_K 110 B and Q6_K 210 B start up to 24 or 28 bytes
// in; an odd count: gm_granules).
//
// Weights become fp16 exactly (small integers under the exponent byte 0x64
// are 1024 + q), so v_mfma_f32_16x16x32_f16 gives the dot product of 32
// weights with the scaled fp16 activations.  Which 32 columns an MFMA sums
// is free as long as both operands agree: KqRow::col names the 8 columns of
// lane group g, chosen so that a lane reads long runs of bytes and needs few
// sub-block scales.  Two 4-bit (or 2-, 6-bit) values at bits 0 and 16 of a
// dword become two halves with one v_and_or, so the 8 columns of a K-quant
// operand go in the order 0 2 1 3 4 6 5 7 (the activations are permuted to
// match when an item starts):
//   * Q8_0 (q8_dequant.h:15-18): one MFMA per 32-weight block (byte ^ 0x80
//     is q + 128), times the block's fp16 scale d;
//   * Q4_K / Q5_K / Q3_K / Q2_K (q4k_dequant.h:112-168, q5k_dequant.h:98-131
//     and the public ggml layouts): q times its sub-block scale is an integer
//     fp16 holds exactly, so the products add up in the MFMA accumulator and
//     the super-block's d multiplies the sum; the mins of Q4_K, Q5_K and Q2_K
//     are a second MFMA of the activations with the replicated min, times
//     dmin;
//   * Q6_K (q6k_dequant.h:112-141): q times its int8 scale needs 13 bits, so
//     the scale is split into 16 s1 + s0, s1 the nearest (a scale of -7 .. 7
//     is s0 alone), and each part multiplies q exactly.
// Down activations carry a power-of-two scale per (pair, 128 columns), which
// multiplies the sum of those columns.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "wm_device.h"
#include "wm_format.h"
#include "wm_wave.h"

namespace wm {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

WM_DEV int pair_token(int p, int T, int K) { return p < T * K ? p / K : p - T * K; }

// Exponent e with m * 2^-e in [2^14, 2^15) for a finite m > 0 (clamped to
// e >= -126 so that 2^e and 2^-e are normal floats); 0 otherwise.  Values of
// a group scaled by 2^-e fit fp16 with its full 11-bit precision down to
// 2^-29 of the group maximum.
WM_DEV int pf_exp(float m) {
    if (!(m > 0.0f) || !(m <= 3.402823466e38f)) return 0;
    int E;
    frexpf(m, &E);                 // m in [2^(E-1), 2^E)
    return max(E - 15, -126);
}

// Expert passes: a pass is up to M pairs of one expert (M = 16 or 32, one
// value per launch), described by a record of GM_REC ints: expert (E =
// shared), pair count, 0, 0, GM_M pair ids (positions past the count repeat
// the last id), then the x scale exponents of the pairs' tokens, 4 signed
// bytes per int, for GM_M pairs.  The record layout is the same for both pass
// sizes.
constexpr int GM_M = 32;
constexpr int GM_REC = 64;

constexpr int GM_ROWS = 128;          // matrix rows per gate/up item; columns per activation scale of down
constexpr int GM_KC = 256;            // columns per super-block (Q8_0: 8 blocks)
constexpr int GM_SLD = GM_ROWS + 16;  // floats per pair in the SwiGLU staging (rows 16 banks apart)

// Granules of 16 B loaded per row and ring slot for format WT (nsb
// super-blocks; Q8_0: nsb x 8 blocks): enough to hold the chunk wherever it
// starts (the chunk plus the row start's and the chunk offset's distances
// past a 16-byte boundary: none for Q8_0, Q4_K and Q5_K, whose rows and
// chunks start aligned; up to 12 bytes each for Q2_K, 14 for Q3_K and Q6_K),
// rounded up to an odd count: a row's LDS slot is then an odd multiple of 4
// dwords long, so the slots of 16 consecutive rows start on 16 different
// groups of 4 banks (of 64).
constexpr int gm_granules(int wt, int nsb) {
    const int bytes = wt == Q8_0 ? nsb * 272 : nsb * block_bytes(wt);
    const int mis = wt == Q2_K ? 12 : (wt == Q3_K || wt == Q6_K) ? 14 : 0;
    return ((bytes + 2 * mis + 15) / 16) | 1;
}

// LDS bytes of a workgroup of cw waves with s ring slots each, passes of m
// pairs, slots of nsb x 256 columns; a CU holds 8 / cw workgroups.
constexpr int gm_lds(int cw, int ahl, int wt, int m, int nsb, int s) {
    return cw * s * 256 * gm_granules(wt, nsb) + 2 * cw * (m / 16) * 1024 + (ahl == 1 ? m * GM_SLD * 4 : 0);
}
// Ring slots per wave: as many as the LDS holds, up to 4.
constexpr int gm_slots(int cw, int ahl, int wt, int m, int nsb) {
    int s = 2;
    while (s < 4 && gm_lds(cw, ahl, wt, m, nsb, s + 1) <= 163840 / (8 / cw)) s++;
    return s;
}

// Columns of a wave's slice: gate/up 512 (or the whole row of 256); down 256,
// or 512 for the longest rows (the activations of a slice, hi and lo, stay in
// registers).  One rule for both pass sizes: the sums are then the same.
WM_HD constexpr int gm_slice(bool gateup, int ncol) { return gateup ? (ncol < 512 ? ncol : 512) : (ncol > 2048 ? 512 : 256); }

template <int AHL, int WT, int M, int NSB, int CW> struct GmGeo {
    static_assert(M == 16 || M == 32, "pass size");
    static_assert(NSB == 1 || NSB == 2, "super-blocks per ring slot");
    static_assert(CW == 4 || CW == 8, "waves");
    static constexpr bool KQ = WT != Q8_0;
    static constexpr bool GU = AHL == 1;                                // gate/up (else down)
    static constexpr int NSUB = GU ? 2 : 1;                             // gate and up tiles in turn; down tiles
    static constexpr int THREADS = 64 * CW;
    static constexpr int MT = M / 16;                                   // row tiles of 16 pairs
    static constexpr int KC = GM_KC * NSB;                              // columns per ring slot
    static constexpr int CHUNK = KQ ? NSB * block_bytes(WT) : KC / 32 * 34;   // bytes of a row's slot chunk
    static constexpr int MSL = NSB == 2 || (!GU && M == 32) ? 1 : 2;    // ring slots per slice, at most
    static constexpr int GR = gm_granules(WT, NSB);
    static constexpr int RSLOT = 16 * GR;                               // LDS bytes of a row's chunk
    static constexpr int SLOT = 16 * RSLOT;
    static constexpr int NI = (16 * GR + 63) / 64;                      // DMA instructions per slot
    static constexpr int S = gm_slots(CW, AHL, WT, M, NSB);
    static constexpr int PART = CW * MT * 1024;                         // partial sums of one tile per wave
    static constexpr int PBASE = CW * S * SLOT;
    static constexpr int STG = PBASE + 2 * PART;                        // gate/up: M pairs x 128 rows fp32
    static constexpr int LDS = STG + (GU ? M * GM_SLD * 4 : 0);
    static_assert(KQ || GR * 16 == CHUNK, "Q8_0 chunks are whole granules");
    static_assert(LDS <= 163840 / (8 / CW) && LDS == gm_lds(CW, AHL, WT, M, NSB, S), "LDS");
    static_assert((S - 1) * NI < 64, "vmcnt");
};

static_assert(4 + GM_M + GM_M / 4 <= GM_REC, "pass record");

struct PfGemm {
    const uint8_t* w0;                 // routed matrices (gate, up) or (down, -): expert e at + e * st
    const uint8_t* w1;
    int64_t st0, st1;
    const uint8_t* s0;                 // shared-expert matrices
    const uint8_t* s1;
    int32_t mb_r, mb_s;                // bytes per matrix: routed, shared
    const uint16_t* a_hi;              // activations, fp16 bits [rows][a_ld]
    const uint16_t* a_lo;
    int64_t a_ld;
    const float* a_sc;                 // activation scales [rows][sc_ld], one per 128 columns
    int64_t sc_ld;
    int32_t T, K;
    int32_t nrb_r, nrb_s;              // row blocks per pass: routed, shared
    int32_t rows_item;                 // matrix rows per item
    int32_t ncol;                      // matrix columns
    int32_t rb;                        // bytes per matrix row
    int32_t ns, lsl;                   // ring slots per slice, log2 of the slices (launch_pf_gemm)
    int32_t sel;                       // passes of this launch: 0 all, 1 routed only, 2 shared only
    const int32_t* recs;
    const int32_t* npass;              // {routed passes, shared passes}
    uint16_t* o_hi;                    // gate/up: SwiGLU output hi / lo [pair][o_ld], scales [pair][osc_ld]
    uint16_t* o_lo;
    float* o_sc;
    int64_t o_ld, osc_ld;
    float* y;                          // down: [pair][y_ld]
    int64_t y_ld;
};

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(4))) int32_t cint_t;       // scalar loads

// Workgroups are dispatched to the 8 XCDs in turn (workgroup b on XCD b % 8)
// and each XCD has its own L2.  Item j of round i goes to workgroup b with
// j - i * grid = slot(b): the R consecutive items of one pass (its row groups,
// which read the same activations) land on workgroups of one XCD, so the
// activations come from HBM once per pass rather than once per XCD.  A
// bijection of [0, grid) when grid is a multiple of 8 R; the identity
// otherwise.
constexpr int PF_XCDS = 8;
WM_HD int pf_item_slot(int b, int grid, int R) {
    if (R <= 0 || grid % (PF_XCDS * R)) return b;
    const int x = b % PF_XCDS, q = b / PF_XCDS;
    return ((q / R) * PF_XCDS + x) * R + q % R;
}

// With passes of 32 pairs (busy experts of several passes), in a round that
// every workgroup has an item of, an XCD takes a contiguous run of them: some
// of the passes of an expert then find its rows in that XCD's L2.  4096 tokens
// top-10, Q8_0 (about 3 passes per expert): L2 misses of gate/up 2.53 times the
// matrices, 3.09 without the runs, of down 2.23 and 3.03; 3631 -> 3541 us per
// batch.  1001 tokens, 64 experts: 1.50 and 2.54 times, 182.5 -> 179.1 us.
// Passes of 16 keep the spread order (512 tokens Q8_0 1374, in runs 1377; Q4_K
// 940, 936), as does the last, partial round (1001 tokens in runs there too:
// 205).
WM_HD int pf_item_slot_full(int b, int grid) {
    return grid % PF_XCDS ? b : (b % PF_XCDS) * (grid / PF_XCDS) + b / PF_XCDS;
}

// Raw buffer resource over [p, p + bytes) (gfx9 word 3: 32-bit data format).
WM_DEV __amdgpu_buffer_rsrc_t gm_rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}

// This wave's LDS accesses are complete.
WM_DEV void gm_wait_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0)
    asm volatile("" ::: "memory");
}

// All waves of the workgroup meet; this wave's LDS accesses are complete.
// (No fence: a fence would also wait for the ring's loads in flight.)
WM_DEV void gm_bar() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// ------------------------------------------------------------------ row chunks in LDS

// N dwords at byte offset o of an LDS row slot whose address is 16-byte
// aligned; AL: the alignment o is known to have (16, 4 or 2).
template <int AL, int N> WM_DEV void ld_dw(const uint8_t* slot, int o, uint32_t* w) {
    if constexpr (AL >= 16) {
        static_assert(N == 4, "one 16-byte read");
        const u32x4 v = *(const u32x4*)(slot + o);
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = v[i];
    } else if constexpr (AL == 4) {
        const uint32_t* p = (const uint32_t*)(slot + o);
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = p[i];
    } else {
        const uint32_t* p = (const uint32_t*)(slot + (o & ~3));
        const uint32_t s = (uint32_t)o & 3u;
        uint32_t r[N + 1];
#pragma unroll
        for (int i = 0; i <= N; i++) r[i] = p[i];
#pragma unroll
        for (int i = 0; i < N; i++) w[i] = alignbyte(r[i + 1], r[i], s);
    }
}

WM_DEV f16x2 h2(float v) { return (f16x2){(_Float16)v, (_Float16)v}; }
WM_DEV f16x2 as_h2(uint32_t u) { return __builtin_bit_cast(f16x2, u); }
WM_DEV f16x2 fma2(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }

// 1024 + byte K of w (lane-varying selector: byte_sel), twice, as fp16.
WM_HD constexpr uint32_t byte_sel(uint32_t p) { return p | (p << 16) | 0x04000400u; }
WM_DEV f16x2 byte_h1024(uint32_t w, uint32_t sel) { return as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)); }

// The bits of mask in both halves of w under the exponent of 1024.  e1024 is
// 0x64006400 in a register the compiler does not know the value of: one
// v_and_or (a VOP3 instruction takes no literals here) instead of two
// instructions with one literal each.
WM_DEV uint32_t opaque_e1024() {
    uint32_t v;
    asm("v_mov_b32 %0, 0x64006400" : "=v"(v));
    return v;
}
WM_DEV uint32_t field(uint32_t w, uint32_t mask, uint32_t e1024) { return (w & mask) | e1024; }

WM_DEV f16x8 cat4(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
    return (f16x8){a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
WM_DEV f16x8 rep4(f16x2 a) { return cat4(a, a, a, a); }

// A super-block of one weight row: load() reads this lane's part (row slot,
// first byte o, lane group g) into registers; the 256 columns are summed in
// 8 MFMAs, unit (h, u) = MFMA u of the 128-column half h, of which this lane
// holds the 8 columns col(h, u, g) .. + 7 (in the order 0 2 1 3 4 6 5 7).
// FOLD formats: after half(h), unit(h, u) is q * sc (an integer that fp16
// holds exactly) and mins(u) the sub-block min; the weight is
// d * unit - dmin * mins.  Values are decoded as (1024 + 2^k q) * (sc / 2^k)
// - 1024 * sc / 2^k, one rounding of an exact result.
// pin(): the loaded registers become unknown to the compiler, so that it does
// not decode ahead of a branch what both sides need (the decoded values of all
// units at once: up to 240 registers in scratch).
template <int WT> struct KqRow;

template <int N> WM_DEV void pin_dw(uint32_t (&w)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("" : "+v"(w[i]));
}

// Q4_K and Q5_K: half h is qs bytes 64 h .. + 63, low nibbles columns 32 i +
// l of byte 32 i + l, high nibbles 32 columns on.  This lane: bytes 16 g ..
// + 15 of the half: low nibbles in sub-block 4 h + 2 (g / 2), high nibbles in
// the next.
template <int BITS> struct Kq45 {
    static constexpr int AL = 16;
    static constexpr bool FOLD = true, MINS = true;
    u32x4 hd;
    uint32_t q[2][4], qh[4];
    float d, dmin;
    uint32_t sc[2], mn[2];                       // 6-bit scales and mins of sub-blocks 0-3, 4-7 (a byte each)
    f16x2 s2[2], c2[2], m2[2];
    uint32_t sel, gg;
    WM_DEV static int col(int h, int u, int g) { return 128 * h + 64 * (g >> 1) + 16 * (g & 1) + 32 * (u >> 1) + 8 * (u & 1); }
    WM_DEV void load(const uint8_t* slot, int o, int g) {
        hd = *(const u32x4*)(slot + o);
        if constexpr (BITS == 5) ld_dw<16, 4>(slot, o + 16 + 16 * (g & 1), qh);
        ld_dw<16, 4>(slot, o + (BITS == 5 ? 48 : 16) + 16 * g, q[0]);
        ld_dw<16, 4>(slot, o + (BITS == 5 ? 48 : 16) + 64 + 16 * g, q[1]);
    }
    WM_DEV void pin() {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t v = hd[i];
            asm volatile("" : "+v"(v));
            hd[i] = v;
        }
        if constexpr (BITS == 5) pin_dw(qh);
        pin_dw(q[0]);
        pin_dw(q[1]);
    }
    WM_DEV void head(int g) {
        d = h2f(hd[0]);
        dmin = h2f(hd[0] >> 16);
        sc[0] = hd[1] & 0x3F3F3F3Fu;
        mn[0] = hd[2] & 0x3F3F3F3Fu;
        sc[1] = (hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u);
        mn[1] = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
        gg = (uint32_t)(g >> 1);
        sel = byte_sel(2 * gg);
    }
    WM_DEV void half(int h) {
        s2[0] = byte_h1024(sc[h], sel) - h2(1024.0f);
        c2[0] = s2[0] * h2(-1024.0f);
        // the high nibbles are decoded as 1024 + 16 q
        s2[1] = fma2(byte_h1024(sc[h], sel + 0x00010001u), h2(0.0625f), h2(-64.0f));
        c2[1] = s2[1] * h2(-1024.0f);
        m2[0] = byte_h1024(mn[h], sel) - h2(1024.0f);
        m2[1] = byte_h1024(mn[h], sel + 0x00010001u) - h2(1024.0f);
    }
    WM_DEV f16x8 unit(int h, int u, uint32_t k64) const {
        const int n = u >> 1;                    // nibble
        f16x2 v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int k = 2 * (u & 1) + i;
            const uint32_t w = q[h][k], m = n ? 0x00F000F0u : 0x000F000Fu;
            uint32_t e = field(w, m, k64), o = field(w >> 8, m, k64);
            if constexpr (BITS == 5) {
                // fifth bits: bit 4 h + 2 gg + n of byte l, to bit 4 (low nibble) or 8 (high) of the half
                const uint32_t b = qh[k] >> (4 * h + 2 * gg), bm = n ? 0x01000100u : 0x00100010u;
                e |= (n ? b << 7 : b << 4) & bm;
                o |= (n ? b >> 1 : b >> 4) & bm;
            }
            v[2 * i] = fma2(as_h2(e), s2[n], c2[n]);
            v[2 * i + 1] = fma2(as_h2(o), s2[n], c2[n]);
        }
        return cat4(v[0], v[1], v[2], v[3]);
    }
    WM_DEV f16x8 mins(int u) const { return rep4(m2[u >> 1]); }
};
template <> struct KqRow<Q4_K> : Kq45<4> {};     // q4k_dequant.h:28-33, 43-60, 112-168
template <> struct KqRow<Q5_K> : Kq45<5> {};     // q5k_dequant.h:19-25, 98-131

// Q6_K (q6k_dequant.h:20-25, 112-141): column 128 h + 32 j + l; ql[64 h +
// 32 (j & 1) + l] (low nibble for j < 2, high else), qh[32 h + l] bits 2 j.
// This lane: ql bytes 64 h + 16 g .. + 15 (j & 1 = g / 2, l = 16 (g & 1) ..):
// low nibbles in sub-block 8 h + g, high nibbles in 8 h + 4 + g.  scale = 16
// s1 + s0 with s0 in [-8, 8]: unit(h, u, 1) = q s1, unit(h, u, 0) = q s0, both
// exact, and 16 |s1| <= |scale| + 8, so that the two sums do not cancel (with
// s0 in [0, 15] a scale of -1 is -16 + 15: rows of such scales then missed the
// negative of the rows with scale 1 by 2.3e-6; now by 3 to 6e-8).
template <> struct KqRow<Q6_K> {
    static constexpr int AL = 2;
    static constexpr bool FOLD = false, MINS = false;
    uint32_t ql[2][4], qh[2][4];
    int sb[4];                                   // scales of sub-blocks 4 i + g
    uint32_t d16, sh;
    float d;
    f16x2 s2[2][2], c2[2][2];                    // [nibble][part]
    WM_DEV static int col(int h, int u, int g) { return 128 * h + 32 * (g >> 1) + 16 * (g & 1) + 64 * (u >> 1) + 8 * (u & 1); }
    WM_DEV void load(const uint8_t* slot, int o, int g) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            ld_dw<AL, 4>(slot, o + 64 * h + 16 * g, ql[h]);
            ld_dw<AL, 4>(slot, o + 128 + 32 * h + 16 * (g & 1), qh[h]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) sb[i] = *(const int8_t*)(slot + o + 192 + 4 * i + g);
        d16 = *(const uint16_t*)(slot + o + 208);
    }
    WM_DEV void pin() {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            pin_dw(ql[h]);
            pin_dw(qh[h]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) asm volatile("" : "+v"(sb[i]));
        asm volatile("" : "+v"(d16));
    }
    WM_DEV void head(int g) {
        d = h2f(d16);
        sh = 4 - 2 * (g >> 1);
    }
    WM_DEV void half(int h) {
#pragma unroll
        for (int n = 0; n < 2; n++) {
            // s1 = the scale / 16 rounded (fp16 holds the integers around 1536 and no fractions), s0 the rest in [-8, 8]
            const _Float16 sv = (_Float16)(int16_t)sb[2 * h + n];
            const f16x2 s = {sv, sv}, s1 = fma2(s, h2(0.0625f), h2(1536.0f)) - h2(1536.0f), s0 = fma2(s1, h2(-16.0f), s);
#pragma unroll
            for (int part = 0; part < 2; part++) {
                const f16x2 f = part ? s1 : s0;
                s2[n][part] = n ? f * h2(0.0625f) : f;
                // 1024 + 32 (values q + 32), or (1024 + 16 * 32) / 16; |f| <= 8: exact
                c2[n][part] = n ? f * h2(-96.0f) : f * h2(-1056.0f);
            }
        }
    }
    // the 8 values as 1024 + (q + 32) (low nibbles) or 1024 + 16 (q + 32)
    WM_DEV void raw(int h, int u, uint32_t k64, f16x2* v) const {
        const int n = u >> 1;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int k = 2 * (u & 1) + i;
            const uint32_t w = ql[h][k], m = n ? 0x00F000F0u : 0x000F000Fu;
            // bits 2 j of qh byte l to bit 4 (j < 2) or 8 (j >= 2: 4 bits further up both)
            const uint32_t bm = n ? 0x03000300u : 0x00300030u;
            v[2 * i] = as_h2(field(w, m, k64) | ((qh[h][k] << sh) & bm));
            v[2 * i + 1] = as_h2(field(w >> 8, m, k64) | ((qh[h][k] >> (8 - sh)) & bm));
        }
    }
    WM_DEV f16x8 unit(const f16x2* v, int u, int part) const {
        const int n = u >> 1;
        return cat4(fma2(v[0], s2[n][part], c2[n][part]), fma2(v[1], s2[n][part], c2[n][part]),
                    fma2(v[2], s2[n][part], c2[n][part]), fma2(v[3], s2[n][part], c2[n][part]));
    }
};

// Q2_K and Q3_K: column 128 h + 32 j + l is (qs[32 h + l] >> 2 j) & 3; unit u
// = j; this lane: bytes l = 8 g .. + 7; sub-block 8 h + 2 j + g / 2.
// Decoded as 1024 + 4^j value.
template <> struct KqRow<Q3_K> {                 // hmask[32] qs[64] scales[12] d
    static constexpr int AL = 2;
    static constexpr bool FOLD = true, MINS = false;
    uint32_t q[2][2], hm[2], s3[3], d16;
    float d, dmin;
    uint32_t sc[4];                              // sub-blocks 4i .. 4i+3: the 6-bit scale + 32 (a byte each)
    uint32_t gg;
    f16x2 s2[4];
    WM_DEV static int col(int h, int u, int g) { return 128 * h + 32 * u + 8 * g; }
    WM_DEV void load(const uint8_t* slot, int o, int g) {
        ld_dw<AL, 2>(slot, o + 8 * g, hm);
        ld_dw<AL, 2>(slot, o + 32 + 8 * g, q[0]);
        ld_dw<AL, 2>(slot, o + 64 + 8 * g, q[1]);
        ld_dw<AL, 3>(slot, o + 96, s3);
        d16 = *(const uint16_t*)(slot + o + 108);
    }
    WM_DEV void pin() {
        pin_dw(hm);
        pin_dw(q[0]);
        pin_dw(q[1]);
        pin_dw(s3);
        asm volatile("" : "+v"(d16));
    }
    WM_DEV void head(int g) {
        d = h2f(d16);
        dmin = 0.0f;
        gg = (uint32_t)(g >> 1);
        // low 4 bits: bytes 0-7 of the scales (sub-blocks 0-7), their high
        // nibbles (8-15); high 2 bits: bits 2(k / 4) of byte 8 + k % 4
        sc[0] = (s3[0] & 0x0F0F0F0Fu) | ((s3[2] << 4) & 0x30303030u);
        sc[1] = (s3[1] & 0x0F0F0F0Fu) | ((s3[2] << 2) & 0x30303030u);
        sc[2] = ((s3[0] >> 4) & 0x0F0F0F0Fu) | (s3[2] & 0x30303030u);
        sc[3] = ((s3[1] >> 4) & 0x0F0F0F0Fu) | ((s3[2] >> 2) & 0x30303030u);
    }
    WM_DEV void half(int h) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = 8 * h + 2 * j;         // + gg
            const float p = 1.0f / (float)(1 << (2 * j));
            s2[j] = fma2(byte_h1024(sc[k >> 2], byte_sel((uint32_t)(k & 3) + gg)), h2(p), h2(-1056.0f * p));
        }
    }
    // value low bits + 4 * (hmask bit 4 h + j) - 4, times 4^j; its product with sc / 4^j is exact (|q sc| <= 128)
    WM_DEV f16x8 unit(int h, int j, uint32_t k64) const {
        const uint32_t m = 0x00030003u << (2 * j), bm = 0x00040004u << (2 * j);
        const int up = j + 2 - 4 * h, dn = 6 + 4 * h - j;      // bit 4 h + j of byte 0 / byte 1 to bit 2 j + 2
        const f16x2 bias = h2(-(float)(1024 + (4 << (2 * j))));
        f16x2 v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t b0 = up >= 0 ? hm[i] << (up & 31) : hm[i] >> ((-up) & 31);
            v[2 * i] = (as_h2(field(q[h][i], m, k64) | (b0 & bm)) + bias) * s2[j];
            v[2 * i + 1] = (as_h2(field(q[h][i] >> 8, m, k64) | ((hm[i] >> dn) & bm)) + bias) * s2[j];
        }
        return cat4(v[0], v[1], v[2], v[3]);
    }
    WM_DEV f16x8 mins(int) const { return (f16x8){}; }
};

template <> struct KqRow<Q2_K> {                 // scales[16] qs[64] d dmin
    static constexpr int AL = 4;
    static constexpr bool FOLD = true, MINS = true;
    uint32_t q[2][2], sb[4], dd;                 // sub-blocks 4i .. 4i+3: scale (low nibble), min (high)
    float d, dmin;
    uint32_t gg;
    f16x2 s2[4], c2[4], m2[4];
    WM_DEV static int col(int h, int u, int g) { return 128 * h + 32 * u + 8 * g; }
    WM_DEV void load(const uint8_t* slot, int o, int g) {
        ld_dw<AL, 4>(slot, o, sb);
        ld_dw<AL, 2>(slot, o + 16 + 8 * g, q[0]);
        ld_dw<AL, 2>(slot, o + 48 + 8 * g, q[1]);
        ld_dw<AL, 1>(slot, o + 80, &dd);
    }
    WM_DEV void pin() {
        pin_dw(sb);
        pin_dw(q[0]);
        pin_dw(q[1]);
        asm volatile("" : "+v"(dd));
    }
    WM_DEV void head(int g) {
        d = h2f(dd);
        dmin = h2f(dd >> 16);
        gg = (uint32_t)(g >> 1);
    }
    WM_DEV void half(int h) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = 8 * h + 2 * j;         // + gg
            const uint32_t sel = byte_sel((uint32_t)(k & 3) + gg);
            const float p = 1.0f / (float)(1 << (2 * j));
            s2[j] = fma2(byte_h1024(sb[k >> 2] & 0x0F0F0F0Fu, sel), h2(p), h2(-1024.0f * p));
            c2[j] = s2[j] * h2(-1024.0f);
            m2[j] = byte_h1024((sb[k >> 2] >> 4) & 0x0F0F0F0Fu, sel) - h2(1024.0f);
        }
    }
    WM_DEV f16x8 unit(int h, int j, uint32_t k64) const {
        const uint32_t m = 0x00030003u << (2 * j);
        f16x2 v[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            v[2 * i] = fma2(as_h2(field(q[h][i], m, k64)), s2[j], c2[j]);
            v[2 * i + 1] = fma2(as_h2(field(q[h][i] >> 8, m, k64)), s2[j], c2[j]);
        }
        return cat4(v[0], v[1], v[2], v[3]);
    }
    WM_DEV f16x8 mins(int j) const { return rep4(m2[j]); }
};

// 8 Q8_0 blocks of a row: block 4 h + u of the chunk is unit (h, u); this lane
// holds columns 8 g .. + 7 of each (in order).  Blocks start 2 bytes past a
// dword (even ones) or at one (odd ones).
template <> struct KqRow<Q8_0> {
    static constexpr int AL = 16;
    static constexpr bool FOLD = false, MINS = false;
    uint32_t w[8][3];
    uint32_t d16[8];
    WM_DEV static int col(int h, int u, int g) { return 128 * h + 32 * u + 8 * g; }
    WM_DEV void load(const uint8_t* slot, int o, int g) {
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int off = 34 * b + 2;
            const uint32_t* p = (const uint32_t*)(slot + o + (off & ~3) + 8 * g);
            w[b][0] = p[0];
            w[b][1] = p[1];
            if ((off & 3) != 0) w[b][2] = p[2];
            d16[b] = *(const uint16_t*)(slot + o + 34 * b);
        }
    }
    // the decode is short: keeping only its start apart was faster (4096 tokens 3584 us per batch, with every
    // register unknown 3627)
    WM_DEV void pin() { asm volatile("" ::: "memory"); }
    WM_DEV float scale(int b) const { return h2f(d16[b]); }
    WM_DEV f16x8 unit(int b) const {
        const uint32_t K = 0x64646464u, X = 0x80808080u;
        const uint32_t d0 = w[b][0] ^ X, d1 = w[b][1] ^ X;
        uint32_t h[4];
        if ((b & 1) != 0) {
            h[0] = __builtin_amdgcn_perm(K, d0, 0x04010400u);
            h[1] = __builtin_amdgcn_perm(K, d0, 0x04030402u);
            h[2] = __builtin_amdgcn_perm(K, d1, 0x04010400u);
            h[3] = __builtin_amdgcn_perm(K, d1, 0x04030402u);
        } else {
            const uint32_t d2 = w[b][2] ^ X;
            h[0] = __builtin_amdgcn_perm(K, d0, 0x04030402u);
            h[1] = __builtin_amdgcn_perm(K, d1, 0x04010400u);
            h[2] = __builtin_amdgcn_perm(K, d1, 0x04030402u);
            h[3] = __builtin_amdgcn_perm(K, d2, 0x04010400u);
        }
        const f16x2 bias = h2(1152.0f);
        return cat4(as_h2(h[0]) - bias, as_h2(h[1]) - bias, as_h2(h[2]) - bias, as_h2(h[3]) - bias);
    }
};

// ------------------------------------------------------------------ the kernel

// N partial sums LD floats apart, added in order.
template <int N, int LD> WM_DEV float sum_slices(const float* p) {
    float t[N];
#pragma unroll
    for (int i = 0; i < N; i++) t[i] = p[i * LD];
    float v = t[0];
#pragma unroll
    for (int i = 1; i < N; i++) v += t[i];
    return v;
}

WM_DEV f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// AHL = 1: gate and up tiles in turn (NSUB = 2; activations: the tokens' x),
// SwiGLU epilogue.  AHL = 2: down (activations: the pairs' SwiGLU outputs as
// hi + lo), fp32 output.  WT: the weight format of every matrix the launch
// reads; M: pairs per pass; NSB: 256-column super-blocks per ring slot.
//
// The items of one launch list (n_r routed ones, then the shared ones, up to
// n_items) that this workgroup takes.  The list begins at position lo of the
// launch's `total`, R row blocks per pass.
#if defined(__HIP_DEVICE_COMPILE__)      // (buffer resources are device types)
template <int AHL, int WT, int M, int NSB, int CW>
WM_DEV void pf_gemm_items(const PfGemm& a, int n_rp, int n_r, int n_items, int lo, int total, int R) {
    typedef GmGeo<AHL, WT, M, NSB, CW> G;
    typedef KqRow<WT> F;
    constexpr int S = G::S, MT = G::MT, NI = G::NI, MSL = G::MSL, NSUB = G::NSUB;
    extern __shared__ __attribute__((aligned(16))) uint8_t gsm[];
    // the wave index is uniform: readfirstlane lets the compiler keep what depends on it in SGPRs
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
    const int grid = (int)gridDim.x, full = total / grid;
    const int kl = pf_item_slot((int)blockIdx.x, grid, R), kf = M == 32 ? pf_item_slot_full((int)blockIdx.x, grid) : kl;
    int i0 = lo / grid;
    if (i0 * grid + (i0 < full ? kf : kl) < lo) ++i0;

    // item i of this workgroup: pass, first matrix row
    auto item = [&](int i, int& pass, int& row) __attribute__((always_inline)) -> bool {
        const int q = i0 + i, j = q * grid + (q < full ? kf : kl) - lo;
        if (j >= n_items) return false;
        if (j < n_r) {
            pass = j / a.nrb_r;
            row = (j - pass * a.nrb_r) * a.rows_item;
        } else {
            const int q = (j - n_r) / a.nrb_s;
            row = ((j - n_r) - q * a.nrb_s) * a.rows_item;
            pass = n_rp + q;
        }
        return true;
    };
    // this wave's slice and row group; a step is 16 rows of each group
    const int nsl = 1 << a.lsl, sl = wave & (nsl - 1), rgrp = wave >> a.lsl, nrg = CW >> a.lsl;
    const int nsteps = a.rows_item / (16 * nrg);
    const int ns = MSL == 2 ? a.ns : 1;
    const uint32_t rb = (uint32_t)a.rb;

    // ---- the weight ring.  DMA instruction t of a slot covers granules p =
    // 64 t + lane: granule p % GR of row p / GR of the tile (16 rows' bytes
    // are a multiple of 16, so the row starts' distances past a 16-byte
    // boundary are those of rows 0-15).  Sources are bounds-checked buffer
    // resources (a read past the matrix returns zeros).
    uint32_t voff[NI];
#pragma unroll
    for (int t = 0; t < NI; t++) {
        const int p = 64 * t + lane, r = p / G::GR;
        voff[t] = (((uint32_t)r * rb) & ~15u) + 16u * (uint32_t)(p - G::GR * r);
    }
    lds8_t* ring = (lds8_t*)gsm + wave * (S * G::SLOT);
    int ii = 0, ip = 0, irow = 0, ist = 0, imat = 0, isl = 0, islot = 0, outst = 0, ige = 0, ipn = 0, irown = 0;
    bool iok = item(0, ip, irow), inok = false;
    __amdgpu_buffer_rsrc_t rW0, rW1;
    auto expert_of = [&](int pass) __attribute__((always_inline)) { return ((cint_t*)a.recs)[(int64_t)pass * GM_REC]; };
    // the issue item's sources; the next item's expert is read ahead
    auto setup_issue = [&](int ge) __attribute__((always_inline)) {
        const bool shared = ip >= n_rp;
        const int mb = shared ? a.mb_s : a.mb_r;
        rW0 = gm_rsrc(shared ? a.s0 : a.w0 + (int64_t)ge * a.st0, mb);
        rW1 = G::GU ? gm_rsrc(shared ? a.s1 : a.w1 + (int64_t)ge * a.st1, mb) : rW0;
        irow += 16 * rgrp;
        inok = item(ii + 1, ipn, irown);
        if (inok) ige = expert_of(ipn);
    };
    auto issue_next = [&]() __attribute__((always_inline)) {
        lds8_t* dst = ring + islot * G::SLOT;
        const uint32_t colb = (uint32_t)((sl * ns + isl) * G::CHUNK);
        const uint32_t soff = (uint32_t)irow * rb + (colb & ~15u);
        // The lanes past a slot's last granule stay out of its last
        // instruction.  The lane number is opaque at each use: a compiler that
        // knows two of these conditions equal may run the code between them
        // once for either side, and a DMA whose lanes are so split writes to
        // one side's address.
        int ln = lane;
        asm volatile("" : "+v"(ln));
#pragma unroll
        for (int t = 0; t < NI; t++)
            if (16 * G::GR >= 64 * (t + 1) || ln < 16 * G::GR - 64 * t)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(NSUB == 2 && imat ? rW1 : rW0, (lds_void*)(dst + 1024 * t), 16,
                                                         voff[t], soff, 0, 0);
        islot = islot + 1 == S ? 0 : islot + 1;
        ++outst;
        if (++isl < ns) return;
        isl = 0;
        if (++imat < NSUB) return;
        imat = 0;
        irow += 16 * nrg;
        if (++ist < nsteps) return;
        ist = 0;
        ++ii;
        iok = inok;
        if (iok) {
            ip = ipn;
            irow = irown;
            setup_issue(ige);
        }
    };

    // ---- items: the record's parts this lane uses, the activations
    // outputs of a tile: thread tid sums position tid & 255 of row tile
    // tmt + q, that is pair om + 16 q of the pass and row orow of the 16
    constexpr int NO = CW == 4 ? MT : 1;
    const int tmt = CW == 8 && MT == 2 ? tid >> 8 : 0, om = 16 * tmt + 4 * ((tid & 255) >> 6) + (tid & 3), orow = (tid >> 2) & 15;
    struct Rec {
        int n, xe[NO];                 // pairs; gate/up: the x exponents of this thread's output pairs
        int pid[MT];                   // pair of operand row c (c = 4g + i: of accumulator row i)
    };
    auto load_rec = [&](int pass, Rec& r) __attribute__((always_inline)) {
        const int32_t* p = a.recs + (int64_t)pass * GM_REC;
        r.n = ((cint_t*)a.recs)[(int64_t)pass * GM_REC + 1];
#pragma unroll
        for (int q = 0; q < NO; q++) r.xe[q] = G::GU ? (int)((const int8_t*)(p + 4 + GM_M))[om + 16 * q] : 0;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) r.pid[mt] = p[4 + 16 * mt + c];
    };
    u32x4 A[AHL][MT][MSL][8 * NSB];
    f32x4 asc[MT][G::GU ? 1 : MSL][G::GU ? 1 : 2 * NSB];
    const int scol = sl * ns * G::KC;              // first column of the slice
    auto load_act = [&](const Rec& r) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            if (mt && r.n <= 16) continue;
            const int64_t row = G::GU ? pair_token(r.pid[mt], a.T, a.K) : r.pid[mt];
            int pr[4];                 // down: pairs of accumulator rows 4g .. 4g + 3
            if constexpr (!G::GU) {
#pragma unroll
                for (int i = 0; i < 4; i++) pr[i] = __shfl(r.pid[mt], 4 * g + i);
            }
#pragma unroll
            for (int s = 0; s < MSL; s++) {
                if (s && s >= ns) continue;
                const int64_t at = row * a.a_ld + scol + s * G::KC;
#pragma unroll
                for (int b = 0; b < 8 * NSB; b++) {
                    const int co = 256 * (b >> 3) + F::col((b >> 2) & 1, b & 3, g);
                    A[0][mt][s][b] = *(const u32x4*)(a.a_hi + at + co);
                    if constexpr (AHL == 2) A[AHL - 1][mt][s][b] = *(const u32x4*)(a.a_lo + at + co);
                }
                if constexpr (!G::GU) {
                    const int k = (scol + s * G::KC) / 128;
#pragma unroll
                    for (int h = 0; h < 2 * NSB; h++)
#pragma unroll
                        for (int i = 0; i < 4; i++) asc[mt][s][h][i] = a.a_sc[(int64_t)pr[i] * a.sc_ld + k + h];
                }
            }
        }
    };
    // the current pass fills its second row tile: a pass of 32 with 16 pairs or
    // fewer leaves that tile's loads, products and sums out (2000 tokens Q4_K,
    // about 12 pairs per expert: 1653 -> 1455 us per batch; a launch whose passes
    // are all full pays up to 4 % for the branch)
    bool two = false;
    // K-quant operands hold their 8 columns in the order 0 2 1 3 4 6 5 7
    auto order_act = [&]() __attribute__((always_inline)) {
        if constexpr (G::KQ) {
#pragma unroll
            for (int h = 0; h < AHL; h++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int s = 0; s < MSL; s++) {
                        if ((mt && !two) || (s && s >= ns)) continue;
#pragma unroll
                        for (int b = 0; b < 8 * NSB; b++) {
                            const u32x4 v = A[h][mt][s][b];
                            A[h][mt][s][b] = (u32x4){__builtin_amdgcn_perm(v[1], v[0], 0x05040100u),
                                                     __builtin_amdgcn_perm(v[1], v[0], 0x07060302u),
                                                     __builtin_amdgcn_perm(v[3], v[2], 0x05040100u),
                                                     __builtin_amdgcn_perm(v[3], v[2], 0x07060302u)};
                        }
                    }
        }
    };

    // ---- one ring slot: wait for it, take it into registers, refill it (take);
    // add its products with the first MN row tiles of the pass to acc (sums)
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t k64 = opaque_e1024();
    const int rsh = (int)(((uint32_t)c * rb) & 15u);         // row c's start past a 16-byte boundary
    int cslot = 0;
    auto take = [&](auto s_tag, F(&row)[NSB]) __attribute__((always_inline)) {
        constexpr int SI = decltype(s_tag)::value;
        if (outst == S) WM_WAIT_VMCNT((S - 1) * NI);
        else WM_WAIT_VMCNT(0);
        asm volatile("" ::: "memory");
        const uint8_t* rowp = gsm + wave * (S * G::SLOT) + cslot * G::SLOT + c * G::RSLOT;
        const int o = F::AL >= 16 ? 0 : rsh + (((sl * ns + SI) * G::CHUNK) & 15);
#pragma unroll
        for (int sb = 0; sb < NSB; sb++) row[sb].load(rowp, o + sb * (G::CHUNK / NSB), g);
        gm_wait_lds();
        --outst;
        cslot = cslot + 1 == S ? 0 : cslot + 1;
        if (iok) issue_next();
    };
    auto sums = [&](auto s_tag, auto m_tag, F(&row)[NSB], f32x4(&acc)[MT]) __attribute__((always_inline)) {
        constexpr int SI = decltype(s_tag)::value, MN = decltype(m_tag)::value;
#pragma unroll
        for (int sb = 0; sb < NSB; sb++) {
            F& f = row[sb];
            if constexpr (!G::KQ) {
                f32x4 t[2][MN];
#pragma unroll
                for (int mt = 0; mt < MN; mt++) t[0][mt] = t[1][mt] = zero;
                // the scaling of a block's products comes after the next
                // block's MFMAs are sent, so that it does not wait for them
                f32x4 P[2][MN];
#pragma unroll
                for (int b = 0; b <= 8; b++) {
                    if (b < 8) {
                        const f16x8 B = f.unit(b);
#pragma unroll
                        for (int mt = 0; mt < MN; mt++) {
                            P[b & 1][mt] = mfma16(__builtin_bit_cast(f16x8, A[0][mt][SI][8 * sb + b]), B, zero);
                            if constexpr (AHL == 2)
                                P[b & 1][mt] = mfma16(__builtin_bit_cast(f16x8, A[AHL - 1][mt][SI][8 * sb + b]), B, P[b & 1][mt]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (b > 0) {
                        const float d = f.scale(b - 1);
#pragma unroll
                        for (int mt = 0; mt < MN; mt++) {
                            f32x4& r = G::GU ? acc[mt] : t[(b - 1) >> 2][mt];
#pragma unroll
                            for (int i = 0; i < 4; i++) r[i] = fmaf(d, P[(b - 1) & 1][mt][i], r[i]);
                        }
                    }
                }
                if constexpr (!G::GU) {
#pragma unroll
                    for (int mt = 0; mt < MN; mt++)
#pragma unroll
                        for (int h = 0; h < 2; h++)
#pragma unroll
                            for (int i = 0; i < 4; i++) acc[mt][i] = fmaf(asc[mt][SI][2 * sb + h][i], t[h][mt][i], acc[mt][i]);
                }
            } else {
                f.head(g);
                // NQ sums: the products with q sc (Q6_K: with q s1 and q s0);
                // the mins.  Gate/up: over the super-block, down: per half.
                constexpr int NQ = F::FOLD ? 1 : 2;
                f32x4 sq[NQ][MN], sm[MN];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if (h == 0 || !G::GU) {
#pragma unroll
                        for (int mt = 0; mt < MN; mt++) {
#pragma unroll
                            for (int k = 0; k < NQ; k++) sq[k][mt] = zero;
                            sm[mt] = zero;
                        }
                    }
                    f.half(h);
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        f16x8 B[NQ], Bm;
                        if constexpr (F::FOLD) {
                            B[0] = f.unit(h, u, k64);
                            if constexpr (F::MINS) Bm = f.mins(u);
                        } else {
                            f16x2 v[4];
                            f.raw(h, u, k64, v);
#pragma unroll
                            for (int k = 0; k < NQ; k++) B[k] = f.unit(v, u, k);
                        }
#pragma unroll
                        for (int mt = 0; mt < MN; mt++)
#pragma unroll
                            for (int l = 0; l < AHL; l++) {
                                const f16x8 av = __builtin_bit_cast(f16x8, A[l][mt][SI][8 * sb + 4 * h + u]);
#pragma unroll
                                for (int k = 0; k < NQ; k++) sq[k][mt] = mfma16(av, B[k], sq[k][mt]);
                                if constexpr (F::MINS) sm[mt] = mfma16(av, Bm, sm[mt]);
                            }
                    }
                    if (h == 1 || !G::GU) {
#pragma unroll
                        for (int mt = 0; mt < MN; mt++) {
                            f32x4 r = G::GU ? acc[mt] : zero;
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                r[i] = fmaf(f.d, sq[0][mt][i], r[i]);
                                if constexpr (!F::FOLD) r[i] = fmaf(16.0f * f.d, sq[NQ - 1][mt][i], r[i]);
                                if constexpr (F::MINS) r[i] = fmaf(-f.dmin, sm[mt][i], r[i]);
                                if constexpr (!G::GU) r[i] = fmaf(asc[mt][SI][2 * sb + h][i], r[i], acc[mt][i]);
                            }
                            acc[mt] = r;
                        }
                    }
                }
            }
        }
    };
    auto slot = [&](auto s_tag, f32x4(&acc)[MT]) __attribute__((always_inline)) {
        F row[NSB];
        take(s_tag, row);
        if constexpr (MT == 1) sums(s_tag, std::integral_constant<int, 1>{}, row, acc);
        else if (two) sums(s_tag, std::integral_constant<int, 2>{}, row, acc);
        else {
#pragma unroll
            for (int sb = 0; sb < NSB; sb++) row[sb].pin();
            sums(s_tag, std::integral_constant<int, 1>{}, row, acc);
        }
    };

    // ---- a tile's partial sums, in slice order, to out(pair slot group, value)
    int pbuf = 0, ci = 0, cp = 0, crow = 0;
    Rec cur, nxt;
    int own[NO];
    float* stg = (float*)(gsm + G::STG);
    auto finish = [&](int mat, int st, const f32x4(&acc)[MT]) __attribute__((always_inline)) {
        float* pb = (float*)(gsm + G::PBASE + pbuf * G::PART);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
            if (!mt || two) *(f32x4*)(pb + (wave * MT + mt) * 256 + 4 * lane) = acc[mt];
        gm_bar();
        pbuf ^= 1;
        // r: row group of this thread's q-th output
        auto reduce = [&](int r, int q) __attribute__((always_inline)) {
            const float* p = pb + (((r << a.lsl) * MT + tmt + q) * 256) + (tid & 255);
            float v;
            if (CW == 8 && a.lsl == 3) v = sum_slices<8, MT * 256>(p);
            else if (a.lsl == 2) v = sum_slices<4, MT * 256>(p);
            else if (a.lsl == 1) v = sum_slices<2, MT * 256>(p);
            else v = p[0];
            const int row = 16 * (st * nrg + r) + orow;
            if constexpr (G::GU) {
                float* sp = stg + (om + 16 * q) * GM_SLD + row;
                if (mat == 0) *sp = v;
                else {
                    const float xs = ldexpf(1.0f, cur.xe[q]);
                    *sp = silu_mul(*sp * xs, v * xs);
                }
            } else {
                if (om + 16 * q < cur.n) a.y[(int64_t)own[q] * a.y_ld + crow + row] = v;
            }
        };
        if constexpr (CW == 4 || MT == 2) {
            for (int r = 0; r < nrg; r++)
#pragma unroll
                for (int q = 0; q < NO; q++)
                    if (!(tmt + q) || two) reduce(r, q);
        } else if (nrg == 1) {
            if ((tid >> 8) == (st & 1)) reduce(0, 0);        // 4 waves each, in turn
        } else {
            for (int r = tid >> 8; r < nrg; r += 2) reduce(r, 0);
        }
    };

    if (!item(0, cp, crow)) return;
    load_rec(cp, cur);
    setup_issue(expert_of(cp));
    for (int s = 0; s < S && iok; s++) issue_next();
    load_act(cur);
    int np = 0, nrow = 0;
    bool nok = item(1, np, nrow);
    if (nok) load_rec(np, nxt);
    else nxt = cur;
    for (;;) {
        two = MT > 1 && cur.n > 16;
        order_act();
        // the next record is in (its loads are older than the activations' wait)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) asm volatile("" : "+v"(nxt.pid[mt]));
#pragma unroll
        for (int q = 0; q < NO; q++) {
            if constexpr (G::GU) asm volatile("" : "+v"(nxt.xe[q]));
            // this thread's output pairs are those of operand rows om % 16
            else own[q] = __shfl(CW == 4 ? cur.pid[q] : tmt ? cur.pid[MT - 1] : cur.pid[0], om & 15);
        }
        f32x4 acc[MT];
        for (int st = 0;; st++) {
#pragma unroll
            for (int mat = 0; mat < NSUB; mat++) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[mt] = zero;
                slot(std::integral_constant<int, 0>{}, acc);
                if constexpr (MSL == 2) {
                    if (ns == 2) slot(std::integral_constant<int, MSL - 1>{}, acc);
                }
                if (mat < NSUB - 1) finish(mat, st, acc);
            }
            if (st == nsteps - 1) break;
            finish(NSUB - 1, st, acc);
        }
        // the next item's activations load while the last tile is finished
        if (nok) load_act(nxt);
        finish(NSUB - 1, nsteps - 1, acc);
        if constexpr (G::GU) {
            // wave w: pairs w, w + CW, ..: scale by a power of two, split into hi + lo
            gm_bar();
            const int32_t* rec = a.recs + (int64_t)cp * GM_REC;
            for (int m = wave; m < cur.n; m += CW) {
                const float2 v = *(const float2*)(stg + m * GM_SLD + 2 * lane);
                float mx = fmaxf(fabsf(v.x), fabsf(v.y));
                mx = fmaxf(mx, dpp_f32<DPP_ROR8>(mx));
                mx = fmaxf(mx, dpp_f32<DPP_ROR4>(mx));
                mx = fmaxf(mx, dpp_f32<DPP_ROR2>(mx));
                mx = fmaxf(mx, dpp_f32<DPP_ROR1>(mx));
                const int mi = __builtin_bit_cast(int, mx);
                const float m01 = fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(mi, 0)),
                                        __builtin_bit_cast(float, __builtin_amdgcn_readlane(mi, 16)));
                const float m23 = fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(mi, 32)),
                                        __builtin_bit_cast(float, __builtin_amdgcn_readlane(mi, 48)));
                const int e = pf_exp(fmaxf(m01, m23));
                const float sc = ldexpf(1.0f, -e);
                const float x0 = v.x * sc, x1 = v.y * sc;
                const f16x2 hv = {(_Float16)x0, (_Float16)x1};
                const f16x2 lv = {(_Float16)(x0 - (float)hv[0]), (_Float16)(x1 - (float)hv[1])};
                const int64_t pr = ((cint_t*)a.recs)[(int64_t)cp * GM_REC + 4 + m], at = pr * a.o_ld + crow + 2 * lane;
                *(uint32_t*)(a.o_hi + at) = __builtin_bit_cast(uint32_t, hv);
                *(uint32_t*)(a.o_lo + at) = __builtin_bit_cast(uint32_t, lv);
                if (lane == 0) a.o_sc[pr * a.osc_ld + crow / GM_ROWS] = ldexpf(1.0f, e);
            }
        }
        if (!nok) break;
        ++ci;
        cp = np;
        crow = nrow;
        cur = nxt;
        nok = item(ci + 1, np, nrow);
        if (nok) load_rec(np, nxt);
    }
}
#endif

// A CU holds 8 waves either way: one workgroup of 8, or two of 4.
template <int AHL, int WT, int M, int NSB, int CW>
__global__ __launch_bounds__(64 * CW, 2) void k_pf_gemm(PfGemm a) {
#if defined(__HIP_DEVICE_COMPILE__)
    const int n_rp = a.npass[0], n_r = a.sel == 2 ? 0 : n_rp * a.nrb_r;
    const int n = n_r + (a.sel == 1 ? 0 : a.npass[1] * a.nrb_s);
    pf_gemm_items<AHL, WT, M, NSB, CW>(a, n_rp, n_r, n, 0, n, a.sel == 2 ? a.nrb_s : a.nrb_r);
#endif
}

// Routed passes in format WT, then the shared expert's in format SWT, in one
// launch: the shared items go on where the routed ones ended, so that the
// workgroups without an item of the last round take them.  A launch of their
// own left most of the chip idle at both ends: 2 passes of gate/up are 16
// items, 38 us.  23 tokens through 512 experts of H 4096, I 1024, Q4_K, Q6_K,
// top-3, Q8_0 shared: 231 us per batch with two launches, 208 with one (the
// same bits).
template <int AHL, int WT, int M, int NSB, int SWT, int CW>
__global__ __launch_bounds__(64 * CW, 2) void k_pf_gemm2(PfGemm r, PfGemm s) {
#if defined(__HIP_DEVICE_COMPILE__)
    const int n_rp = r.npass[0], n_r = n_rp * r.nrb_r, n_s = s.npass[1] * s.nrb_s;
    pf_gemm_items<AHL, WT, M, NSB, CW>(r, n_rp, n_r, n_r, 0, n_r + n_s, r.nrb_r);
    __syncthreads();                             // the ring and the staging change hands
    pf_gemm_items<AHL, SWT, M, 1, CW>(s, n_rp, 0, n_s, n_r, n_r + n_s, r.nrb_r);
#endif
}

// Slices and ring slots of a launch; false if the shape does not fit.
template <class G> bool pf_gemm_plan(PfGemm& h, int cw) {
    const int slice = gm_slice(G::GU, h.ncol), nsl = h.ncol / slice;
    h.ns = slice / G::KC;
    h.lsl = nsl == 1 ? 0 : nsl == 2 ? 1 : nsl == 4 ? 2 : 3;
    // whole slots and slices, no more slices than waves; a step's rows divide an item's
    return !(slice % G::KC || h.ns > G::MSL || h.ncol % slice || (1 << h.lsl) != nsl || nsl > cw || h.rows_item % 128);
}

// Waves of a workgroup: 4, two workgroups to a CU, when the row has no more
// than 4 slices; one of 8 else.  The waves of a workgroup meet once per tile,
// and those of the two workgroups do not wait for each other: one computes
// while the other is at its barrier or waits for its partial sums.  us per
// batch with one workgroup of 8 / two of 4 (the same bits): H 4096, I 1024
// (down alone), Q8_0 top-10 at 512 tokens 1404 / 1399, at 4096 tokens 3988 /
// 3639; Q4_K, Q6_K top-3 at 512 tokens 993 / 959, at 2000 1473 / 1425; H 2048,
// I 512 (both), Q8_0 top-4 of 64 at 1001 tokens 201 / 174 (at 8 tokens, where
// few items are left to share, 63 / 69).
WM_HD inline int gm_waves(bool gateup, int ncol) { return ncol / gm_slice(gateup, ncol) <= 4 ? 4 : 8; }

template <int AHL, int WT, int M, int NSB, int CW>
int launch_pf_gemm_cw(PfGemm h, int n_wg, hipStream_t s) {
    typedef GmGeo<AHL, WT, M, NSB, CW> G;
    if (!pf_gemm_plan<G>(h, CW)) return (int)hipErrorInvalidValue;
    hipError_t e = hipFuncSetAttribute((const void*)k_pf_gemm<AHL, WT, M, NSB, CW>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((k_pf_gemm<AHL, WT, M, NSB, CW>), dim3(n_wg * (8 / CW)), dim3(64 * CW), G::LDS, s, h);
    return (int)hipGetLastError();
}
template <int AHL, int WT, int M, int NSB = 1>
int launch_pf_gemm(const PfGemm& g, int n_wg, hipStream_t s) {
    if (gm_waves(AHL == 1, g.ncol) == 4) return launch_pf_gemm_cw<AHL, WT, M, NSB, 4>(g, n_wg, s);
    return launch_pf_gemm_cw<AHL, WT, M, NSB, 8>(g, n_wg, s);
}

template <int AHL, int WT, int M, int NSB, int SWT, int CW>
int launch_pf_gemm2_cw(PfGemm h, PfGemm hs, int n_wg, hipStream_t s) {
    typedef GmGeo<AHL, WT, M, NSB, CW> GR;
    typedef GmGeo<AHL, SWT, M, 1, CW> GS;
    if (!pf_gemm_plan<GR>(h, CW) || !pf_gemm_plan<GS>(hs, CW)) return (int)hipErrorInvalidValue;
    constexpr int lds = GR::LDS > GS::LDS ? GR::LDS : GS::LDS;
    hipError_t e = hipFuncSetAttribute((const void*)k_pf_gemm2<AHL, WT, M, NSB, SWT, CW>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((k_pf_gemm2<AHL, WT, M, NSB, SWT, CW>), dim3(n_wg * (8 / CW)), dim3(64 * CW), lds, s, h, hs);
    return (int)hipGetLastError();
}
template <int AHL, int WT, int M, int NSB, int SWT>
int launch_pf_gemm2(const PfGemm& r, const PfGemm& sh, int n_wg, hipStream_t s) {
    if (gm_waves(AHL == 1, r.ncol) == 4 && gm_waves(AHL == 1, sh.ncol) == 4)
        return launch_pf_gemm2_cw<AHL, WT, M, NSB, SWT, 4>(r, sh, n_wg, s);
    return launch_pf_gemm2_cw<AHL, WT, M, NSB, SWT, 8>(r, sh, n_wg, s);
}

// The K-quant instances (wm_prefill_kq.hip): gate/up and down of Q2_K ..
// Q6_K, for passes of m = 16 or 32 pairs.  Returns hipErrorInvalidValue for
// another combination.
int launch_pf_gemm_kq(int m, bool gateup, int wt, const PfGemm& g, int n_wg, hipStream_t s);
// Routed K-quant passes and the shared expert's Q8_0 ones in one launch
// (gate/up, or passes of 16: down of 32 has no registers left for both).
int launch_pf_gemm_kq_q8(int m, bool gateup, int wt, const PfGemm& g, const PfGemm& sh, int n_wg, hipStream_t s);

}  // namespace wm
