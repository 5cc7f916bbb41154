// prefill.hip -- prefill GEMM: Y[T][N] = X[T][K] . W[N][K]^T, W in the mx layout,
// dequantized into LDS tiles that feed the 16x16x32 MFMA, fp32 accumulate.
//
// The reference prefill dequantizes one 64x64 tile of a band into a bf16 A
// operand in core memory, then runs mlir-aie's bf16 matmul on it
// (open_kernels/designs/gemm_q4_prefill/gemm_q4_dequant.h:315-376,
// gemm_q4_prefill.py:198-203). Rounding each weight once to bf16 costs a
// maxrel of ~1.8e-3 against the fp64 reference (gemm_q4_dequant.h:283-286),
// over the 1e-3 bar. Two precisions are built from one kernel:
//   PREC 0 (default): fp16 MFMA (CDNA4's dense fp16 and bf16 MFMA peaks are
//     equal) on power-of-two-scaled operands, so fp16's narrow exponent range
//     costs nothing: token row t is scaled by 2^-s_t so its max |x| lands in
//     [2^14, 2^15) (bf16 -> fp16 is then exact: 8 significant bits, no
//     overflow, no subnormal short of 2^-10 of the row max), and weight row n
//     by 2^-e_n so its bound max_kb (15 |d| + |m|) >= max |w| lands there too:
//     w16 = RNE_f16(q (d 2^-e) + m 2^-e) (one v_pk_fma_f16 per pair, 11-bit
//     significand; d 2^-e and m 2^-e are exact in fp16 for every block within
//     2^-24 of the row's bound). The output is ldexp(acc, s_t + e_n), exact.
//     The token exponents come from the activation pre-pass. The weight rows'
//     exponents and their scale words, scaled and in fp16, form the "prefill
//     scales" of a matrix (q4_prefill_scales): a side plane laid out as the mx
//     tiles' scale blocks (256 B per tile) from which the GEMM reads its scale
//     words. Weights are static, so a caller computes them once per matrix
//     (q4_gemm_prefill_scaled); q4_gemm_prefill computes them per call.
//   PREC 1: the reference tile RNE_bf16(fl32(q*d + m)) with bf16 X, bf16 MFMA.
// The exact-code alternative (4-bit codes on the MFMA, d and m applied per
// 32-K block in fp32, as the decode kernel does) needs two VALU FMAs per
// output per block, i.e. twice the MFMA time of the same block at
// 512 MAC/clk vs 16 FMA/clk per SIMD, so it cannot reach the MFMA roofline.
//
// Tiling: a workgroup computes 256 weight rows x 256 tokens, or 128 x 128, in 8 waves (two per
// SIMD). Per LDS stage the waves turn eight mx tiles (64 rows x 32 K each) into 16-bit weights
// in LDS and copy the activations to LDS; the loads and the dequant of later stages overlap
// the MFMAs of stage s, with one barrier per stage, and one wave's dequant and LDS traffic
// hide behind the other's MFMAs.
#include <stdlib.h>

#include "norm_core.h"
#include "q4mi_device.h"
#include "q4mi_internal.h"

using namespace q4mi;

namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kMagic1024 = 0x64006400u;   // fp16 1024.0 in both halves


__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// One codes dword + its row's scale word -> eight 16-bit weights (as u32x4),
// element e = k offset e of the dword's k-group. The scale word is (d << 16 | m):
// PREC 0 reads it from the fp16 side plane (d and m already scaled by the row's
// 2^-e), PREC 1 from the mx tile (bf16).
template <int PREC>
__device__ __forceinline__ u32x4 dequant8(uint32_t w, uint32_t s, uint32_t nib2, uint32_t magic) {
    u32x4 out;
    if constexpr (PREC == 0) {
        const f16x2 sv = __builtin_bit_cast(f16x2, s);                  // [0] m, [1] d
        const f16x2 d2 = __builtin_shufflevector(sv, sv, 1, 1), m2 = __builtin_shufflevector(sv, sv, 0, 0);
        const f16x2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint32_t v = ((w >> (4 * p)) & nib2) | magic;           // 1024 + q, exact
            const f16x2 q = __builtin_bit_cast(f16x2, v) - k1024;         // q, exact
            out[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, d2, m2));
        }
    } else {
        const float d = bf16_hi_to_f32(s), m = bf16_lo_to_f32(s);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float lo = __builtin_fmaf((float)((w >> (4 * p)) & 0xF), d, m);
            const float hi = __builtin_fmaf((float)((w >> (16 + 4 * p)) & 0xF), d, m);
            const bf16x2 b = {(__bf16)lo, (__bf16)hi};
            out[p] = __builtin_bit_cast(uint32_t, b);
        }
    }
    return out;
}

// Store a wave's FN x FT fragments of 16 x 16 (rows from wn0, tokens from wt0): the lane
// holds D[n = 4 kg + r][t = i16] of each, 4 consecutive rows of one token, scaled back by
// 2^(s_t + e_n) when the operands were scaled (texp / wexp not null), exactly; accum adds
// the result to what y holds (the second pass of f32 activations). tmap: token t's exponent
// is texp[tmap[t]] (activations gathered from another row order), else texp[t].
// Token fragment j starts TS j tokens after wt0.
template <int FN, int FT, int TS, bool SCALED>
__device__ __forceinline__ void store_tile(const f32x4 (&acc)[FN][FT], float* __restrict__ y,
                                           const int* __restrict__ texp, const int* __restrict__ wexp, int T, int N,
                                           int wt0, int wn0, int accum, const int* __restrict__ tmap = nullptr) {
    const int lane = threadIdx.x & 63, i16 = lane & 15, kg = lane >> 4;
#pragma unroll
    for (int j = 0; j < FT; ++j) {
        const int t = wt0 + j * TS + i16;
        if (t >= T) continue;
        const int st = SCALED ? texp[tmap ? max(tmap[t], 0) : t] : 0;
#pragma unroll
        for (int i = 0; i < FN; ++i) {
            const int n = wn0 + i * 16 + kg * 4;
            if (n < N) {
                f32x4 v = acc[i][j];
                if constexpr (SCALED) {
                    const int4 e = *(const int4*)(wexp + n);
                    v[0] = ldexpf(v[0], st + e.x);
                    v[1] = ldexpf(v[1], st + e.y);
                    v[2] = ldexpf(v[2], st + e.z);
                    v[3] = ldexpf(v[3], st + e.w);
                }
                if (SCALED && accum) v += *(const f32x4*)(y + (int64_t)t * N + n);   // PREC 0 only
                *(f32x4*)(y + (int64_t)t * N + n) = v;
            }
        }
    }
}

// The SwiGLU epilogue of the gate/up GEMM over an interleaved matrix (per 128-row pair p,
// 64 gate rows of F, then the same 64 rows of up: N = 2F). A wave's first FN / 2 fragments are
// gate rows (from wn0), the others the up rows 64 further on, at the same lane positions, so
// h = bf16(silu(g) * u) (q4_swiglu_prepare's arithmetic) is formed from the accumulators and
// only h [T][F] bf16 is stored: the f32 gate/up output never reaches memory. Token fragment j
// starts at wt0 + TS j.
template <int FN, int FT, int TS, bool SCALED>
__device__ __forceinline__ void store_swiglu(const f32x4 (&acc)[FN][FT], uint16_t* __restrict__ h,
                                             const int* __restrict__ texp, const int* __restrict__ wexp, int T, int N,
                                             int wt0, int wn0, const int* __restrict__ tmap = nullptr) {
    const int lane = threadIdx.x & 63, i16 = lane & 15, kg = lane >> 4;
    const int F = N >> 1, f0 = (wn0 >> 7) * 64 + (wn0 & 127);   // wn0 = 128 p + c: gate rows from 64 p + c
#pragma unroll
    for (int j = 0; j < FT; ++j) {
        const int t = wt0 + j * TS + i16;
        if (t >= T) continue;
        const int st = SCALED ? texp[tmap ? max(tmap[t], 0) : t] : 0;
#pragma unroll
        for (int i = 0; i < FN / 2; ++i) {
            const int ng = wn0 + i * 16 + kg * 4;
            f32x4 g = acc[i][j], u = acc[i + FN / 2][j];
            if constexpr (SCALED) {
                const int4 eg = *(const int4*)(wexp + ng), eu = *(const int4*)(wexp + ng + 64);
                g[0] = ldexpf(g[0], st + eg.x), g[1] = ldexpf(g[1], st + eg.y);
                g[2] = ldexpf(g[2], st + eg.z), g[3] = ldexpf(g[3], st + eg.w);
                u[0] = ldexpf(u[0], st + eu.x), u[1] = ldexpf(u[1], st + eu.y);
                u[2] = ldexpf(u[2], st + eu.z), u[3] = ldexpf(u[3], st + eu.w);
            }
            uint32_t o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float a = g[2 * e] / (1.0f + expf(-g[2 * e])) * u[2 * e];
                const float b = g[2 * e + 1] / (1.0f + expf(-g[2 * e + 1])) * u[2 * e + 1];
                o[e] = f32_to_bf16_rne(a) | (f32_to_bf16_rne(b) << 16);
            }
            *(uint2*)(h + (int64_t)t * F + f0 + i * 16 + kg * 4) = make_uint2(o[0], o[1]);
        }
    }
}

// ---------------------------------------------------------------------------
// The pipelined kernel: 256 x 256 workgroup tile,
// 8 waves (2 along N x 4 along T, 128 x 64 wave tiles), 64-K stages.
//   * weights: each wave loads one mx tile (64 rows x 32 K) per stage into
//     registers three stages ahead (three register sets) and dequantizes
//     stage s+1 into the other 16-bit weight buffer during stage s,
//     interleaved with the MFMAs of the stage's second half;
//   * activations: LDS-DMA (global_load_lds_dwordx4) into a 3-deep ring, two
//     stages ahead;
//   * one barrier per stage; every wait names the youngest loads it may
//     leave in flight (vector memory loads retire in issue order).
// The DMA is issued from inline asm: the compiler's wait insertion would
// otherwise assume the DMA may write the fragments read next and wait for it
// right away.
// LDS tiles are planar: [32-K plane][row][32 halves] (64 B rows, 16 KB per
// plane of 256 rows). The 16-byte chunk c of row r sits at chunk slot
// c ^ ((r >> 1) & 3). A fragment access is 16 consecutive rows x one chunk
// per 16 lanes; with this swizzle ds_read_b128 runs conflict-free on gfx950
// (measured 543 B/ns per CU, against 284 with slot c ^ ((r >> 2) & 3), which
// also spreads each 16-lane group over all 64 banks but conflicts between
// the groups the hardware serves together), and every fragment, store and
// DMA address is one base register plus an immediate.
// LDS map: weight buffers at 0 and 32 KB, activation ring at 64, 96, 128 KB.
constexpr int kPlaneB = 256 * 64;                // one 32-K plane of a 256-row tile: 16 KB
constexpr int kTileB = 2 * kPlaneB;              // one 64-K stage of a 256-row tile: 32 KB
constexpr int kXRing = 2 * kTileB;               // LDS offset of the activation ring

// s_waitcnt immediates (gfx9 encoding: vmcnt[3:0] + vmcnt_hi[15:14], expcnt[6:4], lgkmcnt[11:8]).
constexpr int wait_imm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8); }
constexpr int kWaitVm0 = wait_imm(0, 15);
constexpr int kWaitVm0Lgkm0 = wait_imm(0, 0);
constexpr int kWaitLgkm0 = wait_imm(63, 0);

// 16 bytes per lane from global memory (uniform base + 32-bit lane offset) into LDS at
// m0 + 16 * lane.
__device__ __forceinline__ void lds_dma16(const void* gbase, uint32_t goff, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(goff), "s"(gbase), "s"(lds_base)
                 : "memory", "m0");
}

// The same through a buffer resource: 16 bytes per lane from rsrc's base + soff + voff into
// LDS at m0 + 16 * lane. A lane whose voff is past the resource's num_records reads zeros
// (the buffer range check), with no memory access.
__device__ __forceinline__ void lds_dma16_buf(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff,
                                              uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %3\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff),
                 "s"(lds_base)
                 : "memory", "m0");
}
constexpr uint32_t kPadOffset = 0x80000000u;   // past the gather resource's range: a zero row
constexpr uint64_t kGatherBytes = kPadOffset - 1;   // the resource's range: a longer matrix is not gathered from
constexpr int kBufferWord3 = 0x00020000;       // raw buffer resource, 32-bit data format

// 16 bytes per lane into registers (uniform base + 32-bit lane offset). The compiler does not
// track this load: the caller waits for it (s_waitcnt vmcnt) and then passes the registers
// through vgpr_landed before any other use. No non-temporal hint: every weight tile is read
// by each token tile's workgroup, and kept in the caches it costs less (measured at T = 2048,
// gate/up 224 -> 216 us per call; the chip is at its power limit here, so bytes fetched from
// HBM rather than the MALL show up as time).
__device__ __forceinline__ void load16_async(u32x4& dst, const void* gbase, uint32_t goff) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(dst) : "v"(goff), "s"(gbase) : "memory");
}

// Workgroup b of a launch runs on XCD b % 8. xcd_group maps the b-th of `count` workgroups
// to the tile index that gives each XCD a contiguous run of tiles (count % 8 == 0; else the
// identity): with the token tile fastest in tile order, an XCD's CUs then work on a few row
// tiles across all token tiles, so a weight tile is fetched once per XCD and shared in its
// L2, instead of once per token tile across all XCDs (T = 2048 gate/up: 216 -> 209 us).
__device__ __forceinline__ int xcd_group(int b, int count) {
    return count % 8 ? b : (b % 8) * (count / 8) + b / 8;
}
__device__ __forceinline__ void vgpr_landed(u32x4& v) { asm volatile("" : "+v"(v)); }

// One output tile of the pipelined kernel: 32 * FN weight rows from n0 x 64 * FT tokens from
// t0, K split `split` of `splits` (split s covers stages [st0, st0 + NST) of K / (32 KBS) and
// writes its partial sums to y + s * T * N; the host sums the splits in order).
// KBS: 32-K blocks per stage. A stage always holds eight mx tiles, one per wave, so the row
// tile narrows as the stage deepens: KBS = 2: 256 rows x 64 K, KBS = 4: 128 rows x 128 K.
// Waves are 2 along N x 4 along T. A wave's weight rows are [16 FN wn, +16 FN), its tokens FT
// groups of 16: a tile with few valid tokens (the ragged last tile of T, an expert's tokens) runs
// an instance with a smaller FT in which every wave does the same, smaller share of the MFMAs,
// fragment reads and DMA. Its groups are wt, wt + 4, ... there, which spreads the valid tokens
// and their stores over the waves; a full tile's lie together, FT wt, FT wt + 1, ... (64
// apart, the stores of 512 tokens on 4096 x 14336 made the call 1.09 times as long).
// KBS = 2, FN = 8: 256 rows. FN = 6: 192 rows, with the 256-row tile's loads, DMA and dequant
// unchanged: the waves of row group 3 load row group 2's mx tile again and store it to LDS
// rows 192..255, which no fragment reads, so every wave issues the same loads and the wait
// counts below hold for both.
// Invariant: every wave issues the same loads, DMA, dequant, waits and barriers in every
// stage. Wave w's loads and dequant fill row group w % (8 / KBS), K block w / (8 / KBS) of the
// shared weight buffer for all waves; its DMAs copy XD 1 KB units (16 token rows x 32 K) of
// the stage; its wait counts cover only its own loads. Only a wave's fragment reads and MFMAs
// are private (its accumulators reach memory only for its tokens below T).
// GATHER: x16 is a row-major 16-bit matrix of K columns instead of the pre-tiled image, and
// token slot t0 + s is DMA'd from its row gmap[t0 + s] (gmap null: row t0 + s itself)
// through a buffer resource over x16. A padding slot (a negative entry, or
// a slot at or past T, the tile's valid end) gets a lane offset past the resource's range, so
// its LDS row is zeros and no memory is read: its products feed only that slot's
// accumulators, which are never stored, and zero operands spare the MFMAs' power. Each lane
// fetches the 16-byte chunk that its LDS slot holds under the swizzle, so the LDS image is
// the pre-tiled one's. The token exponents (PREC 0) are then indexed by source row too:
// texp[gmap[s]].
// TAIL: K / 32 is not a multiple of KBS; the last stage's planes past K are zeros on both sides (so
// an infinity or NaN in the data meets no made-up factor): their weight words are masked (the
// loads re-read the row group's last tile) and their activations DMA'd from past a buffer
// resource's range.
// SWI: the matrix alternates 64 gate and 64 up rows. A 256-row tile's wave holds one such pair
// as fragments 0..3 and 4..7; in a 128-row tile (one pair) wave wn holds the pair's gate rows
// [32 wn, +32) as fragments 0, 1 and the same up rows as fragments 2, 3.
template <int PREC, int KBS, int FN, int FT, bool SWI = false, bool GATHER = false, bool TAIL = false>
__device__ __forceinline__ void dma_tile(uint8_t* lds, const uint8_t* __restrict__ packed,
                                         const uint16_t* __restrict__ x16, const int* __restrict__ texp,
                                         const int* __restrict__ wexp, const uint32_t* __restrict__ s16,
                                         float* __restrict__ y, int T, int N, int K, int n0, int t0, int split,
                                         int splits, int accum, const int* __restrict__ gmap = nullptr) {
    static_assert((KBS == 2 && (FN == 8 || FN == 6)) || (KBS == 4 && FN == 4), "256-, 192- or 128-row tiles");
    static_assert(FT >= 1 && FT * KBS <= 8, "a ring slot holds 32 KB of activations");
    static_assert(!SWI || FN != 6, "the SwiGLU epilogue pairs gate and up rows");
    static_assert(!TAIL || (!GATHER && FN != 6), "one DMA source, whole row tiles");
    constexpr int WN = 16 * FN, RGS = 8 / KBS, RG = FN / 2;
    constexpr int WPB = RGS * 64 * 64;               // one 32-K plane of the weight buffer
    constexpr int XPB = FT * 64 * 64;                // one 32-K plane of an activation slot
    constexpr int XD = FT * KBS / 2;                 // activation DMAs per wave and stage
    constexpr bool kFull = FT * KBS == 8;
    constexpr int TS = kFull ? 16 : 64, TW = kFull ? 16 * FT : 16;   // tokens from fragment to fragment, wave to wave
    typedef typename std::conditional<PREC == 0, f16x8, bf16x8>::type frag_t;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, wt = wave >> 1;
    const int KB = K >> 5, NSTK = TAIL ? (KB + KBS - 1) / KBS : KB / KBS;
    const int st0 = (int)((int64_t)split * NSTK / splits), NST = (int)((int64_t)(split + 1) * NSTK / splits) - st0;
    y += (int64_t)split * T * N;
    const int G = N >> 6;
    const int i16 = lane & 15, kg = lane >> 4;
    const uint32_t lane_row = i16 * 64 + ((kg ^ ((i16 >> 1) & 3)) << 4);   // row i16, chunk kg, swizzled

    // weights: this wave's mx tile of each stage (row group wave % RGS, 32-K block wave / RGS)
    const int rgl = wave % RGS, kbl = wave / RGS;
    const int rg = min(n0 / 64 + min(rgl, RG - 1), G - 1);              // clamp ragged N
    const uint8_t* const wsrc = packed + ((int64_t)rg * KB + kbl + KBS * st0) * kTileBytes;
    // scale words: PREC 0 from the fp16 side plane (256 B per tile), PREC 1 from the tile
    constexpr int SSTR = PREC == 0 ? 256 : kTileBytes;
    const uint8_t* const ssrc = PREC == 0 ? (const uint8_t*)s16 + ((int64_t)rg * KB + kbl + KBS * st0) * 256
                                          : wsrc + kCodeBytes;
    const uint32_t coff = lane * 16, soff = i16 * 16;
    const uint32_t wst = kbl * WPB + rgl * 64 * 64 + lane_row;         // + buffer + r * 1 KB

    // activations: pre-tiled as the LDS image of each stage ([256-token tile][32-K plane][256
    // rows], 16 KB per plane, zero-padded to whole 64-token groups); this wave copies the units
    // XD wave .. + XD of the stage, unit u = 16-row group u / KBS of plane u % KBS.
    const int unit0 = XD * wave / KBS;
    const uint8_t* const xsrc = (const uint8_t*)x16 +
                                (((int64_t)(t0 >> 8) * KB + KBS * st0) * kPlaneB + (t0 & 255) * 64 + unit0 * 1024);
    const uint32_t xoff = lane * 16;
    const uint32_t xdst = (uint32_t)(uintptr_t)lds + kXRing + unit0 * 1024;   // LDS byte address
    // GATHER: the byte offset of this lane's chunk in its token row of each unit (row lane / 4
    // of the group; LDS slot lane & 3 holds chunk (lane & 3) ^ ((lane >> 3) & 3))
    constexpr int GQ = FT % 2 ? 1 : KBS;             // units of a wave that share a row group
    uint32_t goff[XD / GQ];
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc((void*)x16, 0, (int)kGatherBytes,
                                                                         kBufferWord3);   // GATHER only
    if constexpr (GATHER) {
        const uint32_t chunk = (uint32_t)((lane & 3) ^ ((lane >> 3) & 3)) * 16;
#pragma unroll
        for (int q = 0; q < XD / GQ; ++q) {
            const int slot = t0 + (XD * wave + q * GQ) / KBS * 16 + (lane >> 2);
            const int r = slot >= T ? -1 : gmap ? gmap[slot] : slot;
            goff[q] = r < 0 ? kPadOffset : (uint32_t)r * (uint32_t)(2 * K) + chunk;
        }
    }

    // fragment bases: A = weight rows, B = token rows TW wt + TS j + i16
    constexpr bool kPair = SWI && KBS == 4;
    const uint32_t abase = (kPair ? wn * 32 : wn * WN) * 64 + lane_row;
    const uint32_t bbase = kXRing + wt * TW * 64 + lane_row;
    const uint32_t bbase2 = bbase + 2 * kTileB;                         // ring slot 2 (offset > 64 KB)
    const uint32_t nib2 = vgpr_const(kNib2);
    const uint32_t magic = vgpr_const(PREC == 0 ? kMagic1024 : kMagic128);

    f32x4 acc[FN][FT];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 wc[3], ws[3];                          // three register sets of weight codes + scales
    auto issue_x = [&](int st, int slot) {
#pragma unroll
        for (int q = 0; q < XD; ++q) {
            // the wave's unit q, from the first row group that the wave's units touch
            const int plane = XD % KBS ? (XD * wave + q) % KBS : q % KBS;
            const int unit = XD % KBS ? (XD * wave + q) / KBS - XD * wave / KBS : q / KBS;
            const uint32_t dst = xdst + slot * kTileB + plane * XPB + unit * 1024;
            if constexpr (GATHER)
                lds_dma16_buf(xrs, goff[q / GQ], (uint32_t)(KBS * (st0 + st) + plane) * 64, dst);
            else if constexpr (TAIL)
                lds_dma16_buf(__builtin_amdgcn_make_buffer_rsrc((void*)(xsrc + (int64_t)KBS * st * kPlaneB), 0,
                                                                (int)kGatherBytes, kBufferWord3),
                              KBS * (st0 + st) + plane < KB ? xoff : kPadOffset, plane * kPlaneB + unit * 1024, dst);
            else
                lds_dma16(xsrc + (int64_t)st * (KBS * kPlaneB) + (plane * kPlaneB + unit * 1024), xoff, dst);
        }
    };
    auto issue_w = [&](int st, u32x4& c, u32x4& sc) {
        if constexpr (TAIL) {                        // tiles past the row group's last: that one again
            const int back = max(KBS * (st0 + st) + kbl - (KB - 1), 0);
            load16_async(c, wsrc + (int64_t)(KBS * st - back) * kTileBytes, coff);
            load16_async(sc, ssrc + (int64_t)(KBS * st - back) * SSTR, soff);
            return;
        }
        load16_async(c, wsrc + st * (KBS * kTileBytes), coff);         // uniform bases
        load16_async(sc, ssrc + st * (KBS * SSTR), soff);
    };
    auto store_w = [&](int st, int buf, const u32x4& c, const u32x4& sc, int r0, int r1) {
        const uint32_t in = !TAIL || KBS * (st0 + st) + kbl < KB ? ~0u : 0u;       // uniform
#pragma unroll
        for (int r = r0; r < r1; ++r)
            *(u32x4*)(lds + wst + buf * kTileB + r * 1024) =
                TAIL ? dequant8<PREC>(c[r] & in, sc[r] & in, nib2, magic) : dequant8<PREC>(c[r], sc[r], nib2, magic);
    };
    auto read_frags = [&](int buf, int slot, int kk, frag_t (&a)[FN], frag_t (&b)[FT]) {
        const uint8_t* xp = lds + (slot == 2 ? bbase2 : bbase + slot * kTileB) + kk * XPB;
        const uint8_t* wp = lds + abase + buf * kTileB + kk * WPB;
#pragma unroll
        for (int j = 0; j < FT; ++j) b[j] = *(const frag_t*)(xp + j * TS * 64);
#pragma unroll
        for (int i = 0; i < FN; ++i) a[i] = *(const frag_t*)(wp + (kPair ? (i >> 1) * 4096 + (i & 1) * 1024 : i * 1024));
    };
    auto mfmas = [&](const frag_t (&a)[FN], const frag_t (&b)[FT]) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FT; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
    };

    // Issue order: stage s's weights two stages before its activations (W(s+3) and X(s+2) at
    // the start of stage s), so the in-order vmcnt lets each wait name the youngest loads it
    // may leave in flight (2 per W, XD per X). Prologue: W(0), W(1), X(0), W(2), X(1).
    issue_w(0, wc[0], ws[0]);
    if (NST > 1) issue_w(1, wc[1], ws[1]);
    issue_x(0, 0);
    if (NST > 2) issue_w(2, wc[2], ws[2]);
    if (NST > 1) issue_x(1, 1);
    if (NST > 2) __builtin_amdgcn_s_waitcnt(wait_imm(2 + XD, 15));   // W(0), W(1), X(0) landed
    else __builtin_amdgcn_s_waitcnt(kWaitVm0);
    vgpr_landed(wc[0]);
    vgpr_landed(ws[0]);
    store_w(0, 0, wc[0], ws[0], 0, 4);
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    asm volatile("s_barrier" ::: "memory");

    // Stage st, phase P = st % 6: weights in buffer P & 1, activations in ring slot P % 3.
    // Start: wait for W(st+1) (issued at the start of stage st-2); W(st+3) -> register set
    // P % 3 (W(st)'s, dequantized in stage st-1); X(st+2) -> slot (P+2) % 3 (X(st-1)'s,
    // released by the barrier that ended stage st-1). The dequantization of W(st+1) into the
    // other weight buffer is spread over the stage's K blocks: an MFMA hides about two
    // independent VALU instructions, not more. End: wait for X(st+1) and the LDS stores,
    // barrier.
    constexpr int DW = 4 / KBS;                           // codes dwords dequantized per K block
    constexpr int NM = FN * FT;                           // MFMAs per K block
    constexpr int VG = NM >= 22 ? 20 : NM - DW;           // MFMAs with VALU work behind them
    constexpr int VN = NM >= 22 ? 2 : (20 * DW + VG - 1) / VG;
    auto stage = [&](auto phase, int st) {
        constexpr int P = decltype(phase)::value;
        constexpr int cur = P & 1, slot = P % 3, nslot = (P + 2) % 3, wset = P % 3, nset = (P + 1) % 3;
        const bool w3 = st + 3 < NST, x2 = st + 2 < NST;
        if (x2) __builtin_amdgcn_s_waitcnt(wait_imm(2 + 2 * XD, 15));   // W(st+1) landed
        else __builtin_amdgcn_s_waitcnt(kWaitVm0);
        vgpr_landed(wc[nset]);
        vgpr_landed(ws[nset]);
        if (w3) issue_w(st + 3, wc[wset], ws[wset]);
        if (x2) issue_x(st + 2, nslot);
#pragma unroll
        for (int kk = 0; kk < KBS; ++kk) {
            frag_t a[FN], b[FT];
            read_frags(cur, slot, kk, a, b);
            store_w(st + 1, cur ^ 1, wc[nset], ws[nset], DW * kk, DW * kk + DW);
            mfmas(a, b);
            __builtin_amdgcn_sched_group_barrier(0x100, FN + FT, 0);
#pragma unroll
            for (int g = 0; g < VG; ++g) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VN, 0);
            }
#pragma unroll
            for (int g = 0; g < DW; ++g) {
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
            }
            if constexpr (NM > VG + DW) __builtin_amdgcn_sched_group_barrier(0x008, NM - VG - DW, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (w3) __builtin_amdgcn_s_waitcnt(wait_imm(2 + XD, 0));        // X(st+1) landed, LDS stores done
        else if (x2) __builtin_amdgcn_s_waitcnt(wait_imm(XD, 0));
        else __builtin_amdgcn_s_waitcnt(kWaitVm0Lgkm0);
        asm volatile("s_barrier" ::: "memory");
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    using I5 = std::integral_constant<int, 5>;
    int st = 0;
    for (; st + 6 <= NST; st += 6) {
        stage(I0{}, st);
        stage(I1{}, st + 1);
        stage(I2{}, st + 2);
        stage(I3{}, st + 3);
        stage(I4{}, st + 4);
        stage(I5{}, st + 5);
    }
    if (st < NST) stage(I0{}, st);
    if (st + 1 < NST) stage(I1{}, st + 1);
    if (st + 2 < NST) stage(I2{}, st + 2);
    if (st + 3 < NST) stage(I3{}, st + 3);
    if (st + 4 < NST) stage(I4{}, st + 4);

    // gathered activations carry their exponents by source row
    const int* tmap = GATHER ? gmap : nullptr;
    if constexpr (SWI)
        store_swiglu<FN, FT, TS, PREC == 0>(acc, (uint16_t*)y, texp, wexp, T, N, t0 + wt * TW,
                                        n0 + (kPair ? wn * 32 : wn * WN), tmap);
    else
        store_tile<FN, FT, TS, PREC == 0>(acc, y, texp, wexp, T, N, t0 + wt * TW, n0 + wn * WN, accum, tmap);
}

// dma_tile with the smallest token tile that covers the valid tokens [t0, T) of a tile of
// 64 * FTMAX (workgroup-uniform). A 256-row stage takes 0.66, 0.88, 1.05 and 1.28 us with 1 to 4
// groups of 64 tokens (tile_us): the dequantization and the LDS traffic of the weights remain.
template <int PREC, int KBS, int FN, int FTMAX, bool SWI = false, bool GATHER = false, bool TAIL = false, class... A>
__device__ __forceinline__ void dma_tile_valid(uint8_t* lds, const uint8_t* packed, const uint16_t* x16,
                                               const int* texp, const int* wexp, const uint32_t* s16, float* y, int T,
                                               int N, int K, int n0, int t0, A... rest) {
    const int groups = (T - t0 + 63) >> 6;
    if (groups >= FTMAX)
        dma_tile<PREC, KBS, FN, FTMAX, SWI, GATHER, TAIL>(lds, packed, x16, texp, wexp, s16, y, T, N, K, n0, t0,
                                                          rest...);
    else if constexpr (FTMAX > 1)
        dma_tile_valid<PREC, KBS, FN, FTMAX - 1, SWI, GATHER, TAIL>(lds, packed, x16, texp, wexp, s16, y, T, N, K, n0,
                                                                    t0, rest...);
}

// Workgroups [0, wide_wgs) take the 256-row tiles of rows [0, narrow_row0), the rest the
// 192-row tiles from narrow_row0 on (token tile fastest, then K split innermost). The longer
// tiles come first in dispatch order, so the shorter ones fill the CUs the last round of
// long tiles leaves idle. MIXED = false: 256-row tiles only (wide_wgs = the grid), an
// instance without the 192-row body.
template <int PREC, bool MIXED>
__global__ __launch_bounds__(512) void prefill_dma_kernel(const uint8_t* __restrict__ packed,
                                                          const uint16_t* __restrict__ x16,
                                                          const int* __restrict__ texp, const int* __restrict__ wexp,
                                                          const uint32_t* __restrict__ s16, float* __restrict__ y,
                                                          int T, int N, int K, int tiles_t, int splits, int wide_wgs,
                                                          int narrow_row0, int accum) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int G = (int)gridDim.x, wide = MIXED ? wide_wgs : G;
    const int b = (int)blockIdx.x < wide ? xcd_group((int)blockIdx.x, wide)
                                         : wide + xcd_group((int)blockIdx.x - wide, G - wide);
    if (!MIXED || b < wide_wgs) {
        const int tile = b / splits;
        dma_tile<PREC, 2, 8, 4>(lds, packed, x16, texp, wexp, s16, y, T, N, K, (tile / tiles_t) * 256,
                                (tile % tiles_t) * 256, b % splits, splits, accum);
    } else {
        const int i = b - wide_wgs, tile = i / splits;
        dma_tile<PREC, 2, 6, 4>(lds, packed, x16, texp, wexp, s16, y, T, N, K, narrow_row0 + (tile / tiles_t) * 192,
                                (tile % tiles_t) * 256, i % splits, splits, accum);
    }
}

// prefill_dma_kernel for a last token tile of at most 192 tokens: each tile runs the instance
// for its valid 64-token groups.
template <int PREC, bool MIXED>
__global__ __launch_bounds__(512) void prefill_ragged_kernel(const uint8_t* __restrict__ packed,
                                                             const uint16_t* __restrict__ x16,
                                                             const int* __restrict__ texp,
                                                             const int* __restrict__ wexp,
                                                             const uint32_t* __restrict__ s16, float* __restrict__ y,
                                                             int T, int N, int K, int tiles_t, int splits,
                                                             int wide_wgs, int narrow_row0, int accum) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int G = (int)gridDim.x, wide = MIXED ? wide_wgs : G;
    const int b = (int)blockIdx.x < wide ? xcd_group((int)blockIdx.x, wide)
                                         : wide + xcd_group((int)blockIdx.x - wide, G - wide);
    if (!MIXED || b < wide_wgs) {
        const int tile = b / splits;
        dma_tile_valid<PREC, 2, 8, 4>(lds, packed, x16, texp, wexp, s16, y, T, N, K, (tile / tiles_t) * 256,
                                      (tile % tiles_t) * 256, b % splits, splits, accum);
    } else {
        const int i = b - wide_wgs, tile = i / splits;
        dma_tile_valid<PREC, 2, 6, 4>(lds, packed, x16, texp, wexp, s16, y, T, N, K,
                                      narrow_row0 + (tile / tiles_t) * 192, (tile % tiles_t) * 256, i % splits, splits,
                                      accum);
    }
}

// The same GEMM in 128 x 128 tiles of 128-K stages (K % 128 == 0): four times the tiles of the
// 256 x 256 form, so short prompts and small matrices fill the CUs with fewer K splits, and a
// workgroup's epilogue stores a quarter of the bytes. What bounds a call here is the start-up,
// the tile stores and the split planes, not the MFMAs. GEMM + reduce at 4096 x 4096, each
// form at its best split (graph replays): T = 64 18.9 -> 15.4 us, 128 25.3 -> 21.4, 256 33.4 ->
// 22.5, 512 40.0 -> 31.3; at 14336 x 4096 T = 512 the 256-row form wins (74.9 against 82.2).
template <int PREC>
__global__ __launch_bounds__(512) void prefill_dma128_kernel(const uint8_t* __restrict__ packed,
                                                             const uint16_t* __restrict__ x16,
                                                             const int* __restrict__ texp,
                                                             const int* __restrict__ wexp,
                                                             const uint32_t* __restrict__ s16, float* __restrict__ y,
                                                             int T, int N, int K, int tiles_t, int splits, int accum) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int b = xcd_group((int)blockIdx.x, (int)gridDim.x), tile = b / splits;
    dma_tile_valid<PREC, 4, 4, 2>(lds, packed, x16, texp, wexp, s16, y, T, N, K, (tile / tiles_t) * 128,
                                  (tile % tiles_t) * 128, b % splits, splits, accum);
}

// Either form for a K that ends inside a stage (KBS = 2: K % 64 == 32, KBS = 4: K % 128 != 0), the rest of
// the last stage zeros. An unpipelined kernel without K splits took such shapes before:
// 147 f32 tokens on 1600 x 10656 798 -> 61 us, 89 on 5376 x 2656 109 -> 22, 2048 on 8192 x 2080 106
// -> 78; and K % 128 == 64 had 256 x 256 tiles only: 260 on 4096 x 2752 38 -> 32.
template <int PREC, int KBS>
__global__ __launch_bounds__(512) void prefill_tail_kernel(const uint8_t* __restrict__ packed,
                                                           const uint16_t* __restrict__ x16,
                                                           const int* __restrict__ texp, const int* __restrict__ wexp,
                                                           const uint32_t* __restrict__ s16, float* __restrict__ y,
                                                           int T, int N, int K, int tiles_t, int splits, int accum) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int b = xcd_group((int)blockIdx.x, (int)gridDim.x), tile = b / splits;
    constexpr int R = 512 / KBS;
    dma_tile_valid<PREC, KBS, 16 / KBS, 8 / KBS, false, false, true>(lds, packed, x16, texp, wexp, s16, y, T, N, K,
                                                                     (tile / tiles_t) * R, (tile % tiles_t) * R,
                                                                     b % splits, splits, accum);
}

// The gate/up GEMM with the SwiGLU epilogue: workgroup b takes the 256-row tile of pair rows
// (b / tiles_t) * 256 and token tile b % tiles_t over all of K (no split), writing h.
template <int PREC>
__global__ __launch_bounds__(512) void prefill_swiglu_kernel(const uint8_t* __restrict__ packed,
                                                             const uint16_t* __restrict__ x16,
                                                             const int* __restrict__ texp,
                                                             const int* __restrict__ wexp,
                                                             const uint32_t* __restrict__ s16,
                                                             uint16_t* __restrict__ h, int T, int N, int K,
                                                             int tiles_t) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int b = xcd_group((int)blockIdx.x, (int)gridDim.x);
    dma_tile<PREC, 2, 8, 4, true>(lds, packed, x16, texp, wexp, s16, (float*)h, T, N, K, (b / tiles_t) * 256,
                                  (b % tiles_t) * 256, 0, 1, 0);
}

// The same for a last token tile of at most 192 tokens (KBS = 2), or in 128 x 128 tiles (KBS = 4).
template <int PREC, int KBS>
__global__ __launch_bounds__(512) void prefill_swiglu_ragged_kernel(const uint8_t* __restrict__ packed,
                                                                    const uint16_t* __restrict__ x16,
                                                                    const int* __restrict__ texp,
                                                                    const int* __restrict__ wexp,
                                                                    const uint32_t* __restrict__ s16,
                                                                    uint16_t* __restrict__ h, int T, int N, int K,
                                                                    int tiles_t) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int b = xcd_group((int)blockIdx.x, (int)gridDim.x);
    constexpr int R = 512 / KBS;
    dma_tile_valid<PREC, KBS, 16 / KBS, 8 / KBS, true>(lds, packed, x16, texp, wexp, s16, (float*)h, T, N, K,
                                                       (b / tiles_t) * R, (b % tiles_t) * R, 0, 1, 0);
}

// Whether the last 256-token tile leaves a 64-token group or more over.
bool ragged_tokens(int T) { return T % 256 != 0 && T % 256 <= 192; }

// The exponent that puts a positive finite magnitude v in [2^14, 2^15) after scaling by
// 2^-e: v in [2^(x-1), 2^x) -> e = x - 15. 0 for zero, inf and NaN (those are passed
// through unscaled).
__device__ __forceinline__ int fp16_fit_exponent(float v) {
    if (!(v > 0.0f) || v > 3.0e38f) return 0;
    int x;
    frexpf(v, &x);
    return x - 15;
}

// Activations -> the MFMA's 16-bit type, one workgroup per token row (padded to whole
// token tiles). PREC 0: fp16, token row t scaled by 2^-s_t with s_t = fp16_fit_exponent(max
// |x_t|), and texp[t] = s_t. PREC 1: bf16 (RNE from f32), no exponents.
// TILED: the 16-byte chunk i (k = 8i..8i+7) of token t goes to its place in the LDS image
// of the pipelined kernel's activation tiles: [token tile][32-K plane][256 rows][4 chunks],
// chunk c of row r at slot c ^ ((r >> 1) & 3). Each stage of a token tile is then
// one contiguous 32 KB block, copied to LDS verbatim. Otherwise rows stay [T][K].
__device__ __forceinline__ int64_t xchunk_dst(int t, int i, int K) {
    const int r = t & 255, plane = i >> 2, c = i & 3;
    return (((int64_t)(t >> 8) * (K >> 5) + plane) * 256 + r) * 4 + (c ^ ((r >> 1) & 3));
}

// Block-wide max of a non-negative value over 256 threads (result in every thread).
__device__ __forceinline__ float block_max256(float v, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// The prefill scales of an [N, K] mx matrix, in two launches over (row group g, chunk c of
// kScaleChunk 32-K blocks) workgroups, each of 64 rows x 4 parts (thread (part, row) takes
// blocks part, part + 4, ... of the chunk):
//   max pass:   cmax[n][c] = max over the chunk's blocks of 15 |d| + |m| for row n;
//   write pass: wexp[n] = fp16_fit_exponent(max over c of cmax[n][c]) (chunk 0 stores it),
//               s16 word (g KB + kb) * 64 + (n % 16) * 4 + (n % 64) / 16 = fp16(d 2^-e) << 16 |
//               fp16(m 2^-e), the mx scale block's word order.
constexpr int kScaleChunk = 32;

__device__ __forceinline__ const uint8_t* scale_word_base(const uint8_t* packed, int64_t g, int KB, int row) {
    return packed + g * KB * kTileBytes + kCodeBytes + ((row & 15) * 4 + (row >> 4)) * 4;
}

__global__ __launch_bounds__(256) void prefill_scale_max_kernel(const uint8_t* __restrict__ packed, int K, int nchunk,
                                                                float* __restrict__ cmax) {
    __shared__ float red[4][64];
    const int64_t g = blockIdx.x / nchunk;
    const int c = blockIdx.x % nchunk, row = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int KB = K >> 5, kb0 = c * kScaleChunk, kb1 = min(kb0 + kScaleChunk, KB);
    const uint8_t* base = scale_word_base(packed, g, KB, row);
    float b = 0.f;
#pragma unroll 8
    for (int kb = kb0 + part; kb < kb1; kb += 4) {
        const uint32_t sw = load_global<uint32_t>(base + (int64_t)kb * kTileBytes);
        b = fmaxf(b, __builtin_fmaf(15.0f, fabsf(bf16_hi_to_f32(sw)), fabsf(bf16_lo_to_f32(sw))));
    }
    red[part][row] = b;
    __syncthreads();
    if (part == 0)
        cmax[(g * 64 + row) * nchunk + c] = fmaxf(fmaxf(red[0][row], red[1][row]), fmaxf(red[2][row], red[3][row]));
}

__global__ __launch_bounds__(256) void prefill_scale_write_kernel(const uint8_t* __restrict__ packed, int K,
                                                                  int nchunk, const float* __restrict__ cmax,
                                                                  int* __restrict__ wexp, uint32_t* __restrict__ s16) {
    const int64_t g = blockIdx.x / nchunk;
    const int c = blockIdx.x % nchunk, row = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int KB = K >> 5, kb0 = c * kScaleChunk, kb1 = min(kb0 + kScaleChunk, KB);
    const float* cm = cmax + (g * 64 + row) * nchunk;
    float m = 0.f;
    for (int i = 0; i < nchunk; ++i) m = fmaxf(m, cm[i]);
    const int e = fp16_fit_exponent(m);
    if (c == 0 && part == 0) wexp[g * 64 + row] = e;
    const uint8_t* base = scale_word_base(packed, g, KB, row);
    uint32_t* out = s16 + g * KB * 64 + ((row & 15) * 4 + (row >> 4));
#pragma unroll 8
    for (int kb = kb0 + part; kb < kb1; kb += 4) {
        const uint32_t sw = load_global<uint32_t>(base + (int64_t)kb * kTileBytes);
        const uint32_t dh = __builtin_bit_cast(uint16_t, (_Float16)ldexpf(bf16_hi_to_f32(sw), -e));
        const uint32_t mh = __builtin_bit_cast(uint16_t, (_Float16)ldexpf(bf16_lo_to_f32(sw), -e));
        out[(int64_t)kb * 64] = (dh << 16) | mh;
    }
}

// Eight values of a row into the MFMA's 16-bit type. PREC 0: fp16 of v 2^-s, or on the lo pass of
// an f32 source its remainder; PREC 1: bf16.
template <bool F32SRC, int PREC>
__device__ __forceinline__ u32x4 cvt8(const float (&v)[8], int s, int lo_pass) {
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t lo, hi;
        if constexpr (PREC == 0) {
            const float a = ldexpf(v[2 * e], -s), b = ldexpf(v[2 * e + 1], -s);
            _Float16 ha = (_Float16)a, hb = (_Float16)b;
            if (F32SRC && lo_pass) {
                ha = (_Float16)(a - (float)ha);
                hb = (_Float16)(b - (float)hb);
            }
            lo = __builtin_bit_cast(uint16_t, ha);
            hi = __builtin_bit_cast(uint16_t, hb);
        } else {
            lo = f32_to_bf16_rne(v[2 * e]);
            hi = f32_to_bf16_rne(v[2 * e + 1]);
        }
        o[e] = lo | (hi << 16);
    }
    return o;
}

// lo_pass (f32 activations, PREC 0): the fp16 remainder x 2^-s - fp16(x 2^-s) instead of the
// rounded value; the two passes' products add up to the f32 activations' to ~2^-22.
// One token row of prefill_xprep (all 256 threads): ld8(i, v) loads the row's 8-element
// group i as f32 (zero: a padding row, written as zeros). F32SRC: the source is f32, so the
// lo pass of PREC 0 writes the fp16 remainder. HELD: 8-element groups per thread kept in
// registers between the max and the conversion (0: ld8 is called twice, for a row in LDS).
template <bool F32SRC, int PREC, bool TILED, int HELD = 8, class Load>
__device__ __forceinline__ void xprep_row(Load ld8, bool zero, uint16_t* __restrict__ x16, int* __restrict__ texp,
                                          int t, int K, int lo_pass) {
    const int n8 = K >> 3;                       // 8-element groups of the row (K % 32 == 0)
    const int64_t row = (int64_t)t * K;
    u32x4* const out = (u32x4*)x16;
    auto dst = [&](int i) -> int64_t { return TILED ? xchunk_dst(t, i, K) : row / 8 + i; };
    if (zero) {
        for (int i = threadIdx.x; i < n8; i += 256) out[dst(i)] = u32x4{0u, 0u, 0u, 0u};
        return;
    }
    // Rows of up to 256 HELD chunks (K <= 16384 for the default) are read once and held in
    // registers for both the max and the conversion; longer rows are read twice.
    constexpr int kHeld = HELD > 0 ? HELD : 1;
    const bool held = HELD > 0 && n8 <= 256 * HELD;
    float hv[kHeld][8];
    if (held) {
#pragma unroll
        for (int c = 0; c < kHeld; ++c) {
            const int i = threadIdx.x + 256 * c;
            if (i < n8) ld8(i, hv[c]);
        }
    }
    int s = 0;
    if constexpr (PREC == 0) {
        __shared__ float red[4];
        float mx = 0.f;
        if (held) {
#pragma unroll
            for (int c = 0; c < kHeld; ++c)
                if (threadIdx.x + 256 * c < n8) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(hv[c][e]));
                }
        } else {
            for (int i = threadIdx.x; i < n8; i += 256) {
                float v[8];
                ld8(i, v);
#pragma unroll
                for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
            }
        }
        s = fp16_fit_exponent(block_max256(mx, red));
        if (threadIdx.x == 0) texp[t] = s;
    }
    if (held) {
#pragma unroll
        for (int c = 0; c < kHeld; ++c) {
            const int i = threadIdx.x + 256 * c;
            if (i < n8) out[dst(i)] = cvt8<F32SRC, PREC>(hv[c], s, lo_pass);
        }
    } else {
        for (int i = threadIdx.x; i < n8; i += 256) {
            float v[8];
            ld8(i, v);
            out[dst(i)] = cvt8<F32SRC, PREC>(v, s, lo_pass);
        }
    }
}

// The 8 activations of group i of a row, as f32.
template <bool XF32>
__device__ __forceinline__ void load_x8(const void* __restrict__ xrow, int i, float (&v)[8]) {
    if constexpr (XF32) {
        const f32x4* p = (const f32x4*)xrow + 2 * i;
        const f32x4 a = p[0], b = p[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = a[e], v[e + 4] = b[e];
    } else {
        const u32x4 w = ((const u32x4*)xrow)[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[2 * e] = bf16_lo_to_f32(w[e]), v[2 * e + 1] = bf16_hi_to_f32(w[e]);
    }
}

template <bool XF32, int PREC, bool TILED>
__global__ __launch_bounds__(256) void prefill_xprep(const void* __restrict__ x, uint16_t* __restrict__ x16,
                                                     int* __restrict__ texp, int T, int K, int lo_pass) {
    const int t = blockIdx.x;
    const void* xrow = (const uint8_t*)x + (int64_t)t * K * (XF32 ? 4 : 2);
    xprep_row<XF32, PREC, TILED>([&](int i, float (&v)[8]) { load_x8<XF32>(xrow, i, v); }, t >= T, x16, texp, t,
                                 K, lo_pass);
}

// The RMSNorm producer writing the prefill's prepared activations directly: per token row t
// (one workgroup; rows past T are the tile padding, written as zeros)
//   y  = x + add (f32, stored when y is given; y may be x: the row is read before y is written),
//   xn = bf16((y * r) * w) with r as q4_rmsnorm_add forms it (norm_core.h),
// then xn goes through prefill_xprep's conversion (bf16 source) from an LDS copy of the row.
// The same bits as q4_rmsnorm_add (bf16 xn) followed by q4_prefill_prepare(xn, bf16), with
// one launch and no bf16 row in memory. Bound by the loads of x and the planes (T = 512, K = 4096:
// 8 MB each), so a thread takes PER / 4 groups of four neighbouring values and issues all of a
// row's loads, PB planes at a time, before the first is used (16 bytes each; vec 0: some pointer
// is not 16-byte aligned, four 4-byte loads). One plane and one value at a time, each behind the
// last, took 29.4 us at five planes, this 13.3; K = 14336 with two planes 55.4 and 34.7. PER fits K, and
// PB is 1 for one plane or planes past the caches: registers and loads of values that are not
// there cost a wave more than they hide (T = 2048, K = 1024, one plane: 9.6 us before, 11.5 with PER =
// 16 and PB = 4 for it too, 7.3 now; K = 4096 20.2, 21.6 and 20.3). The row also goes to LDS, from which thread
// tid sums the squares of elements tid + 256 j, j ascending, as rmsnorm_add_kernel does (values
// past K are zeros there and are skipped here: the fp64 sum is the same).
template <int PER, int PREC, int PB>
__global__ __launch_bounds__(256) void rmsnorm_prepare_kernel(const float* x, const float* __restrict__ add,
                                                              int add_planes, const void* __restrict__ w, int w_bf16,
                                                              int vec, float* y, uint16_t* __restrict__ x16,
                                                              int* __restrict__ texp, int T, int K, float eps) {
    constexpr int C = PER / 4;
    __shared__ double part[4];
    __shared__ __attribute__((aligned(16))) float row[256 * PER];   // f32 x, then the bf16 xn
    uint16_t* const xs = (uint16_t*)row;
    const int t = blockIdx.x, tid = threadIdx.x;
    if (t < T) {
        auto ld4 = [&](const float* p) -> f32x4 {
            if (vec) return load_global<f32x4>(p);
            return f32x4{load_global<float>(p), load_global<float>(p + 1), load_global<float>(p + 2),
                         load_global<float>(p + 3)};
        };
        const float* xr = x + (int64_t)t * K;
        const int64_t pstride = (int64_t)T * K;      // plane q of add at add + q T K
        f32x4 v[C], wv[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = min(4 * (tid + 256 * c), K - 4);          // loads stay in the row
            v[c] = ld4(xr + i);
            if (w_bf16) {
                const uint16_t* p = (const uint16_t*)w + i;
                u32x2 d;
                if (vec) d = load_global<u32x2>(p);
                else d = u32x2{load_global<uint16_t>(p) | ((uint32_t)load_global<uint16_t>(p + 1) << 16),
                               load_global<uint16_t>(p + 2) | ((uint32_t)load_global<uint16_t>(p + 3) << 16)};
                wv[c] = f32x4{bf16_lo_to_f32(d[0]), bf16_hi_to_f32(d[0]), bf16_lo_to_f32(d[1]), bf16_hi_to_f32(d[1])};
            } else {
                wv[c] = ld4((const float*)w + i);
            }
        }
        if (add) {                                   // the planes in prefill_reduce_kernel's order
            const float* ar = add + (int64_t)t * K;
            f32x4 s[C];
            for (int q0 = 0; q0 < add_planes; q0 += PB) {
                f32x4 a[PB][C];
#pragma unroll
                for (int u = 0; u < PB; ++u)
                    if (q0 + u < add_planes) {
#pragma unroll
                        for (int c = 0; c < C; ++c)
                            a[u][c] = ld4(ar + (int64_t)(q0 + u) * pstride + min(4 * (tid + 256 * c), K - 4));
                    }
#pragma unroll
                for (int u = 0; u < PB; ++u)
                    if (q0 + u < add_planes) {
#pragma unroll
                        for (int c = 0; c < C; ++c) s[c] = q0 + u == 0 ? a[u][c] : s[c] + a[u][c];
                    }
            }
#pragma unroll
            for (int c = 0; c < C; ++c) v[c] = v[c] + s[c];
        }
        float* yr = y ? y + (int64_t)t * K : nullptr;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = 4 * (tid + 256 * c);
            if (i < K) *(f32x4*)(row + i) = v[c];
        }
        __syncthreads();
        double ss = 0.0;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = tid + 256 * j;
            if (i < K) ss += (double)row[i] * (double)row[i];
        }
        const double ws = wave_sum_ss(ss);
        if ((tid & 63) == 0) part[tid >> 6] = ws;
        __syncthreads();                             // row free: xs takes its place
        if (yr) {                                    // y may be x: the row was read above
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int i = 4 * (tid + 256 * c);
                if (i >= K) continue;
                if (vec) {
                    *(f32x4*)(yr + i) = v[c];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) yr[i + e] = v[c][e];
                }
            }
        }
        const float r = inv_rms(part, K, eps);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = 4 * (tid + 256 * c);
            if (i < K)
                *(u32x2*)(xs + i) = u32x2{f32_to_bf16_rne(v[c][0] * r * wv[c][0]) |
                                              (f32_to_bf16_rne(v[c][1] * r * wv[c][1]) << 16),
                                          f32_to_bf16_rne(v[c][2] * r * wv[c][2]) |
                                              (f32_to_bf16_rne(v[c][3] * r * wv[c][3]) << 16)};
        }
        __syncthreads();
    }
    xprep_row<false, PREC, true, 0>(            // the row sits in LDS: read it there twice
        [&](int i, float (&o)[8]) {
            const u32x4 wd = *(const u32x4*)(xs + 8 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[2 * e] = bf16_lo_to_f32(wd[e]), o[2 * e + 1] = bf16_hi_to_f32(wd[e]);
        },
        t >= T, x16, texp, t, K, 0);
}

// The SwiGLU producer writing the down projection's prepared activations: per token row t
//   h[f] = bf16(silu(g[t][f]) * u[t][f]), silu(g) = g / (1 + exp(-g))
// (the reference's h, moe_batch.h:181-202 mb_silu_tile; the decode kernels' silu), staged
// in LDS and converted as prefill_xprep converts a bf16 row; h is also stored [T][F] when
// h_out is given. g and u are f32 rows with strides ldg / ldu (one fused gate/up output:
// u = g + F, both strides 2F). Rows past T are the tile padding (zeros).
template <int PREC>
__global__ __launch_bounds__(256) void swiglu_prepare_kernel(const float* __restrict__ g, const float* __restrict__ u,
                                                             int64_t ldg, int64_t ldu, uint16_t* __restrict__ h_out,
                                                             uint16_t* __restrict__ x16, int* __restrict__ texp,
                                                             int T, int F) {
    __shared__ __attribute__((aligned(16))) uint16_t hs[256 * 64];
    const int t = blockIdx.x, tid = threadIdx.x;
    if (t < T) {
        const float* gr = g + (int64_t)t * ldg;
        const float* ur = u + (int64_t)t * ldu;
        for (int i = 4 * tid; i < F; i += 4 * 256) {
            const f32x4 gv = *(const f32x4*)(gr + i), uv = *(const f32x4*)(ur + i);
            uint32_t o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float a = gv[2 * e] / (1.0f + expf(-gv[2 * e])) * uv[2 * e];
                const float b = gv[2 * e + 1] / (1.0f + expf(-gv[2 * e + 1])) * uv[2 * e + 1];
                o[e] = f32_to_bf16_rne(a) | (f32_to_bf16_rne(b) << 16);
            }
            *(uint2*)(hs + i) = make_uint2(o[0], o[1]);
            if (h_out) *(uint2*)(h_out + (int64_t)t * F + i) = make_uint2(o[0], o[1]);
        }
        __syncthreads();
    }
    xprep_row<false, PREC, true, 0>(
        [&](int i, float (&o)[8]) {
            const u32x4 wd = *(const u32x4*)(hs + 8 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[2 * e] = bf16_lo_to_f32(wd[e]), o[2 * e + 1] = bf16_hi_to_f32(wd[e]);
        },
        t >= T, x16, texp, t, F, 0);
}

// One GEMM launch of the plan's form: tile 256 or 128 (see PrefillPlan).
template <int PREC>
void launch_prefill(int tile, int64_t grid, hipStream_t st, const uint8_t* w, const uint16_t* x16, const int* te,
                    const int* we, const uint32_t* s16, float* y, int T, int N, int K, int tiles_t, int splits,
                    int wide_wgs, int narrow_row0, int accum) {
#define Q4MI_DMA(KERN, ...)                                                                                         \
    hipLaunchKernelGGL(KERN, dim3((unsigned)grid), dim3(512), 0, st, w, x16, te, we, s16, y, T, N, K, tiles_t, splits, \
                       ##__VA_ARGS__, accum)
    if (tile == 128) {
        if (K % 128) Q4MI_DMA((prefill_tail_kernel<PREC, 4>));
        else Q4MI_DMA((prefill_dma128_kernel<PREC>));
    } else if (K % 64) {
        Q4MI_DMA((prefill_tail_kernel<PREC, 2>));
    } else if (ragged_tokens(T)) {
        if (wide_wgs < grid) Q4MI_DMA((prefill_ragged_kernel<PREC, true>), wide_wgs, narrow_row0);
        else Q4MI_DMA((prefill_ragged_kernel<PREC, false>), wide_wgs, narrow_row0);
    } else {
        if (wide_wgs < grid) Q4MI_DMA((prefill_dma_kernel<PREC, true>), wide_wgs, narrow_row0);
        else Q4MI_DMA((prefill_dma_kernel<PREC, false>), wide_wgs, narrow_row0);
    }
#undef Q4MI_DMA
}

// y = sum of the S partials in split order (deterministic), 4 floats per thread; accum adds
// it to what y holds. S > 0: all planes' loads go out together; S = 0: `splits` of them, one
// behind the other.
template <int S>
__global__ __launch_bounds__(256) void prefill_reduce_kernel(const f32x4* __restrict__ part, f32x4* __restrict__ y,
                                                             int64_t MN4, int splits, int accum) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= MN4) return;
    f32x4 s;
    if constexpr (S > 0) {
        f32x4 t[S];
#pragma unroll
        for (int q = 0; q < S; ++q) t[q] = part[(int64_t)q * MN4 + i];
        s = t[0];
#pragma unroll
        for (int q = 1; q < S; ++q) s += t[q];
    } else {
        s = part[i];
        for (int q = 1; q < splits; ++q) s += part[(int64_t)q * MN4 + i];
    }
    y[i] = accum ? y[i] + s : s;
}

constexpr int kMaxSplits = 16;

// Whether a thread's loads of all planes go out together. Small planes wait for latency (16 of
// 25 x 4096 f32: 4.9 us one behind the other, 2.9 together; 8 of 300 x 4096, 39 MB: 7.2 and 5.9),
// planes past the caches for memory, which many open streams slow down (8 of 512 x 4096,
// 67 MB: 11.5 and 14.4; 5 of 640 x 4096, 52 MB: 10.0 and 10.1).
bool planes_together(int planes, int64_t TN) { return planes * TN * 4 <= (int64_t)48 << 20; }

template <int S = kMaxSplits>
void launch_reduce(int splits, hipStream_t st, const float* part, float* y, int64_t TN, int accum) {
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(TN / 4, 256)), dim3(256), 0, st, (const f32x4*)part,
                           (f32x4*)y, TN / 4, splits, accum);
    };
    if (!planes_together(splits, TN)) launch(prefill_reduce_kernel<0>);
    else if (splits == S) launch(prefill_reduce_kernel<S>);
    else if constexpr (S > 2) launch_reduce<S - 1>(splits, st, part, y, TN, accum);
}

// CUs of the current device (the MI355X's 256 when no device is visible, e.g. for a
// workspace query on a host without a GPU).
int device_cus() {
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
            (void)hipGetLastError();
            return 256;
        }
        return n;
    }();
    return cus;
}

// Launch plan of one prefill GEMM: its tile (256 x 256 or 128 x 128), token tiles and K splits,
// and for the 256-row form the rows covered by 256-row tiles ([0, narrow_row0), wide_wgs
// workgroups) and by 192-row tiles (the rest; K % 64 == 0). Both forms hold one workgroup per
// CU (160 KB of LDS). Three levers fit the work to the CUs: the tile (128 x 128: four times
// the tiles, so small grids need fewer K splits and their partial traffic, at 0.5 to 0.6
// of the MFMA rate), a K split (partial sums
// reduced in order afterwards) and 192-row tiles, which fill the CUs the last round of 256-row
// tiles leaves idle without any partial traffic (Llama-3-8B gate_up at T = 2048: 448 tiles of
// 256 rows run in 2 rounds of 256 CUs; 256 of 256 rows + 256 of 192 rows in 1 + 3/4).
// 192-row strips also cover N % 256 != 0 without repeating rows.
// Q4MI_PREFILL_SPLITS and Q4MI_PREFILL_NARROW (the count of 192-row strips) override (256-row
// tiles only).
struct PrefillPlan {
    int tile, tiles_t, splits, wide_wgs, narrow_row0;
    int64_t grid;
};

// Microseconds of one workgroup of the pipelined kernel while `busy` (0 to 1) of the CUs hold one:
// nst stages of a tile of `rows` rows x 64 ft tokens and the store of the tile (out_bytes per row
// and token; the CUs share the memory). Fitted, with the reduce below, to the graph replay times
// of every sensible plan of 906 calls (25 to 4096 tokens, N 512 to 28672, K 1024 to 14336; 578 in
// precision 0, 328 in precision 1, whose dequantization is slower: one plan serves both). The
// planned form is 0.7 % slower than the call's fastest (geometric mean; 5 % in the slowest
// twentieth). Stage times taken at 64 to 256 tokens on few CUs have the 128-row form a tenth
// too fast on a full chip: 148 tokens on 19712 x 2304 took 51 us where the fastest takes 34,
// 848 on 3136 x 5824 61 where it takes 54, and 2 % were lost on average.
double tile_us(int rows, int ft, int nst, double out_bytes, double busy) {
    static constexpr double s256[5] = {0, 0.66, 0.88, 1.05, 1.28};
    const double stage = rows == 128 ? (ft == 1 ? 0.56 + 0.32 * busy : 1.03 + 0.26 * busy)
                                     : s256[ft] * (rows == 192 ? 0.89 : 1.0);
    return nst * stage + 0.5 + rows * ft / 1024.0 * (out_bytes / 4.0) * (4.8 + 4.5 * busy);
}

// Finish time of n equal workgroups on C CUs: whole rounds, then the rest on fewer of them.
template <class Cost>
double rounds_us(int64_t n, int64_t C, Cost cost) {
    return (double)(n / C) * cost(1.0) + (n % C ? cost((double)(n % C) / (double)C) : 0.0);
}

// Finish time of A units of cost cw followed by B units of cost cn when each starts on the
// earliest free of C CUs (workgroups dispatch in index order, one per CU).
double makespan(int64_t A, int64_t B, int64_t C, double cw, double cn) {
    const int64_t q = A / C, r = A % C;
    const double wide_end = (double)(q + (r ? 1 : 0)) * cw;
    if (B == 0) return wide_end;
    double t[2] = {(double)q * cw, (double)(q + 1) * cw};   // C - r CUs free at t[0], r at t[1]
    const int64_t cnt[2] = {C - r, r};
    double last = 0;
    for (int64_t left = B; left > 0;) {
        const int g = (cnt[1] > 0 && t[1] < t[0]) ? 1 : 0;
        last = t[g];
        left -= cnt[g];
        t[g] += cn;
    }
    return last + cn > wide_end ? last + cn : wide_end;
}

PrefillPlan make_plan_uncached(int T, int64_t N, int64_t K) {
    PrefillPlan p;
    p.tile = 256;
    p.tiles_t = (int)ceil_div(T, 256);
    int64_t tiles = ceil_div(N, 256) * p.tiles_t;
    p.splits = 1;
    p.wide_wgs = (int)tiles;
    p.narrow_row0 = (int)N;
    static const int forced = [] {
        const char* e = getenv("Q4MI_PREFILL_SPLITS");
        return e ? atoi(e) : 0;
    }();
    static const int forced_narrow = [] {
        const char* e = getenv("Q4MI_PREFILL_NARROW");
        return e ? atoi(e) : -1;
    }();
    const int nst = (int)ceil_div(K, 64), cap = nst < kMaxSplits ? nst : kMaxSplits;
    const int64_t G = N / 64, tt = p.tiles_t;
    const int cus = device_cus();
    // 64-token groups of a token tile: a row tile's token tiles are neighbours in the grid, so a
    // ragged one lies among the full ones and a round lasts as long as a full one
    const int ft = tt > 1 ? 4 : (int)ceil_div(T, 64);
    // the split reduce: a launch and its traffic
    auto reduce_us = [&](int S) { return S > 1 ? 2.0 + (double)(S + 1) * T * N * 4 / 4.15e6 : 0.0; };
    // a forced strip count is used only where it fits: 3b <= G and 4 | G - 3b
    const int64_t fb = forced_narrow > 0 && 3 * (int64_t)forced_narrow <= G &&
                               (G - 3 * (int64_t)forced_narrow) % 4 == 0
                           ? forced_narrow
                           : forced_narrow == 0 ? 0 : -1;
    double best = 1e300;
    // b 192-row strips and a 256-row strips with 4a + 3b = G (b = 0: 256-row strips only,
    // the last one clamped when G % 4 != 0). 192-row tiles only fill the last round of
    // 256-row ones, so at most two rounds of them are considered.
    for (int64_t b = 0; 3 * b <= G && (b * tt <= 2 * cus || b == fb); ++b) {
        if (b > 0 && ((G - 3 * b) % 4 || K % 64)) continue;
        if (fb >= 0 && b != fb) continue;
        const int64_t a = b > 0 ? (G - 3 * b) / 4 : ceil_div(G, 4);
        for (int S = 1; S <= cap; ++S) {
            if (forced > 0 && S != (forced < cap ? forced : cap)) continue;
            if (b > 0 && b != fb && b * tt * S > 2 * cus) break;
            const int ns = (int)ceil_div(nst, S);
            double cost;
            if (b > 0) {
                const double busy = (a + b) * tt * S < cus ? (double)((a + b) * tt * S) / cus : 1.0;
                cost = makespan(a * tt * S, b * tt * S, cus, tile_us(256, ft, ns, 4, busy),
                                tile_us(192, ft, ns, 4, busy));
            } else {
                cost = rounds_us(a * tt * S, cus, [&](double busy) { return tile_us(256, ft, ns, 4, busy); });
            }
            // ties: fewer rows computed (a clamped last 256-row strip repeats rows)
            cost += reduce_us(S) + 1e-6 * (double)(256 * a + 192 * b);
            if (cost < best) {
                best = cost;
                p.splits = S;
                p.wide_wgs = (int)(a * tt * S);
                p.narrow_row0 = b > 0 ? (int)(256 * a) : (int)N;
                tiles = (a + b) * tt;
            }
        }
    }
    // 128 x 128 tiles, 128-K stages
    if (forced <= 0 && forced_narrow < 0) {
        const int64_t r2 = ceil_div(G, 2), t2 = ceil_div(T, 128);
        const int nst2 = (int)ceil_div(K, 128), cap2 = nst2 < kMaxSplits ? nst2 : kMaxSplits;
        const int ft2 = t2 > 1 ? 2 : (int)ceil_div(T, 64);
        for (int S = 1; S <= cap2; ++S) {
            const int ns = (int)ceil_div(nst2, S);
            const double cost = rounds_us(r2 * t2 * S, cus,
                                          [&](double busy) { return tile_us(128, ft2, ns, 4, busy); }) + reduce_us(S);
            if (cost < best) {
                best = cost;
                p.tile = 128;
                p.tiles_t = (int)t2;
                p.splits = S;
                p.wide_wgs = 0;
                p.narrow_row0 = (int)N;
                tiles = r2 * t2;
            }
        }
    }
    p.grid = tiles * p.splits;
    return p;
}

// Whether the SwiGLU gate/up GEMM (no K split; bf16 h, one value per gate and up row pair) is
// planned to finish sooner in 128 x 128 tiles than in 256 x 256 ones.
bool swiglu_tile128(int T, int64_t N, int64_t K) {
    if (K % 128) return false;
    const int cus = device_cus();
    auto finish = [&](int tile, int nst) {
        const int64_t tt = ceil_div(T, tile);
        const int ft = tt > 1 ? tile / 64 : (int)ceil_div(T, 64);
        // and the epilogue's expf and divisions, 4 us for a 256 x 256 tile: of 200 shapes in both
        // precisions the faster form in all but one, which it misses by 0.5 %
        return rounds_us(N / tile * tt, cus, [&](double busy) {
            return tile_us(tile, ft, nst, 1, busy) + tile * ft / 1024.0 * 4.0;
        });
    };
    return finish(128, (int)(K / 128)) < finish(256, (int)(K / 64));
}

// The plans of the last few shapes per host thread (the workspace query and the call that
// follows it plan the same shape).
PrefillPlan make_plan(int T, int64_t N, int64_t K) {
    struct Entry {
        int T;
        int64_t N, K;
        PrefillPlan p;
    };
    thread_local Entry cache[4] = {};
    thread_local int next = 0;
    for (const Entry& e : cache)
        if (e.T == T && e.N == N && e.K == K && T > 0) return e.p;
    const PrefillPlan p = make_plan_uncached(T, N, K);
    cache[next] = Entry{T, N, K, p};
    next = (next + 1) & 3;
    return p;
}

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// The pre-pass of a GEMM's activations into the pipelined kernel's tiled image.
void launch_xprep(bool xf32, int prec, dim3 g, hipStream_t st, const void* x, uint16_t* x16, int* te, int T, int K,
                  int lo_pass) {
    auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, g, dim3(256), 0, st, x, x16, te, T, K, lo_pass); };
    if (prec == 0) xf32 ? launch(prefill_xprep<true, 0, true>) : launch(prefill_xprep<false, 0, true>);
    else xf32 ? launch(prefill_xprep<true, 1, true>) : launch(prefill_xprep<false, 1, true>);
}

}  // namespace

// Activation rows are padded with zeros to a multiple of 256 tokens (the widest token tile).
static size_t padded_tokens(int T) { return ((size_t)T + 255) / 256 * 256; }

// The prefill scales of an [N, K] matrix: wexp int32[N], then the fp16 scale plane (4 bytes
// per row and 32-K block), then the max pass's per-chunk maxima (f32 [N][chunks]).
static int64_t scale_chunks(int64_t K) { return ceil_div(K / 32, kScaleChunk); }
static size_t scales_wexp_bytes(int64_t N) { return align256((size_t)N * 4); }
static size_t scales_plane_bytes(int64_t N, int64_t K) { return align256((size_t)N * (K / 32) * 4); }
static size_t scales_bytes(int64_t N, int64_t K) {
    return scales_wexp_bytes(N) + scales_plane_bytes(N, K) + align256((size_t)N * scale_chunks(K) * 4);
}

extern "C" size_t q4_prefill_scales_bytes(int64_t N, int64_t K) {
    if (N <= 0 || K <= 0 || N % 64 || K % 32) return 0;
    return scales_bytes(N, K);
}

extern "C" int q4_prefill_scales(const uint8_t* packed, int64_t N, int64_t K, void* scales, size_t scales_bytes_,
                                 void* stream) {
    if (N < 0 || K <= 0 || N % 64 || K % 32) return Q4MI_E_SHAPE;
    if (N > 0x7FFFFFFF || K > 0x7FFFFFFF) return Q4MI_E_RANGE;
    if (N == 0) return Q4MI_OK;
    if (!packed || !scales || misaligned16(packed) || misaligned16(scales)) return Q4MI_E_ARG;
    if (scales_bytes_ < scales_bytes(N, K)) return Q4MI_E_WORKSPACE;
    int* wexp = (int*)scales;
    uint32_t* s16 = (uint32_t*)((char*)scales + scales_wexp_bytes(N));
    float* cmax = (float*)((char*)s16 + scales_plane_bytes(N, K));
    const int nchunk = (int)scale_chunks(K);
    const dim3 grid((unsigned)((N / 64) * nchunk));
    const hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(prefill_scale_max_kernel, grid, dim3(256), 0, st, packed, (int)K, nchunk, cmax);
    if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    hipLaunchKernelGGL(prefill_scale_write_kernel, grid, dim3(256), 0, st, packed, (int)K, nchunk,
                       (const float*)cmax, wexp, s16);
    return launch_status();
}

// Workspace of the GEMM proper: activations in the kernel's 16-bit layout, the token
// exponents, and the K-split partial sums when the plan splits K.
static size_t x16_bytes(int T, int64_t K) { return align256(padded_tokens(T) * K * 2); }
static size_t xprep_bytes(int T, int64_t K) { return x16_bytes(T, K) + align256((size_t)T * 4); }
static size_t gemm_ws_bytes(int T, int64_t N, int64_t K) {
    const PrefillPlan p = make_plan(T, N, K);
    return xprep_bytes(T, K) + (p.splits > 1 ? align256((size_t)p.splits * T * N * 4) : 0);
}

extern "C" size_t q4_gemm_prefill_scaled_workspace_bytes(int T, int64_t N, int64_t K) {
    if (T <= 0 || K <= 0 || N < 0 || N % 64 || K % 32) return 0;
    return gemm_ws_bytes(T, N, K);
}

// q4_gemm_prefill's workspace also holds the matrix's prefill scales (precision 0).
extern "C" size_t q4_gemm_prefill_workspace_bytes(int T, int64_t N, int64_t K) {
    if (T <= 0 || K <= 0 || N < 0 || N % 64 || K % 32) return 0;
    return gemm_ws_bytes(T, N, K) + scales_bytes(N, K);
}

namespace {

// The GEMM with the matrix's prefill scales (precision 0) given; workspace of gemm_ws_bytes.
// One GEMM pass over activation plane x16 (exponents te): pass 0 writes y, later passes add
// their products to it (f32 activations' remainder). part: the split partials, when the plan
// splits K; the in-order reduce then writes (or adds to) y.
int gemm_pass(const uint8_t* packed, const void* scales, const uint16_t* x16, const int* te, float* y, int T,
              int64_t N, int64_t K, int precision, float* part, int pass, hipStream_t st) {
    const int* we = precision == 0 ? (const int*)scales : nullptr;
    const uint32_t* s16 = precision == 0 ? (const uint32_t*)((const char*)scales + scales_wexp_bytes(N)) : nullptr;
    const PrefillPlan plan = make_plan(T, N, K);
    float* out = plan.splits > 1 ? part : y;
    const int accum = plan.splits > 1 ? 0 : pass;
    if (precision == 0)
        launch_prefill<0>(plan.tile, plan.grid, st, packed, x16, te, we, s16, out, T, (int)N, (int)K, plan.tiles_t,
                          plan.splits, plan.wide_wgs, plan.narrow_row0, accum);
    else
        launch_prefill<1>(plan.tile, plan.grid, st, packed, x16, nullptr, nullptr, nullptr, out, T, (int)N, (int)K,
                          plan.tiles_t, plan.splits, plan.wide_wgs, plan.narrow_row0, accum);
    if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    if (plan.splits > 1) {
        launch_reduce(plan.splits, st, out, y, (int64_t)T * N, pass);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    }
    return Q4MI_OK;
}

// f32 activations in precision 0 take two passes: their fp16 rounding, then the fp16
// remainder, whose product the second pass adds to y.
int activation_passes(int x_dtype, int precision) { return x_dtype == Q4MI_F32 && precision == 0 ? 2 : 1; }

// The GEMM with the matrix's prefill scales (precision 0) given; workspace of gemm_ws_bytes:
// one activation plane, prepared and consumed pass by pass.
int prefill_impl(const uint8_t* packed, const void* scales, const void* x, int x_dtype, float* y, int T, int64_t N,
                 int64_t K, int precision, void* workspace, hipStream_t st) {
    uint16_t* x16 = (uint16_t*)workspace;
    int* te = (int*)((char*)workspace + x16_bytes(T, K));
    float* part = (float*)((char*)workspace + xprep_bytes(T, K));
    for (int pass = 0; pass < activation_passes(x_dtype, precision); ++pass) {
        // rows up to whole 64-token groups: the kernels read no others
        launch_xprep(x_dtype == Q4MI_F32, precision, dim3((unsigned)(ceil_div(T, 64) * 64)), st, x, x16, te, T,
                     (int)K, pass);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
        const int rc = gemm_pass(packed, scales, x16, te, y, T, N, K, precision, part, pass, st);
        if (rc != Q4MI_OK) return rc;
    }
    return launch_status();
}

int prefill_args(const uint8_t* packed, const void* x, int x_dtype, float* y, int T, int64_t N, int64_t K,
                 void* workspace) {
    if (x_dtype != Q4MI_F32 && x_dtype != Q4MI_BF16) return Q4MI_E_ARG;
    if (T < 0 || N < 0 || K <= 0 || N % 64 || K % 32) return Q4MI_E_SHAPE;
    if (N > 0x7FFFFFFF || K > 0x7FFFFFFF) return Q4MI_E_RANGE;
    if (T == 0 || N == 0) return 1;                              // nothing to compute
    if (!packed || !x || !y) return Q4MI_E_ARG;
    if (misaligned16(packed) || misaligned16(x) || misaligned16(y) || misaligned16(workspace)) return Q4MI_E_ARG;
    return Q4MI_OK;
}

}  // namespace

extern "C" int q4_gemm_prefill(const uint8_t* packed, const void* x, int x_dtype, float* y, int T, int64_t N,
                               int64_t K, int precision, void* workspace, size_t workspace_bytes, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    const int a = prefill_args(packed, x, x_dtype, y, T, N, K, workspace);
    if (a != Q4MI_OK) return a > 0 ? Q4MI_OK : a;
    if (!workspace || workspace_bytes < q4_gemm_prefill_workspace_bytes(T, N, K)) return Q4MI_E_WORKSPACE;
    const hipStream_t st = (hipStream_t)stream;
    void* scales = (char*)workspace + gemm_ws_bytes(T, N, K);
    if (precision == 0) {
        const int rc = q4_prefill_scales(packed, N, K, scales, scales_bytes(N, K), stream);
        if (rc != Q4MI_OK) return rc;
    }
    return prefill_impl(packed, scales, x, x_dtype, y, T, N, K, precision, workspace, st);
}

extern "C" int q4_gemm_prefill_scaled(const uint8_t* packed, const void* scales, const void* x, int x_dtype, float* y,
                                      int T, int64_t N, int64_t K, void* workspace, size_t workspace_bytes,
                                      void* stream) {
    const int a = prefill_args(packed, x, x_dtype, y, T, N, K, workspace);
    if (a != Q4MI_OK) return a > 0 ? Q4MI_OK : a;
    if (!scales || misaligned16(scales)) return Q4MI_E_ARG;
    if (!workspace || workspace_bytes < gemm_ws_bytes(T, N, K)) return Q4MI_E_WORKSPACE;
    return prefill_impl(packed, scales, x, x_dtype, y, T, N, K, 0, workspace, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// Prepared activations: the pre-pass on its own, so a producer's output is converted once
// and read by several projections (gate and up of an FFN, Q, K and V), or written in this
// layout by the producer itself. Layout: the activation planes of the GEMM's passes (two for
// f32 x in precision 0: value and remainder), each x16_bytes(T, K), then the token exponents.
// ---------------------------------------------------------------------------
namespace {
size_t prepared_bytes(int T, int64_t K, int x_dtype, int precision) {
    return (size_t)activation_passes(x_dtype, precision) * x16_bytes(T, K) + align256((size_t)T * 4);
}
}  // namespace

extern "C" size_t q4_prefill_prepared_bytes(int T, int64_t K, int x_dtype, int precision) {
    if (T <= 0 || K <= 0 || K % 32 || (x_dtype != Q4MI_F32 && x_dtype != Q4MI_BF16) || (precision != 0 && precision != 1))
        return 0;
    return prepared_bytes(T, K, x_dtype, precision);
}

extern "C" int q4_prefill_prepare(const void* x, int x_dtype, int T, int64_t K, int precision, void* prepared,
                                  size_t prepared_bytes_, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    if (x_dtype != Q4MI_F32 && x_dtype != Q4MI_BF16) return Q4MI_E_ARG;
    if (T < 0 || K <= 0 || K % 32) return Q4MI_E_SHAPE;
    if (K > 0x7FFFFFFF) return Q4MI_E_RANGE;
    if (T == 0) return Q4MI_OK;
    if (!x || !prepared || misaligned16(x) || misaligned16(prepared)) return Q4MI_E_ARG;
    if (prepared_bytes_ < prepared_bytes(T, K, x_dtype, precision)) return Q4MI_E_WORKSPACE;
    const int passes = activation_passes(x_dtype, precision);
    int* te = (int*)((char*)prepared + passes * x16_bytes(T, K));
    for (int pass = 0; pass < passes; ++pass) {
        launch_xprep(x_dtype == Q4MI_F32, precision, dim3((unsigned)padded_tokens(T)),
                     (hipStream_t)stream, x, (uint16_t*)((char*)prepared + pass * x16_bytes(T, K)), te, T, (int)K,
                     pass);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    }
    return Q4MI_OK;
}

extern "C" int q4_rmsnorm_prepare(const float* x, const float* add, int add_planes, const void* w, int w_dtype,
                                  float* y, int T, int64_t K, float eps, int precision, void* prepared,
                                  size_t prepared_bytes_, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    if (add_planes < 0 || add_planes > 64 || (add_planes > 0) != (add != nullptr)) return Q4MI_E_ARG;
    if (w_dtype != Q4MI_F32 && w_dtype != Q4MI_BF16) return Q4MI_E_ARG;
    if (T < 0 || K <= 0 || K % 32) return Q4MI_E_SHAPE;
    if (K > 256 * 64) return Q4MI_E_RANGE;
    if (!(eps >= 0.0f)) return Q4MI_E_ARG;
    if (T == 0) return Q4MI_OK;
    if (!x || !w || !prepared || misaligned16(prepared)) return Q4MI_E_ARG;
    const size_t need = prepared_bytes(T, K, Q4MI_BF16, precision);
    if (prepared_bytes_ < need) return Q4MI_E_WORKSPACE;
    // y may be x itself, but no output may overlap another argument otherwise
    auto overlaps = [](const void* a, size_t na, const void* b, size_t nb) {
        const char *ca = (const char*)a, *cb = (const char*)b;
        return a && b && ca < cb + nb && cb < ca + na;
    };
    const size_t row_bytes = (size_t)T * K * 4, add_bytes = row_bytes * (size_t)add_planes;
    if (overlaps(prepared, need, x, row_bytes) || overlaps(prepared, need, add, add_bytes) ||
        overlaps(prepared, need, y, row_bytes) ||
        overlaps(prepared, need, w, (size_t)K * (w_dtype == Q4MI_BF16 ? 2 : 4)) ||
        (y != x && overlaps(y, row_bytes, x, row_bytes)) || overlaps(y, row_bytes, add, add_bytes))
        return Q4MI_E_ARG;
    uint16_t* x16 = (uint16_t*)prepared;
    int* te = (int*)((char*)prepared + x16_bytes(T, K));
    const dim3 grid((unsigned)padded_tokens(T)), block(256);
    const hipStream_t st = (hipStream_t)stream;
    const int wb = w_dtype == Q4MI_BF16;
    const bool one = !add || add_planes == 1 || !planes_together(add_planes, (int64_t)T * K);
    const int vec = !misaligned16(x) && !misaligned16(add) && !misaligned16(w) && !misaligned16(y);
#define Q4MI_RP(PER, PR, PB)                                                                                           \
    hipLaunchKernelGGL((rmsnorm_prepare_kernel<PER, PR, PB>), grid, block, 0, st, x, add, add_planes, w, wb, vec, y, x16, \
                       te, T, (int)K, eps)
#define Q4MI_RP_P(PER, PR, PB)                                                    \
    {                                                                             \
        if (one) Q4MI_RP(PER, PR, 1);                                             \
        else Q4MI_RP(PER, PR, PB);                                                \
    }
#define Q4MI_RP_K(PR)                                       \
    do {                                                    \
        if (K <= 256 * 4) Q4MI_RP_P(4, PR, 4)               \
        else if (K <= 256 * 8) Q4MI_RP_P(8, PR, 4)          \
        else if (K <= 256 * 16) Q4MI_RP_P(16, PR, 4)        \
        else if (K <= 256 * 32) Q4MI_RP_P(32, PR, 2)        \
        else Q4MI_RP(64, PR, 1);                            \
    } while (0)
    if (precision == 0) Q4MI_RP_K(0);
    else Q4MI_RP_K(1);
#undef Q4MI_RP_K
#undef Q4MI_RP_P
#undef Q4MI_RP
    return launch_status();
}

extern "C" int q4_swiglu_prepare(const float* g, const float* u, int64_t ldg, int64_t ldu, int T, int64_t F,
                                 int precision, void* h, void* prepared, size_t prepared_bytes_, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    if (T < 0 || F <= 0 || F % 32 || ldg < F || ldu < F || ldg % 4 || ldu % 4) return Q4MI_E_SHAPE;
    if (F > 256 * 64) return Q4MI_E_RANGE;
    if (T == 0) return Q4MI_OK;
    if (!g || !u || !prepared || misaligned16(g) || misaligned16(u) || misaligned16(prepared) || misaligned16(h))
        return Q4MI_E_ARG;
    const size_t need = prepared_bytes(T, F, Q4MI_BF16, precision);
    if (prepared_bytes_ < need) return Q4MI_E_WORKSPACE;
    auto overlaps = [](const void* a, size_t na, const void* b, size_t nb) {
        const char *ca = (const char*)a, *cb = (const char*)b;
        return a && b && ca < cb + nb && cb < ca + na;
    };
    const size_t gb = ((size_t)(T - 1) * ldg + F) * 4, ub = ((size_t)(T - 1) * ldu + F) * 4, hb = (size_t)T * F * 2;
    if (overlaps(prepared, need, g, gb) || overlaps(prepared, need, u, ub) || overlaps(h, hb, g, gb) ||
        overlaps(h, hb, u, ub) || overlaps(h, hb, prepared, need))
        return Q4MI_E_ARG;
    uint16_t* x16 = (uint16_t*)prepared;
    int* te = (int*)((char*)prepared + x16_bytes(T, F));
    const dim3 grid((unsigned)padded_tokens(T)), block(256);
    const hipStream_t st = (hipStream_t)stream;
#define Q4MI_SP(PR)                                                                                               \
    hipLaunchKernelGGL((swiglu_prepare_kernel<PR>), grid, block, 0, st, g, u, ldg, ldu, (uint16_t*)h, x16, te, T, (int)F)
    if (precision == 0) Q4MI_SP(0);
    else Q4MI_SP(1);
#undef Q4MI_SP
    return launch_status();
}

extern "C" int q4_gemm_prefill_swiglu(const uint8_t* gate_up, const void* scales, const void* prepared, int x_dtype,
                                      void* h, int T, int64_t F, int64_t K, int precision, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    if (x_dtype != Q4MI_F32 && x_dtype != Q4MI_BF16) return Q4MI_E_ARG;
    if (activation_passes(x_dtype, precision) != 1) return Q4MI_E_ARG;   // f32 x in precision 0: two passes
    if (T < 0 || F <= 0 || K <= 0 || F % 128 || K % 64) return Q4MI_E_SHAPE;
    if (2 * F > 0x7FFFFFFF || K > 0x7FFFFFFF) return Q4MI_E_RANGE;
    if (T == 0) return Q4MI_OK;
    if (!gate_up || !prepared || !h || misaligned16(gate_up) || misaligned16(prepared) || misaligned16(h))
        return Q4MI_E_ARG;
    if (precision == 0 && (!scales || misaligned16(scales))) return Q4MI_E_ARG;
    const int64_t N = 2 * F;
    const int* we = precision == 0 ? (const int*)scales : nullptr;
    const uint32_t* s16 = precision == 0 ? (const uint32_t*)((const char*)scales + scales_wexp_bytes(N)) : nullptr;
    const int* te = precision == 0 ? (const int*)((const char*)prepared + x16_bytes(T, K)) : nullptr;
    const bool t128 = swiglu_tile128(T, N, K);
    const int tile = t128 ? 128 : 256, tiles_t = (int)ceil_div(T, tile);
    const dim3 grid((unsigned)((N / tile) * tiles_t)), block(512);
    const hipStream_t st = (hipStream_t)stream;
#define Q4MI_SG(KERN)                                                                                            \
    hipLaunchKernelGGL(KERN, grid, block, 0, st, gate_up, (const uint16_t*)prepared, te, we, s16, (uint16_t*)h, T, \
                       (int)N, (int)K, tiles_t)
#define Q4MI_SG_FORM(PR)                                                    \
    do {                                                                    \
        if (t128) Q4MI_SG((prefill_swiglu_ragged_kernel<PR, 4>));           \
        else if (ragged_tokens(T)) Q4MI_SG((prefill_swiglu_ragged_kernel<PR, 2>)); \
        else Q4MI_SG((prefill_swiglu_kernel<PR>));                          \
    } while (0)
    if (precision == 0) Q4MI_SG_FORM(0);
    else Q4MI_SG_FORM(1);
#undef Q4MI_SG_FORM
#undef Q4MI_SG
    return launch_status();
}

extern "C" size_t q4_gemm_prefill_prepared_workspace_bytes(int T, int64_t N, int64_t K) {
    if (T <= 0 || K <= 0 || N < 0 || N % 64 || K % 32) return 0;
    const PrefillPlan p = make_plan(T, N, K);
    return p.splits > 1 ? align256((size_t)p.splits * T * N * 4) : 0;
}

extern "C" int q4_gemm_prefill_prepared(const uint8_t* packed, const void* scales, const void* prepared, int x_dtype,
                                        float* y, int T, int64_t N, int64_t K, int precision, void* workspace,
                                        size_t workspace_bytes, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    const int a = prefill_args(packed, prepared, x_dtype, y, T, N, K, workspace);
    if (a != Q4MI_OK) return a > 0 ? Q4MI_OK : a;
    if (precision == 0 && (!scales || misaligned16(scales))) return Q4MI_E_ARG;
    const PrefillPlan plan = make_plan(T, N, K);
    if (plan.splits > 1 && (!workspace || workspace_bytes < q4_gemm_prefill_prepared_workspace_bytes(T, N, K)))
        return Q4MI_E_WORKSPACE;
    const int passes = activation_passes(x_dtype, precision);
    const int* te = (const int*)((const char*)prepared + passes * x16_bytes(T, K));
    for (int pass = 0; pass < passes; ++pass) {
        const uint16_t* x16 = (const uint16_t*)((const char*)prepared + pass * x16_bytes(T, K));
        const int rc = gemm_pass(packed, scales, x16, te, y, T, N, K, precision, (float*)workspace, pass,
                                 (hipStream_t)stream);
        if (rc != Q4MI_OK) return rc;
    }
    return Q4MI_OK;
}

extern "C" int q4_prefill_split_count(int T, int64_t N, int64_t K) {
    if (T <= 0 || N <= 0 || K <= 0 || N % 64 || K % 32) return 0;
    return make_plan(T, N, K).splits;
}

extern "C" int q4_prefill_tile_rows(int T, int64_t N, int64_t K, int swiglu) {
    if (T <= 0 || N <= 0 || K <= 0 || N % 64 || K % 32 || (swiglu && (N % 256 || K % 64))) return 0;
    if (swiglu) return swiglu_tile128(T, N, K) ? 128 : 256;
    const PrefillPlan p = make_plan(T, N, K);
    return p.tile == 256 && p.wide_wgs < p.grid ? 192 : p.tile;
}

extern "C" int q4_gemm_prefill_prepared_partials(const uint8_t* packed, const void* scales, const void* prepared,
                                                 int x_dtype, float* part, size_t part_bytes, int T, int64_t N,
                                                 int64_t K, int precision, void* stream) {
    if (precision != 0 && precision != 1) return Q4MI_E_ARG;
    if (activation_passes(x_dtype, precision) != 1) return Q4MI_E_ARG;   // f32 x in precision 0: two passes
    const int a = prefill_args(packed, prepared, x_dtype, part, T, N, K, nullptr);
    if (a != Q4MI_OK) return a > 0 ? Q4MI_OK : a;
    if (precision == 0 && (!scales || misaligned16(scales))) return Q4MI_E_ARG;
    const PrefillPlan plan = make_plan(T, N, K);
    // the planes this call writes follow this process's plan, not a count queried elsewhere
    if (part_bytes < (size_t)plan.splits * T * N * sizeof(float)) return Q4MI_E_WORKSPACE;
    const int* te = (const int*)((const char*)prepared + x16_bytes(T, K));
    const int* we = precision == 0 ? (const int*)scales : nullptr;
    const uint32_t* s16 = precision == 0 ? (const uint32_t*)((const char*)scales + scales_wexp_bytes(N)) : nullptr;
    const hipStream_t st = (hipStream_t)stream;
    // plane s of the K split at part + s T N (one plane, the whole product, when unsplit)
    if (precision == 0)
        launch_prefill<0>(plan.tile, plan.grid, st, packed, (const uint16_t*)prepared, te, we, s16, part, T, (int)N,
                          (int)K, plan.tiles_t, plan.splits, plan.wide_wgs, plan.narrow_row0, 0);
    else
        launch_prefill<1>(plan.tile, plan.grid, st, packed, (const uint16_t*)prepared, nullptr, nullptr, nullptr, part, T,
                          (int)N, (int)K, plan.tiles_t, plan.splits, plan.wide_wgs, plan.narrow_row0, 0);
    return launch_status();
}

// ---------------------------------------------------------------------------
// Routed MoE at prefill scale: out[t] = sum_j w[t][j] down_e(silu(gate_e x_t) (up_e x_t)).
//
// The reference batches an expert's tokens into slots and runs them through its expert
// GEMM dispatch by dispatch (moe_batch.h:98-172, a host loop over dispatches in
// Core::moe_block, core.cpp:5163-5178). Here the batching is on the device and the expert
// GEMMs are the pipelined prefill tiles (dma_tile) over all experts in one launch each:
//   1. route (one workgroup): tokens per expert from an LDS histogram of ids; expert e's
//      slots are [off_e, off_e + n_e), padded to whole 256-token tiles, experts in
//      ascending order; per tile its expert and the end of that expert's slots.
//   2. slots (a workgroup per expert): the pairs routed to e, in pair order, get the slots
//      off_e, off_e + 1, ...; slot -> token row (pads -1) and pair -> slot.
//   3. the token rows gathered into the slots in the GEMM's tiled 16-bit layout (pads 0);
//   4. gate/up: workgroup (tile, 256-row tile) runs dma_tile on expert e's [2F, H] matrix
//      into G[slot][2F] (f32);
//   5. h = silu(g) u from G (gate and up row groups alternate), into the 16-bit layout;
//   6. down: as 4 on the [H, F] matrices into Y[slot][H];
//   7. combine: out[t] = sum_j w[t][j] Y[slot(t, j)] in slot order j.
// Precision 0 (fp16 tiles with power-of-two scaling, the matrices' prefill scales given)
// takes f32 activations and h in two passes (fp16 value + remainder), as q4_gemm_prefill
// does; precision 1 (the reference's bf16 tile, RNE(q d + m)) rounds x and h to bf16, as
// the reference's moe_batch rounds h (moe_batch.h:181-202). A token row's result does not
// depend on its slot (MFMA rows are independent), and the combine sums in slot order, so
// results are deterministic.
// ---------------------------------------------------------------------------
namespace {

constexpr int kMoePfMaxExperts = 8192;
constexpr int64_t kMoePfMaxPairs = (int64_t)1 << 22;

__global__ __launch_bounds__(1024) void moe_route_kernel(const int32_t* __restrict__ ids, int P, int E,
                                                         int* __restrict__ cnt, int* __restrict__ off,
                                                         int* __restrict__ tile_e, int* __restrict__ tile_end,
                                                         int* __restrict__ meta) {
    __shared__ int hist[kMoePfMaxExperts];
    __shared__ int wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < E; e += 1024) hist[e] = 0;
    __syncthreads();
    constexpr int kR = 8;                           // ids per thread in flight together
    for (int p0 = 0; p0 < P; p0 += 1024 * kR) {
        int ev[kR];
#pragma unroll
        for (int j = 0; j < kR; ++j) {
            const int p = p0 + tid + 1024 * j;
            ev[j] = p < P ? ids[p] : -1;
        }
#pragma unroll
        for (int j = 0; j < kR; ++j)
            if (ev[j] >= 0 && ev[j] < E) atomicAdd(&hist[ev[j]], 1);
    }
    __syncthreads();
    const int per = (E + 1023) / 1024;               // experts per thread, consecutive
    int tiles = 0;
    for (int j = 0; j < per; ++j) {
        const int e = tid * per + j;
        if (e < E) tiles += (hist[e] + 255) >> 8;
    }
    int incl = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int tp = incl - tiles;
    for (int w = 0; w < wave; ++w) tp += wsum[w];
    for (int j = 0; j < per; ++j) {
        const int e = tid * per + j;
        if (e >= E) break;
        const int n = hist[e], nt = (n + 255) >> 8;
        cnt[e] = n;
        off[e] = tp * 256;
        for (int i = 0; i < nt; ++i) {
            tile_e[tp + i] = e;
            tile_end[tp + i] = tp * 256 + n;
        }
        tp += nt;
    }
    if (tid == 1023) meta[0] = tp;
}

// A workgroup barrier for LDS only: this wave's LDS operations are complete, its global
// stores may still be in flight (__syncthreads would also wait for those).
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    asm volatile("s_barrier" ::: "memory");
}

// Expert e's pairs, in pair order, take slots off[e], off[e] + 1, ...: slot_of_pair and the
// slot -> token row map (padding slots -1). A batch is 4096 pairs: thread t holds the 16
// consecutive ids [16 t, 16 t + 16) in registers (four 16-byte loads, issued together), so
// a block-wide prefix sum of the per-thread counts orders the matches; only the waves' sums
// go through LDS, and the slot stores are never waited for inside the loop.
__device__ __forceinline__ void moe_slots(int e, const int32_t* __restrict__ ids, int P, int topk,
                                          const int* __restrict__ cnt, const int* __restrict__ off,
                                          int* __restrict__ slot_of_pair, int* __restrict__ rowmap) {
    constexpr int kPer = 16, kBatch = 256 * kPer;
    __shared__ int wsum[2][4];
    const int n = cnt[e];
    if (n == 0) return;
    const int o = off[e];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool vec = ((uintptr_t)ids & 15) == 0;    // 16-byte loads of ids
    int base = 0;                                   // slots given out before this batch
    for (int b0 = 0, par = 0; b0 < P && base < n; b0 += kBatch, par ^= 1) {
        const int i0 = b0 + tid * kPer;
        int iv[kPer];
        if (vec && i0 + kPer <= P) {
#pragma unroll
            for (int q = 0; q < kPer / 4; ++q) {
                const int4 v = *(const int4*)(ids + i0 + 4 * q);
                iv[4 * q] = v.x, iv[4 * q + 1] = v.y, iv[4 * q + 2] = v.z, iv[4 * q + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < kPer; ++j) iv[j] = i0 + j < P ? ids[i0 + j] : -1;
        }
        int c = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) c += iv[j] == e;
        int incl = c;
#pragma unroll
        for (int sft = 1; sft < 64; sft <<= 1) {
            const int v = __shfl_up(incl, sft);
            if (lane >= sft) incl += v;
        }
        if (lane == 63) wsum[par][wave] = incl;     // two sets: no barrier needed before reuse
        lds_sync();
        int r = base + incl - c;
        for (int w = 0; w < wave; ++w) r += wsum[par][w];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            if (iv[j] == e) {
                const int p = i0 + j;
                slot_of_pair[p] = o + r;
                rowmap[o + r] = p / topk;
                ++r;
            }
        }
        base += wsum[par][0] + wsum[par][1] + wsum[par][2] + wsum[par][3];
    }
    const int pad = ((n + 255) >> 8) << 8;
    for (int i = n + tid; i < pad; i += 256) rowmap[o + i] = -1;
}

__global__ __launch_bounds__(256) void moe_slots_kernel(const int32_t* __restrict__ ids, int P, int topk,
                                                        const int* __restrict__ cnt, const int* __restrict__ off,
                                                        int* __restrict__ slot_of_pair, int* __restrict__ rowmap) {
    moe_slots(blockIdx.x, ids, P, topk, cnt, off, slot_of_pair, rowmap);
}

// The slots (workgroups below E) and the token rows' fp16 pre-pass (prefill_xprep, one workgroup
// per token behind them) in one launch: neither reads what the other writes, and the slots are a
// chain of trips to memory on E CUs. 128 experts, 2048 tokens: 9.8 + 7.6 us (and the gap between the
// launches) as two, 12.0 as one.
template <bool XF32>
__global__ __launch_bounds__(256) void moe_slots_xprep_kernel(const int32_t* __restrict__ ids, int P, int topk, int E,
                                                              const int* __restrict__ cnt, const int* __restrict__ off,
                                                              int* __restrict__ slot_of_pair,
                                                              int* __restrict__ rowmap, const void* __restrict__ x,
                                                              uint16_t* __restrict__ x16, int* __restrict__ texp,
                                                              int H) {
    if ((int)blockIdx.x < E) {
        moe_slots(blockIdx.x, ids, P, topk, cnt, off, slot_of_pair, rowmap);
        return;
    }
    const int t = (int)blockIdx.x - E;
    const void* xrow = (const uint8_t*)x + (int64_t)t * H * (XF32 ? 4 : 2);
    xprep_row<XF32, 0, false>([&](int i, float (&v)[8]) { load_x8<XF32>(xrow, i, v); }, false, x16, texp, t, H, 0);
}

// One slot row per wave (4 per workgroup) of the MoE activation preps: xprep_row's
// conversion with the row max reduced within the wave. ld8(i, v) loads 8-element group i
// of the row as f32; zero writes a padding row. Rows of up to 512 groups (K <= 4096) are
// held in registers, longer ones read twice.
template <bool F32SRC, int PREC, class Load>
__device__ __forceinline__ void xprep_row_wave(Load ld8, bool zero, uint16_t* __restrict__ x16,
                                               int* __restrict__ texp, int t, int K, int lo_pass) {
    const int n8 = K >> 3, lane = threadIdx.x & 63;
    u32x4* const out = (u32x4*)x16;
    if (zero) {
        for (int i = lane; i < n8; i += 64) out[xchunk_dst(t, i, K)] = u32x4{0u, 0u, 0u, 0u};
        return;
    }
    constexpr int kHeld = 8;
    const bool held = n8 <= 64 * kHeld;
    float hv[kHeld][8];
    if (held) {
#pragma unroll
        for (int c = 0; c < kHeld; ++c) {
            const int i = lane + 64 * c;
            if (i < n8) ld8(i, hv[c]);
        }
    }
    int s = 0;
    if constexpr (PREC == 0) {
        float mx = 0.f;
        if (held) {
#pragma unroll
            for (int c = 0; c < kHeld; ++c)
                if (lane + 64 * c < n8) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(hv[c][e]));
                }
        } else {
            for (int i = lane; i < n8; i += 64) {
                float v[8];
                ld8(i, v);
#pragma unroll
                for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        s = fp16_fit_exponent(mx);
        if (lane == 0) texp[t] = s;
    }
    if (held) {
#pragma unroll
        for (int c = 0; c < kHeld; ++c) {
            const int i = lane + 64 * c;
            if (i < n8) out[xchunk_dst(t, i, K)] = cvt8<F32SRC, PREC>(hv[c], s, lo_pass);
        }
    } else {
        for (int i = lane; i < n8; i += 64) {
            float v[8];
            ld8(i, v);
            out[xchunk_dst(t, i, K)] = cvt8<F32SRC, PREC>(v, s, lo_pass);
        }
    }
}

template <bool XF32, int PREC>
__global__ __launch_bounds__(256) void moe_xprep_kernel(const void* __restrict__ x, const int* __restrict__ rowmap,
                                                        const int* __restrict__ meta, uint16_t* __restrict__ x16,
                                                        int* __restrict__ texp, int K, int lo_pass) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= meta[0] * 256) return;
    const int row = rowmap[t];
    const void* xrow = (const uint8_t*)x + (int64_t)(row < 0 ? 0 : row) * K * (XF32 ? 4 : 2);
    xprep_row_wave<XF32, PREC>([&](int i, float (&v)[8]) { load_x8<XF32>(xrow, i, v); }, row < 0, x16, texp, t, K,
                               lo_pass);
}

// h[f] = silu(g[f]) u[f] of slot t from G[t][2F], where the 64 gate rows of row group j are
// columns 128 j .. 128 j + 63 and its up rows the next 64. HB16 (PREC 0): h rounded to bf16
// first (the reference's h, moe_batch.h:181-202), so the fp16 tile takes it in one pass.
template <int PREC, bool HB16 = false>
__global__ __launch_bounds__(256) void moe_hprep_kernel(const float* __restrict__ G, const int* __restrict__ rowmap,
                                                        const int* __restrict__ meta, uint16_t* __restrict__ x16,
                                                        int* __restrict__ texp, int F, int lo_pass) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= meta[0] * 256) return;
    const float* g = G + (int64_t)t * 2 * F;
    auto ld8 = [&](int i, float (&v)[8]) {
        const int f = 8 * i, c = (f >> 6) * 128 + (f & 63);
        const f32x4 g0 = *(const f32x4*)(g + c), g1 = *(const f32x4*)(g + c + 4);
        const f32x4 u0 = *(const f32x4*)(g + c + 64), u1 = *(const f32x4*)(g + c + 68);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = g0[e] / (1.0f + expf(-g0[e])) * u0[e];
            v[e + 4] = g1[e] / (1.0f + expf(-g1[e])) * u1[e];
        }
        if constexpr (HB16) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = bf16_hi_to_f32(f32_to_bf16_rne(v[e]) << 16);
        }
    };
    xprep_row_wave<!HB16, PREC>(ld8, rowmap[t] < 0, x16, texp, t, F, lo_pass);
}

// Bf16 h rows (from the gate/up GEMM's SwiGLU epilogue, h[S][F]) into down's 16-bit layout, pad
// slots (from the tile's valid end on) as zeros. ragged: the down GEMM takes only a tile's
// 64-slot groups that hold a valid slot, so the groups past them are left alone (128 experts,
// top-8 of 2048 tokens: half of the slots are padding). Bound by the trips to memory in front
// of a row's few bytes: the tile's end, uniform, comes through the scalar cache, and for rows
// of up to 128 kH16Held values a wave takes four neighbouring slots at once, 16 lanes each (F %
// 128 == 0: no idle lane), their loads issued together; the stores are then 256 B runs of the
// image. Longer rows: one slot per wave, xprep_row_wave. The same bytes.
// 2048 tokens, F = 768: 19.8 -> 13.3 us (17.0 with the skipped groups alone).
constexpr int kH16Held = 12;
template <int PREC, bool FOUR>
__global__ __launch_bounds__(256) void moe_h16prep_kernel(const uint16_t* __restrict__ h,
                                                          const int* __restrict__ tile_end,
                                                          const int* __restrict__ meta, uint16_t* __restrict__ x16,
                                                          int* __restrict__ texp, int F, int ragged) {
    const int t0 = blockIdx.x * (FOUR ? 16 : 4);       // a workgroup's slots share a 64-slot group
    if (t0 >= meta[0] * 256) return;
    const int end = tile_end[t0 >> 8];
    if (ragged && t0 >= ((end + 63) & ~63)) return;
    const int t = t0 + (threadIdx.x >> (FOUR ? 4 : 6));
    const uint16_t* hrow = h + (int64_t)t * F;
    if constexpr (!FOUR) {
        xprep_row_wave<false, PREC>([&](int i, float (&v)[8]) { load_x8<false>(hrow, i, v); }, t >= end, x16, texp, t,
                                    F, 0);
    } else {
        const int sub = threadIdx.x & 15, n = F >> 7;
        u32x4 raw[kH16Held];
#pragma unroll
        for (int c = 0; c < kH16Held; ++c) {
            raw[c] = u32x4{0u, 0u, 0u, 0u};
            if (c < n && t < end) raw[c] = ((const u32x4*)hrow)[sub + 16 * c];
        }
        int s = 0;
        if constexpr (PREC == 0) {
            float mx = 0.f;
#pragma unroll
            for (int c = 0; c < kH16Held; ++c)
                if (c < n) {
                    float v[8];
                    load_x8<false>(&raw[c], 0, v);
#pragma unroll
                    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
                }
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
            s = fp16_fit_exponent(mx);
            if (sub == 0 && t < end) texp[t] = s;
        }
#pragma unroll
        for (int c = 0; c < kH16Held; ++c)
            if (c < n) {
                float v[8];
                load_x8<false>(&raw[c], 0, v);
                ((u32x4*)x16)[xchunk_dst(t, sub + 16 * c, F)] = cvt8<false, PREC>(v, s, 0);
            }
    }
}

template <int PREC>
void launch_h16prep(unsigned S, hipStream_t st, const uint16_t* h, const int* tile_end, const int* meta, uint16_t* x16,
                    int* texp, int F, bool ragged) {
    if (F <= 128 * kH16Held)
        hipLaunchKernelGGL((moe_h16prep_kernel<PREC, true>), dim3(S / 16), dim3(256), 0, st, h, tile_end, meta, x16,
                           texp, F, (int)ragged);
    else
        hipLaunchKernelGGL((moe_h16prep_kernel<PREC, false>), dim3(S / 4), dim3(256), 0, st, h, tile_end, meta, x16,
                           texp, F, (int)ragged);
}

// Workgroup (token tile tt, 256-row tile rt) of a grouped expert GEMM: dma_tile on tile tt's
// expert's matrix (N rows, ebytes each expert), slots [256 tt, tile_end) valid. GATHER: x16
// is row-major ([rows][K]), slot s's row gmap[s] (gmap null: row s).
template <int PREC, bool SWI = false, bool GATHER = false>
__global__ __launch_bounds__(512) void moe_dma_kernel(const uint8_t* __restrict__ packed, int64_t ebytes,
                                                      const uint16_t* __restrict__ x16, const int* __restrict__ texp,
                                                      const int* __restrict__ wexp, const uint32_t* __restrict__ s16,
                                                      int64_t s16_words, float* __restrict__ y,
                                                      const int* __restrict__ tile_e, const int* __restrict__ tile_end,
                                                      const int* __restrict__ meta, int N, int K, int tiles_n, int accum,
                                                      const int* __restrict__ gmap) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int b = blockIdx.x, tt = b / tiles_n, rt = b % tiles_n;
    if (tt >= meta[0]) return;
    const int e = tile_e[tt];
    dma_tile<PREC, 2, 8, 4, SWI, GATHER>(lds, packed + e * ebytes, x16, texp,
                                 PREC == 0 ? wexp + (int64_t)e * N : nullptr,
                                 PREC == 0 ? s16 + e * s16_words : nullptr, y, tile_end[tt], N, K, rt * 256, tt * 256,
                                 0, 1, accum, gmap);
}

// The same with each tile's work sized by its valid 64-slot groups. An XCD takes a contiguous run of
// the tiles there are (meta[0], not the grid's bound; the last count % 8 stay where they are), so an
// expert's row tiles fetch its gathered token rows into one L2 instead of each into another's: 128
// experts, top-8 of 2048 tokens, the block 1.203 -> 1.231 times the speed of the same earlier build.
template <int PREC, bool SWI = false, bool GATHER = false>
__global__ __launch_bounds__(512) void moe_ragged_kernel(const uint8_t* __restrict__ packed, int64_t ebytes,
                                                         const uint16_t* __restrict__ x16, const int* __restrict__ texp,
                                                         const int* __restrict__ wexp, const uint32_t* __restrict__ s16,
                                                         int64_t s16_words, float* __restrict__ y,
                                                         const int* __restrict__ tile_e, const int* __restrict__ tile_end,
                                                         const int* __restrict__ meta, int N, int K, int tiles_n, int accum,
                                                         const int* __restrict__ gmap) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[5 * kTileB];
    const int count = meta[0] * tiles_n, whole = count & ~7;
    if ((int)blockIdx.x >= count) return;
    const int b = (int)blockIdx.x < whole ? xcd_group((int)blockIdx.x, whole) : (int)blockIdx.x;
    const int tt = b / tiles_n, rt = b % tiles_n;
    const int e = tile_e[tt];
    dma_tile_valid<PREC, 2, 8, 4, SWI, GATHER>(lds, packed + e * ebytes, x16, texp,
                                 PREC == 0 ? wexp + (int64_t)e * N : nullptr,
                                 PREC == 0 ? s16 + e * s16_words : nullptr, y, tile_end[tt], N, K, rt * 256, tt * 256,
                                 0, 1, accum, gmap);
}

// The grouped expert GEMM of a launch: one ragged tile per expert, so up to kMoeFullTiles tiles per
// expert on average the kernel whose tiles follow their valid slots (128 experts, top-8 of
// 2048 tokens, 128 of a tile's 256 slots valid: gate/up 191 -> 165 us, down 147 -> 118; 144 and
// 103 with the runs above, in the middle of 400 passes), beyond
// that the one-body kernel, where at most 1 / kMoeFullTiles of the tiles could gain.
constexpr int kMoeFullTiles = 16;
template <int PREC, bool SWI = false, bool GATHER = false>
void launch_moe_dma(bool ragged, unsigned grid, hipStream_t st, const uint8_t* packed, int64_t ebytes,
                    const uint16_t* x16, const int* texp, const int* wexp, const uint32_t* s16, int64_t s16_words,
                    float* y, const int* tile_e, const int* tile_end, const int* meta, int N, int K, int tiles_n,
                    int accum, const int* gmap = nullptr) {
    if (ragged)
        hipLaunchKernelGGL((moe_ragged_kernel<PREC, SWI, GATHER>), dim3(grid), dim3(512), 0, st, packed, ebytes, x16,
                           texp, wexp, s16, s16_words, y, tile_e, tile_end, meta, N, K, tiles_n, accum, gmap);
    else
        hipLaunchKernelGGL((moe_dma_kernel<PREC, SWI, GATHER>), dim3(grid), dim3(512), 0, st, packed, ebytes, x16,
                           texp, wexp, s16, s16_words, y, tile_e, tile_end, meta, N, K, tiles_n, accum, gmap);
}

// out[t][n..n+3] = sum_j w[t][j] Y[slot(t, j)][n..n+3], slot order j.
__global__ __launch_bounds__(256) void moe_prefill_combine_kernel(const float* __restrict__ Y,
                                                                  const int* __restrict__ slot_of_pair,
                                                                  const int32_t* __restrict__ ids,
                                                                  const float* __restrict__ w, int topk, int E,
                                                                  int H, float* __restrict__ out) {
    const int64_t t = blockIdx.y, n = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (n >= H) return;
    // the token's ids, weights and slots first, then all its Y loads, then the sum in slot
    // order j (topk <= 16): no load waits on the previous slot's
    constexpr int kMaxK = 16;
    int slot[kMaxK];
    float wv[kMaxK];
#pragma unroll
    for (int j = 0; j < kMaxK; ++j) {
        const int64_t p = t * topk + j;
        const int e = j < topk ? ids[p] : -1;
        const bool ok = e >= 0 && e < E;
        slot[j] = ok ? slot_of_pair[p] : -1;
        wv[j] = ok ? w[p] : 0.f;
    }
    f32x4 v[kMaxK];
#pragma unroll
    for (int j = 0; j < kMaxK; ++j)
        if (slot[j] >= 0) v[j] = *(const f32x4*)(Y + (int64_t)slot[j] * H + n);
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kMaxK; ++j)
        if (slot[j] >= 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) s[c] += wv[j] * v[j][c];
        }
    *(f32x4*)(out + t * H + n) = s;
}

struct MoePfWs {
    size_t cnt, off, meta, tile_e, tile_end, sop, rowmap, texp, x16, gy, total;
    int64_t tiles_max;
};

// Workspace layout for T tokens x topk over E experts (slots: every tile an expert could use).
MoePfWs moe_pf_ws(int T, int E, int topk, int64_t H, int64_t F) {
    MoePfWs w{};
    const int64_t P = (int64_t)T * topk;
    w.tiles_max = ceil_div(P, 256) + (E < P ? E : P);
    const size_t S = (size_t)w.tiles_max * 256;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += align256(bytes);
        return at;
    };
    w.cnt = take((size_t)E * 4);
    w.off = take((size_t)E * 4);
    w.meta = take(16);
    w.tile_e = take((size_t)w.tiles_max * 4);
    w.tile_end = take((size_t)w.tiles_max * 4);
    w.sop = take((size_t)P * 4);
    w.rowmap = take(S * 4);
    w.texp = take(S * 4);
    const size_t x16a = S * H * 2, x16b = 2 * S * F * 2;
    w.x16 = take(x16a > x16b ? x16a : x16b);       // x, then h (value and remainder planes)
    w.gy = take(S * (2 * F > H ? 2 * F : H) * 4);  // G, then Y
    w.total = o;
    return w;
}

}  // namespace

extern "C" size_t q4_moe_prefill_workspace_bytes(int T, int E, int topk, int H, int F) {
    if (T <= 0 || E <= 0 || topk <= 0 || H <= 0 || F <= 0) return 0;
    return moe_pf_ws(T, E, topk, H, F).total;
}

extern "C" int q4_moe_prefill(const uint8_t* gate_up, const uint8_t* down, const void* gate_up_scales,
                              const void* down_scales, const void* x, int x_dtype, const int32_t* topk_ids,
                              const float* topk_w, float* out, int T, int E, int topk, int64_t H, int64_t F,
                              int precision, void* workspace, size_t workspace_bytes, void* stream) {
    if (precision < 0 || precision > 2) return Q4MI_E_ARG;
    // precision 2: the fp16 tile of precision 0 with h rounded to bf16 (one down pass)
    const bool hb16 = precision != 0;
    precision = precision == 2 ? 0 : precision;
    if (x_dtype != Q4MI_F32 && x_dtype != Q4MI_BF16) return Q4MI_E_ARG;
    if (H <= 0 || F <= 0 || H % 256 || F % 128) return Q4MI_E_SHAPE;
    if (H > (1 << 20) || F > (1 << 20)) return Q4MI_E_RANGE;
    if (T < 0 || E <= 0 || E > kMoePfMaxExperts || topk <= 0 || topk > 16 || (int64_t)T * topk > kMoePfMaxPairs)
        return Q4MI_E_RANGE;
    if (T == 0) return Q4MI_OK;
    if (!gate_up || !down || !x || !topk_ids || !topk_w || !out) return Q4MI_E_ARG;
    if (misaligned16(gate_up) || misaligned16(down) || misaligned16(x) || misaligned16(out) || misaligned16(workspace))
        return Q4MI_E_ARG;
    if (precision == 0 && (!gate_up_scales || !down_scales || misaligned16(gate_up_scales) ||
                           misaligned16(down_scales)))
        return Q4MI_E_ARG;
    const MoePfWs w = moe_pf_ws(T, E, topk, H, F);
    if (!workspace || workspace_bytes < w.total) return Q4MI_E_WORKSPACE;
    char* ws = (char*)workspace;
    int* cnt = (int*)(ws + w.cnt);
    int* off = (int*)(ws + w.off);
    int* meta = (int*)(ws + w.meta);
    int* tile_e = (int*)(ws + w.tile_e);
    int* tile_end = (int*)(ws + w.tile_end);
    int* sop = (int*)(ws + w.sop);
    int* rowmap = (int*)(ws + w.rowmap);
    int* texp = (int*)(ws + w.texp);
    uint16_t* x16 = (uint16_t*)(ws + w.x16);
    float* gy = (float*)(ws + w.gy);
    const int P = T * topk;
    const hipStream_t st = (hipStream_t)stream;
    const unsigned S = (unsigned)(w.tiles_max * 256), SP = S / 4;
    const bool xf32 = x_dtype == Q4MI_F32;
    const bool ragged = P < (int64_t)256 * kMoeFullTiles * E;

    hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(1024), 0, st, topk_ids, P, E, cnt, off, tile_e, tile_end, meta);
    if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    // precision 0, token rows within a gather resource's range: the gate/up GEMM gathers them
    // (below), and their pre-pass rides in the slots' launch
    const bool gx = precision == 0 && (uint64_t)T * H * 2 <= kGatherBytes;
    if (gx && xf32)
        hipLaunchKernelGGL((moe_slots_xprep_kernel<true>), dim3((unsigned)(E + T)), dim3(256), 0, st, topk_ids, P,
                           topk, E, cnt, off, sop, rowmap, x, x16, texp, (int)H);
    else if (gx)
        hipLaunchKernelGGL((moe_slots_xprep_kernel<false>), dim3((unsigned)(E + T)), dim3(256), 0, st, topk_ids, P,
                           topk, E, cnt, off, sop, rowmap, x, x16, texp, (int)H);
    else
        hipLaunchKernelGGL(moe_slots_kernel, dim3((unsigned)E), dim3(256), 0, st, topk_ids, P, topk, cnt, off, sop,
                           rowmap);
    if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;

    // the prefill scales: wexp int32[N], then the fp16 plane, per stacked matrix
    auto plane = [](const void* sc, int64_t N) {
        return (const uint32_t*)((const char*)sc + align256((size_t)N * 4));
    };
    const int64_t N1 = 2 * F, N2 = H;
    const int64_t eb1 = (N1 / 64) * (H / 32) * kTileBytes, eb2 = (N2 / 64) * (F / 32) * kTileBytes;
    const int64_t sw1 = (N1 / 64) * (H / 32) * 64, sw2 = (N2 / 64) * (F / 32) * 64;
    const int* we1 = precision == 0 ? (const int*)gate_up_scales : nullptr;
    const int* we2 = precision == 0 ? (const int*)down_scales : nullptr;
    const uint32_t* s1 = precision == 0 ? plane(gate_up_scales, (int64_t)E * N1) : nullptr;
    const uint32_t* s2 = precision == 0 ? plane(down_scales, (int64_t)E * N2) : nullptr;
    const unsigned g1 = (unsigned)(w.tiles_max * (N1 / 256)), g2 = (unsigned)(w.tiles_max * (N2 / 256));

    // precision 1 on bf16 x: the expert GEMMs DMA their token rows straight from x (gate/up,
    // slot s <- token rowmap[s]) and from h (down, slot s <- h row s): no per-slot activation
    // images. h [S][F] bf16 from the gate/up epilogue goes to the x16 region, Y to gy. Rows past
    // a gather resource's range would read as zeros, so longer x or h take the images.
    const bool gather = precision == 1 && !xf32 && (uint64_t)T * H * 2 <= kGatherBytes &&
                        (uint64_t)S * F * 2 <= kGatherBytes;
    if (gather) {
        launch_moe_dma<1, true, true>(ragged, g1, st, gate_up, eb1,
                           (const uint16_t*)x, texp, we1, s1, sw1, (float*)x16, tile_e, tile_end, meta, (int)N1,
                           (int)H, (int)(N1 / 256), 0, (const int*)rowmap);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
        launch_moe_dma<1, false, true>(ragged, g2, st, down, eb2, x16, texp, we2, s2,
                           sw2, gy, tile_e, tile_end, meta, (int)N2, (int)F, (int)(N2 / 256), 0, (const int*)nullptr);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
        hipLaunchKernelGGL(moe_prefill_combine_kernel, dim3((unsigned)ceil_div(H / 4, 256), (unsigned)T), dim3(256), 0,
                           st, gy, sop, topk_ids, topk_w, topk, E, (int)H, out);
        return launch_status();
    }

    // gate/up: G = X . [gate; up]^T per expert. Precision 0: the token rows go through the
    // pre-pass once per token ([T][H] fp16 and the token exponents, in the x16 and texp
    // regions) and the GEMM gathers them per slot; the h preps overwrite both afterwards.
    const int xpasses = precision == 0 && xf32 ? 2 : 1;
    const bool swi = hb16 && xpasses == 1;
    for (int pass = 0; pass < xpasses; ++pass) {
        if (gx && pass == 0) {
            // done with the slots
        } else if (gx) {
            // the remainder pass of f32 x, in rows for the gather
            hipLaunchKernelGGL((prefill_xprep<true, 0, false>), dim3((unsigned)T), dim3(256), 0, st, x, x16, texp, T,
                               (int)H, pass);
        } else if (xf32) {
            if (precision == 0)
                hipLaunchKernelGGL((moe_xprep_kernel<true, 0>), dim3(SP), dim3(256), 0, st, x, rowmap, meta, x16, texp,
                                   (int)H, pass);
            else
                hipLaunchKernelGGL((moe_xprep_kernel<true, 1>), dim3(SP), dim3(256), 0, st, x, rowmap, meta, x16, texp,
                                   (int)H, pass);
        } else {
            if (precision == 0)
                hipLaunchKernelGGL((moe_xprep_kernel<false, 0>), dim3(SP), dim3(256), 0, st, x, rowmap, meta, x16,
                                   texp, (int)H, pass);
            else
                hipLaunchKernelGGL((moe_xprep_kernel<false, 1>), dim3(SP), dim3(256), 0, st, x, rowmap, meta, x16,
                                   texp, (int)H, pass);
        }
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
        // bf16 h from one activation pass: SwiGLU in the gate/up epilogue, h [S][F] bf16 in
        // the G/Y buffer (G itself is never written)
        if (swi && gx)
            launch_moe_dma<0, true, true>(ragged, g1, st, gate_up, eb1, x16, texp,
                               we1, s1, sw1, gy, tile_e, tile_end, meta, (int)N1, (int)H, (int)(N1 / 256), 0,
                               (const int*)rowmap);
        else if (swi && precision == 0)
            launch_moe_dma<0, true>(ragged, g1, st, gate_up, eb1, x16, texp, we1, s1,
                               sw1, gy, tile_e, tile_end, meta, (int)N1, (int)H, (int)(N1 / 256), 0);
        else if (swi)
            launch_moe_dma<1, true>(ragged, g1, st, gate_up, eb1, x16, texp, we1, s1,
                               sw1, gy, tile_e, tile_end, meta, (int)N1, (int)H, (int)(N1 / 256), 0);
        else if (gx)
            launch_moe_dma<0, false, true>(ragged, g1, st, gate_up, eb1, x16, texp,
                               we1, s1, sw1, gy, tile_e, tile_end, meta, (int)N1, (int)H, (int)(N1 / 256), pass,
                               (const int*)rowmap);
        else if (precision == 0)
            launch_moe_dma<0>(ragged, g1, st, gate_up, eb1, x16, texp, we1, s1, sw1,
                               gy, tile_e, tile_end, meta, (int)N1, (int)H, (int)(N1 / 256), pass);
        else
            launch_moe_dma<1>(ragged, g1, st, gate_up, eb1, x16, texp, we1, s1, sw1,
                               gy, tile_e, tile_end, meta, (int)N1, (int)H, (int)(N1 / 256), 0);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    }
    // h = silu(g) u into the 16-bit layout (precision 0: value and remainder planes, both
    // made before the down GEMM overwrites G with Y)
    const int hpasses = precision == 0 && !hb16 ? 2 : 1;
    uint16_t* h16[2] = {x16, x16 + (size_t)S * F};
    for (int pass = 0; pass < hpasses; ++pass) {
        if (swi && precision == 0)
            launch_h16prep<0>(S, st, (const uint16_t*)gy, tile_end, meta, h16[0], texp, (int)F, ragged);
        else if (swi)
            launch_h16prep<1>(S, st, (const uint16_t*)gy, tile_end, meta, h16[0], texp, (int)F, ragged);
        else if (precision == 0 && hb16)
            hipLaunchKernelGGL((moe_hprep_kernel<0, true>), dim3(SP), dim3(256), 0, st, gy, rowmap, meta, h16[pass],
                               texp, (int)F, 0);
        else if (precision == 0)
            hipLaunchKernelGGL((moe_hprep_kernel<0>), dim3(SP), dim3(256), 0, st, gy, rowmap, meta, h16[pass], texp,
                               (int)F, pass);
        else
            hipLaunchKernelGGL((moe_hprep_kernel<1>), dim3(SP), dim3(256), 0, st, gy, rowmap, meta, h16[pass], texp,
                               (int)F, pass);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    }
    for (int pass = 0; pass < hpasses; ++pass) {
        if (precision == 0)
            launch_moe_dma<0>(ragged, g2, st, down, eb2, h16[pass], texp, we2, s2,
                               sw2, gy, tile_e, tile_end, meta, (int)N2, (int)F, (int)(N2 / 256), pass);
        else
            launch_moe_dma<1>(ragged, g2, st, down, eb2, h16[pass], texp, we2, s2,
                               sw2, gy, tile_e, tile_end, meta, (int)N2, (int)F, (int)(N2 / 256), 0);
        if (launch_status() != Q4MI_OK) return Q4MI_E_LAUNCH;
    }
    hipLaunchKernelGGL(moe_prefill_combine_kernel, dim3((unsigned)ceil_div(H / 4, 256), (unsigned)T), dim3(256), 0, st,
                       gy, sop, topk_ids, topk_w, topk, E, (int)H, out);
    return launch_status();
}
