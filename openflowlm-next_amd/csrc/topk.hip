// topk.hip -- the lm_head's sampling epilogue: for each token row of logits, the k largest
// (value descending, the lower id first on a tie), as ids and values; k = 1 is the greedy
// argmax. Plus q4_lm_head_topk, the lm_head GEMV followed by it on one stream.
//
// Reference semantics followed:
//   greedy: Sampler::sample_greedy (src/common/modules/sampler.cpp:355-430) over
//     Engine::logits_view's bf16 logits (src/open_qwen36/engine.cpp:125-131), stated
//     for the tests as argmax_bf16 (src/open_qwen36/cli.cpp:103-113): each f32 logit
//     rounded to bf16 (RNE, the plain formula), an f32 subnormal read as 0, strict '>'
//     from -inf so the lowest id wins a tie and an all -inf / NaN row gives id 0; rows
//     past the real vocabulary read as -inf.
//   top-k: Sampler::sampler_topk_apply (sampler.cpp:222-245): value descending, lower id
//     first when the values are equal.
//
// Every (value, id) becomes one uint64 key whose unsigned order is that order:
//   high word: the value's bits made monotone (sign set -> all bits flipped, else the
//   sign bit set), with -0 read as +0 and NaN as 0, below every number; low word: ~id.
// Padding slots are key 0, below every real key. Each lane holds 4 keys. For k <= 8 a
// block of 4 waves takes 1024 logits: each lane sorts its 4 keys in registers, each
// wave pops its k largest with k pairs of DPP wave reductions, and wave 0 merges the
// four wave lists the same way. For larger k a block of 16 waves takes up to 4096: the keys
// that reach a bound that 64 of them reach are ranked by counting. Blocks emit k (64 for the
// larger k) keys each; the same kernel then runs over those keys until one block per token
// remains, which writes ids and values.
#include "q4mi_device.h"
#include "q4mi_internal.h"

using namespace q4mi;

namespace {

constexpr int kLanes = 64, kWaves = 4, kThreads = kLanes * kWaves, kPerLane = 4;
constexpr int kChunk = kThreads * kPerLane;     // 1024 inputs per block
constexpr int kMaxK = 64;

__device__ __forceinline__ uint32_t monotone(float v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float from_monotone(uint32_t k) {
    return __builtin_bit_cast(float, (k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// mode 0: the f32 logit; mode 1: what the sampler sees (bf16 RNE, f32 subnormal -> 0).
__device__ __forceinline__ uint64_t logit_key(float v, uint32_t id, int mode) {
    if (mode == 1) {
        const uint32_t u = __builtin_bit_cast(uint32_t, v);
        v = ((u & 0x7F800000u) == 0) ? 0.0f : __builtin_bit_cast(float, f32_to_bf16_rne(v) << 16);
    }
    if (v == 0.0f) v = 0.0f;                          // -0 ties with +0
    const uint32_t hi = (v != v) ? 0u : monotone(v);  // NaN below every number
    return ((uint64_t)hi << 32) | (uint32_t)~id;
}

// Wave-wide unsigned max / min with the result in every lane: DPP steps (xor 1 and 2
// within quads, half-row and row mirrors, then the row broadcasts of lanes 15 and 31)
// leave the total in lane 63, which readlane hands to the whole wave.
template <bool MAX>
__device__ __forceinline__ uint32_t dpp_step(uint32_t v, uint32_t o) {
    return MAX ? (o > v ? o : v) : (o < v ? o : v);
}

template <bool MAX>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v) {
    v = dpp_step<MAX>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xF, 0xF, false));
    v = dpp_step<MAX>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xF, 0xF, false));
    v = dpp_step<MAX>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xF, 0xF, false));
    v = dpp_step<MAX>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xF, 0xF, false));
    v = dpp_step<MAX>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xA, 0xF, false));
    v = dpp_step<MAX>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xC, 0xF, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Sort N keys descending in registers (bitonic network, all indices compile-time).
template <int N>
__device__ __forceinline__ void sort_desc(uint64_t (&a)[N]) {
#pragma unroll
    for (int s = 2; s <= N; s <<= 1)
#pragma unroll
        for (int j = s >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int l = i ^ j;
                if (l > i) {
                    const bool desc = (i & s) == 0;
                    const uint64_t x = a[i], y = a[l];
                    const bool swap = desc ? (x < y) : (x > y);
                    a[i] = swap ? y : x;
                    a[l] = swap ? x : y;
                }
            }
}

// Pop the k largest keys of the wave (each lane's a[] sorted descending): lane t < k
// returns the t-th largest, or 0 when the wave held fewer than t + 1 real keys. Each
// pop is two 32-bit wave reductions: the largest value, then the lowest id holding it
// (a padding slot is value 0 with id 0xFFFFFFFF; a NaN is value 0 with its own id).
template <int N>
__device__ __forceinline__ uint64_t wave_pop(uint64_t (&a)[N], int k, int lane) {
    uint64_t mine = 0;
    for (int t = 0; t < k; ++t) {
        const uint32_t hv = (uint32_t)(a[0] >> 32), hid = ~(uint32_t)a[0];
        const uint32_t mv = wave_reduce_u32<true>(hv);
        const uint32_t mid = wave_reduce_u32<false>(hv == mv ? hid : 0xFFFFFFFFu);
        if (mv == 0 && mid == 0xFFFFFFFFu) break;          // only padding left (wave-uniform)
        if (lane == t) mine = ((uint64_t)mv << 32) | (uint32_t)~mid;
        if (hv == mv && hid == mid) {                       // the one lane that held it
#pragma unroll
            for (int i = 0; i + 1 < N; ++i) a[i] = a[i + 1];
            a[N - 1] = 0;
        }
    }
    return mine;
}

// The k > 8 block: 16 waves over up to 4096 inputs, 4 per lane, its top 64 found by
// filtering and counting. The lanes' quads are 256 groups of up to 16 keys; a bound that 64 of
// the groups' maxima reach is one that at least 64 keys reach, so only the keys that reach it
// can be among the top 64. The largest value (a key's high word) that serves, to its top
// kBoundBits, is found bit by bit with ballots (by one wave: the counting is scalar work, and a
// CU has one scalar unit for its 16 waves): 70 to 90 of a full block's keys reach it in any
// order that does not depend on the position. They are compacted into LDS (in any order) and
// each one's rank is the number of larger ones, counted by 1024 / slots threads per key; keys
// are distinct, so the ranks are too. Keys of an earlier pass arrive as sorted runs of 64: quad
// q of a wave takes a run's places q mod 16, so the groups' maxima are the runs' leading keys.
// Where more than kRanked keys reach the bound (a masked row: most logits one value) it is found
// again to the last bit of the key, value and id: then exactly 64 groups reach it, which hold at
// most 1024 keys. (Ranking costs 1.7 us for 256 keys, 2.9 for 260 and 7 for 500; finding the
// bound again and ranking what is left about 4.) Where more than kRanked of those do, they are
// one per lane, so quads of them are groups of 4 and the same bound over these leaves at most
// 256. Non-final passes write their top 64 (a superset of the top k); the final pass writes the
// first k as ids and values. Cost does not depend on k. 8 rows of 128256 f32 logits, k = 40,
// both passes: a bitonic sort of the block's keys 21.4 us for any values; this 10.3 (N(0, 1)),
// 18.3 (all but 50 logits -inf) and 21.3 (values that repeat every 256 logits, filtered twice).
constexpr int kFilterWaves = 16, kFilterThreads = kFilterWaves * kLanes, kFilterChunk = kFilterThreads * kPerLane;
constexpr int kRanked = 320, kSlots = 512, kGroups = kFilterThreads / 4, kBoundBits = 18;
static_assert(kGroups == 4 * kLanes, "four groups per lane");

// The largest value over each quad of lanes, in all of them.
__device__ __forceinline__ uint32_t quad_max_u32(uint32_t v) {
    v = dpp_step<true>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xF, 0xF, false));
    return dpp_step<true>(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xF, 0xF, false));
}

// One wave, four groups per lane: the largest number that 64 of the groups' reach and that has
// from's bits above hi and zeros below lo (from itself is reached by 64).
__device__ __forceinline__ uint32_t reached_by_64(const uint4& g, uint32_t from, int hi, int lo) {
    for (int b = hi; b >= lo; --b) {
        const uint32_t v = from | 1u << b;
        const int reach = __popcll(__ballot(g.x >= v)) + __popcll(__ballot(g.y >= v)) + __popcll(__ballot(g.z >= v)) +
                          __popcll(__ballot(g.w >= v));
        if (reach >= kLanes) from = v;
    }
    return from;
}

struct FilterLds {
    alignas(16) uint64_t found[kFilterThreads];  // the keys that reach the bound, zeros behind them
    alignas(16) uint32_t high[kGroups], low[kGroups];   // the groups' maxima
    uint64_t top[kLanes], bound;
    int rank[kSlots], count[3];
};

// The largest key that 64 of the groups' maxima reach, the threads' keys a in quads; the `known`
// leading bits of its value are those of from. found is cleared. Every thread calls it (barriers
// inside).
template <int N>
__device__ __forceinline__ uint64_t exact_bound(const uint64_t (&a)[N], uint32_t from, int known, FilterLds& m) {
    const int tid = threadIdx.x;
    uint32_t high = 0, low = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) high = dpp_step<true>(high, (uint32_t)(a[j] >> 32));
    high = quad_max_u32(high);
#pragma unroll
    for (int j = 0; j < N; ++j)
        if ((uint32_t)(a[j] >> 32) == high) low = dpp_step<true>(low, (uint32_t)a[j]);
    low = quad_max_u32(low);
    if ((tid & 3) == 0) m.high[tid >> 2] = high, m.low[tid >> 2] = low;
    __syncthreads();
    m.found[tid] = 0;
    if (tid < kLanes) {
        const uint4 g = *(const uint4*)(m.high + 4 * tid);
        uint4 l = *(const uint4*)(m.low + 4 * tid);
        const uint32_t v = reached_by_64(g, from, 31 - known, 0);
        // fewer than 64 lead with more: the id's word is among those that lead with v, and has the
        // bits that these share
        uint32_t most = 0, least = ~0u;
        auto leading = [&](uint32_t gv, uint32_t& lv) {
            if (gv == v) most = dpp_step<true>(most, lv), least = dpp_step<false>(least, lv);
            else lv = gv > v ? ~0u : 0u;
        };
        leading(g.x, l.x), leading(g.y, l.y), leading(g.z, l.z), leading(g.w, l.w);
        most = wave_reduce_u32<true>(most), least = wave_reduce_u32<false>(least);
        const int hi = 31 - __builtin_clz((most ^ least) | 1u);
        const uint32_t i = reached_by_64(l, most & ~((2u << hi) - 1u), hi, 0);
        if (tid == 0) m.bound = (uint64_t)v << 32 | i;
    }
    __syncthreads();
    return m.bound;
}

// The keys that reach the bound (padding, key 0, never does) into found; their number, counted in
// count (zero before). Every thread calls it (a barrier inside).
template <int N>
__device__ __forceinline__ int collect(const uint64_t (&a)[N], uint64_t bound, FilterLds& m, int* count) {
    const int lane = threadIdx.x & (kLanes - 1);
    uint64_t hit[N];
    int c = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        hit[j] = __ballot(a[j] != 0 && a[j] >= bound);
        c += __popcll(hit[j]);
    }
    int o = 0;
    if (lane == 0 && c) o = atomicAdd(count, c);
    o = __builtin_amdgcn_readfirstlane(o);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int to = o + __popcll(hit[j] & ((1ull << lane) - 1ull));
        if ((hit[j] >> lane & 1) && to < kFilterThreads) m.found[to] = a[j];
        o += __popcll(hit[j]);
    }
    __syncthreads();
    return *count;
}

// Block s: inputs [s * chunk, min(n, (s + 1) * chunk)) of token row m, chunk <= kFilterChunk.
template <bool KEYS, bool FINAL>
__global__ __launch_bounds__(kFilterThreads) void topk_filter_kernel(const void* __restrict__ in, int64_t ld,
                                                                     int64_t n, int chunk, int k, int mode,
                                                                     uint64_t* __restrict__ out_keys,
                                                                     int32_t* __restrict__ ids,
                                                                     float* __restrict__ vals) {
    __shared__ FilterLds lds;
    const int tid = threadIdx.x, lane = tid & (kLanes - 1), wave = tid / kLanes;
    const int64_t s = blockIdx.x, m = blockIdx.y, base = s * chunk;
    const int at = wave * kLanes + (KEYS ? (lane >> 2) + 16 * (lane & 3) : lane);
    uint64_t a[kPerLane];
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int o = j * kFilterThreads + at;
        const int64_t i = base + o;
        if (o < chunk && i < n) {
            if constexpr (KEYS)
                a[j] = ((const uint64_t*)in)[m * ld + i];
            else
                a[j] = logit_key(((const float*)in)[m * ld + i], (uint32_t)i, mode);
        } else {
            a[j] = 0;
        }
    }
    lds.found[tid] = 0;
    if (tid < kSlots) lds.rank[tid] = 0;
    if (tid < kLanes) lds.top[tid] = 0;
    if (tid < 3) lds.count[tid] = 0;
    uint32_t high = 0;
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) high = dpp_step<true>(high, (uint32_t)(a[j] >> 32));
    high = quad_max_u32(high);
    if ((lane & 3) == 0) lds.high[tid >> 2] = high;
    __syncthreads();
    if (wave == 0) {
        const uint32_t v = reached_by_64(*(const uint4*)(lds.high + 4 * lane), 0, 31, 32 - kBoundBits);
        if (lane == 0) lds.bound = (uint64_t)v << 32;
    }
    __syncthreads();
    const uint64_t bound = lds.bound;
    int total = collect(a, bound, lds, &lds.count[0]);
    if (total > kRanked) {
        total = collect(a, exact_bound(a, (uint32_t)(bound >> 32), kBoundBits, lds), lds, &lds.count[1]);
        if (total > kRanked) {
            const uint64_t one[1] = {lds.found[tid]};
            total = collect(one, exact_bound(one, 0, 0, lds), lds, &lds.count[2]);
        }
    }
    // thread (slot, part): the larger keys among part's share of those found (an even number
    // from an even place; the zeros behind the last one count for none)
    const int slots = total <= kSlots / 4 ? kSlots / 4 : total <= kSlots / 2 ? kSlots / 2 : kSlots;
    const int parts = kFilterThreads / slots;
    const int slot = tid & (slots - 1), part = tid / slots;
    const int share = ((total + parts - 1) / parts + 1) & ~1;
    const int j0 = min(part * share, total), j1 = min(j0 + share, total);
    const uint64_t key = lds.found[slot];
    int larger = 0;
    if ((slot & ~(kLanes - 1)) < total) {                 // wave-uniform
#pragma unroll 4
        for (int j = j0; j < j1; j += 2) {
            const ulonglong2 v = *(const ulonglong2*)(lds.found + j);
            larger += (v.x > key) + (v.y > key);
        }
        atomicAdd(&lds.rank[slot], larger);
    }
    __syncthreads();
    if (tid < total && lds.rank[tid] < kLanes) lds.top[lds.rank[tid]] = lds.found[tid];
    __syncthreads();
    if (wave != 0) return;
    const uint64_t out = lds.top[lane];
    if constexpr (FINAL) {
        if (lane < k) {
            ids[m * k + lane] = out ? (int32_t)~(uint32_t)out : -1;
            if (vals) vals[m * k + lane] = out ? from_monotone((uint32_t)(out >> 32)) : -__builtin_inff();
        }
    } else {
        out_keys[(m * gridDim.x + s) * kLanes + lane] = out;
    }
}

// One block: inputs [s*1024, min(n, (s+1)*1024)) of token row m -> its k largest keys.
// KEYS: the inputs are keys of an earlier pass (uint64[M][n]); else f32 logits (row
// stride ld). FINAL: write ids / values; else keys to out_keys[m][s][k].
template <bool KEYS, bool FINAL>
__global__ __launch_bounds__(kThreads) void topk_kernel(const void* __restrict__ in, int64_t ld, int64_t n,
                                                        int k, int mode, uint64_t* __restrict__ out_keys,
                                                        int32_t* __restrict__ ids, float* __restrict__ vals) {
    __shared__ uint64_t lists[kWaves][kLanes];
    const int lane = threadIdx.x & (kLanes - 1), wave = threadIdx.x / kLanes;
    const int64_t s = blockIdx.x, m = blockIdx.y;
    const int64_t base = s * kChunk + wave * (kLanes * kPerLane);
    uint64_t a[kPerLane];
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int64_t i = base + j * kLanes + lane;          // coalesced: 64 consecutive per j
        if (i < n) {
            if constexpr (KEYS)
                a[j] = ((const uint64_t*)in)[m * ld + i];
            else
                a[j] = logit_key(((const float*)in)[m * ld + i], (uint32_t)i, mode);
        } else {
            a[j] = 0;
        }
    }
    sort_desc(a);
    lists[wave][lane] = wave_pop(a, k, lane);
    __syncthreads();
    if (wave != 0) return;
    uint64_t b[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) b[w] = lists[w][lane];
    sort_desc(b);
    const uint64_t key = wave_pop(b, k, lane);
    if (lane < k) {
        if constexpr (FINAL) {
            ids[m * k + lane] = key ? (int32_t)~(uint32_t)key : -1;
            if (vals) vals[m * k + lane] = key ? from_monotone((uint32_t)(key >> 32)) : -__builtin_inff();
        } else {
            out_keys[(m * gridDim.x + s) * k + lane] = key;
        }
    }
}

constexpr int kPopMaxK = 8;     // k above this: the filtering block

// Pass geometry: inputs per block and keys each non-final block writes.
struct TopkPlan {
    bool pop;
    int64_t chunk;
    int out;
};

inline TopkPlan topk_plan(int k) {
    return k <= kPopMaxK ? TopkPlan{true, kChunk, k} : TopkPlan{false, kFilterChunk, 64};
}

template <bool KEYS>
void launch_topk(const TopkPlan& p, bool final_pass, dim3 grid, hipStream_t st, const void* in, int64_t ld,
                 int64_t n, int k, int mode, uint64_t* out_keys, int32_t* ids, float* vals) {
    if (p.pop) {
        if (final_pass)
            hipLaunchKernelGGL((topk_kernel<KEYS, true>), grid, dim3(kThreads), 0, st, in, ld, n, k, mode, out_keys,
                               ids, vals);
        else
            hipLaunchKernelGGL((topk_kernel<KEYS, false>), grid, dim3(kThreads), 0, st, in, ld, n, k, mode,
                               out_keys, ids, vals);
    } else {
        // even chunks, whole runs of 64: a short last block would pass its group bound too easily
        const int chunk = (int)(ceil_div(ceil_div(n, (int64_t)grid.x), (int64_t)kLanes) * kLanes);
        if (final_pass)
            hipLaunchKernelGGL((topk_filter_kernel<KEYS, true>), grid, dim3(kFilterThreads), 0, st, in, ld, n, chunk, k,
                               mode, out_keys, ids, vals);
        else
            hipLaunchKernelGGL((topk_filter_kernel<KEYS, false>), grid, dim3(kFilterThreads), 0, st, in, ld, n, chunk, k,
                               mode, out_keys, ids, vals);
    }
}

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Two key buffers, ping-ponged: the first pass's output, and the second's (every later
// pass writes fewer keys than the one two before it).
size_t topk_ws(int M, int64_t n, int k) {
    const TopkPlan p = topk_plan(k);
    const int64_t s1 = ceil_div(n, p.chunk);
    if (s1 <= 1) return 0;
    const int64_t s2 = ceil_div(s1 * p.out, p.chunk);
    return align256((size_t)M * s1 * p.out * 8) + (s2 > 1 ? align256((size_t)M * s2 * p.out * 8) : 0);
}

}  // namespace

extern "C" size_t q4_topk_workspace_bytes(int M, int64_t n, int k) {
    if (M <= 0 || n <= 0 || k < 1 || k > kMaxK) return 0;
    return topk_ws(M, n, k);
}

extern "C" int q4_logits_topk(const float* logits, int64_t ld, int M, int64_t n, int k, int mode, int32_t* ids,
                              float* vals, void* workspace, size_t workspace_bytes, void* stream) {
    if (k < 1 || k > kMaxK || (mode != 0 && mode != 1)) return Q4MI_E_RANGE;
    if (M < 0 || M > 65535) return Q4MI_E_RANGE;
    if (M == 0) return Q4MI_OK;
    if (n <= 0 || ld < n) return Q4MI_E_SHAPE;
    if (!logits || !ids) return Q4MI_E_ARG;
    if ((uintptr_t)workspace & 7) return Q4MI_E_ARG;
    const size_t need = topk_ws(M, n, k);
    if (need && (!workspace || workspace_bytes < need)) return Q4MI_E_WORKSPACE;
    const hipStream_t st = (hipStream_t)stream;
    const TopkPlan p = topk_plan(k);
    int64_t s = ceil_div(n, p.chunk);
    uint64_t* buf[2] = {(uint64_t*)workspace,
                        need ? (uint64_t*)((char*)workspace + align256((size_t)M * s * p.out * 8)) : nullptr};
    launch_topk<false>(p, s == 1, dim3((unsigned)s, (unsigned)M), st, logits, ld, n, k, mode, buf[0], ids, vals);
    int cur = 0;
    while (s > 1) {                 // reduce the keys of s blocks per token until one block is left
        const int64_t len = s * p.out;
        s = ceil_div(len, p.chunk);
        launch_topk<true>(p, s == 1, dim3((unsigned)s, (unsigned)M), st, buf[cur], len, len, k, mode, buf[cur ^ 1],
                          ids, vals);
        cur ^= 1;
    }
    return launch_status();
}

extern "C" size_t q4_lm_head_workspace_bytes(int M, int64_t N, int64_t K, int k) {
    if (M <= 0 || M > 16 || N <= 0 || k < 1 || k > kMaxK) return 0;
    return align256(q4_gemv_workspace_bytes(M, N, K)) + topk_ws(M, N, k);
}

extern "C" int q4_lm_head_topk(const uint8_t* packed, const void* x, int x_dtype, float* logits, int M, int64_t N,
                               int64_t K, int64_t n_valid, int k, int mode, int32_t* ids, float* vals,
                               void* workspace, size_t workspace_bytes, void* stream) {
    if (n_valid <= 0 || n_valid > N) return Q4MI_E_SHAPE;
    if (k < 1 || k > kMaxK || (mode != 0 && mode != 1)) return Q4MI_E_RANGE;
    if (M < 0 || M > 16) return Q4MI_E_RANGE;
    if (M == 0) return Q4MI_OK;
    if (!ids) return Q4MI_E_ARG;
    const size_t gws = q4_gemv_workspace_bytes(M, N, K);
    const size_t need = align256(gws) + topk_ws(M, n_valid, k);
    if (need && (!workspace || workspace_bytes < need)) return Q4MI_E_WORKSPACE;
    int rc = q4_gemv(packed, x, x_dtype, logits, M, N, K, gws ? workspace : nullptr, gws, stream);
    if (rc != Q4MI_OK) return rc;
    void* tws = need > align256(gws) ? (void*)((char*)workspace + align256(gws)) : nullptr;
    return q4_logits_topk(logits, N, M, n_valid, k, mode, ids, vals, tws, need - align256(gws), stream);
}
