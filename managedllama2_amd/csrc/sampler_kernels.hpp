// The stochastic sampler of src/Sampler.cs:48-67 on many workgroups: softmax_logits, sort,
// cumulative_sum, sample_top_p (native/softmax_logits_kernel.cu, sort_kernel.cu, cumulative_sum_kernel.cu,
// sample_top_p_kernel.cu) as four launches, one for every point where a value of the whole vocabulary has to
// be known before the next step:
//   sampler_exp_kernel    the largest logit (every workgroup reads all of them), exp, sums of 32 or 64 terms
//   sampler_tile_kernel   the sum, the probabilities, tiles of 1024 of them sorted
//   sampler_rank_kernel   the place of every item: how many items of each tile sort in front of it
//   sampler_pick_kernel   prefix sums and the pick
// A short vector that need not be sorted takes one launch of one workgroup (sampler_one_kernel).
//
// What bounds it: nothing but latency; 32000 logits are 64 KB.  The reference's shape, one workgroup of 1024
// threads for everything, kept one of 256 compute units busy: the two divisions and the exp of every logit took 14 us
// of its vector units, a radix sort in its LDS 44 us, 67.8 us in all.  These launches take 4.0, 5.8, 5.6 and 6.6 us (profiler),
// 20 us together.  By size, with the 2.5 us copy of the logits in front, one workgroup -> these: 500 logits 39.8 -> 16.8 us,
// 5000 43.7 -> 18.3, 32000 69.6 -> 22.4, 32768 (too many for its LDS) 212 -> 22.3, 65536 388 -> 34.8.
//
// The sums are those of one workgroup of 1024 threads, addition by addition: thread t adds up the 8-element chunks
// t, t + 1024, ... of the exponentials and the chunks t CH .. t CH + CH - 1 of the sorted probabilities, wavefronts
// and the workgroup add up as wave_sum and prefix_totals do.  Every result has the same bits on any grid.
#pragma once

#include "persist.hpp"

namespace l2 {

constexpr int kSampBlock = 1024;
constexpr int kSampWaves = kSampBlock / 64;
constexpr int kSampTile = 1024;                                   // items sorted by one workgroup
constexpr int kSampTiles = LLAMA2_MAX_SAMPLER_SIZE / kSampTile;   // 64
constexpr int kSampRun = 128;                                     // sorted items of a tile placed by one workgroup
constexpr int kSampBuckets = 16;
// The head of the distribution alone is sorted (see SampleArgs::head) for vocabularies up to this size and heads up
// to half of it; both bounds are part of what a caller finds in `logits` and `indices` afterwards.
constexpr int kSampHeadItems = 32256;

// 8-element chunks per thread of the 1024 whose sums the results are: 4 up to 32768 elements, 8 up to 65536
inline int sampler_chunks(int size) { return size <= 4 * 8 * kSampBlock ? 4 : 8; }

// Device memory between the launches, which are in order on the library's stream: one for the modules, and one per decoder.
struct SamplerScratch {
    uint16_t exps[LLAMA2_MAX_SAMPLER_SIZE];  // half(exp(l - max))
    uint16_t keys[LLAMA2_MAX_SAMPLER_SIZE];  // probabilities in the order that the prefix sums take them
    uint16_t ranks[LLAMA2_MAX_SAMPLER_SIZE]; // of the sorted tiles
    uint32_t items[LLAMA2_MAX_SAMPLER_SIZE]; // (rank << 16) | position, sorted tiles
    int payload[LLAMA2_MAX_SAMPLER_SIZE];    // llama2_sort: values of the sorted tiles
    float sums[kSampBlock];                  // of the exponentials, per thread of the 1024
    uint32_t mass[kSampTiles][kSampBuckets]; // probability per binade below the largest, in units of 2^-24
    uint32_t count[kSampTiles][kSampBuckets];
    int probabilities; // the keys are numbers in [0, 1]
    int go;            // a step whose next token is known draws none
    float coin;
};

struct SampleArgs {
    uint16_t* logits;
    int* indices;
    int size;
    float temperature, top_p, coin;
    int* result; // token -> result[pos]
    int pos;
    SamplerScratch* s;
    // The caller reads the token alone: when the largest probabilities together hold more than top_p, they alone are
    // sorted and summed (the token is the same, since Sampler.Sample reads the sorted order only up to the first
    // position whose cumulative sum reaches coin * top_p); `logits` and `indices` hold the head in front and the
    // unsorted probabilities behind it.
    int head;
    // decode step: the position and the prompt's length are read from the device, the coin is that of (seed, pos)
    int* state;
    int* tokens;
    unsigned long long seed;
    float theta;
    HostStep host; // a host's own loop
};

// Queues the four launches (without a sort three, or one); checks nothing.
int sample_enqueue(const char* name, const SampleArgs& a);

inline bool sample_sorts(float top_p) { return !(top_p <= 0.0f || top_p >= 1.0f); } // src/Sampler.cs:56

// Uniform number in [0, 1) for position `pos` of the stream `seed`: splitmix64
// of seed + pos, top 24 bits.  (The reference draws from an unseeded
// System.Random, src/Sampler.cs:24,42.)
__host__ __device__ inline float sampler_coin(unsigned long long seed, int pos)
{
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * static_cast<unsigned long long>(pos + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return static_cast<float>(z >> 40) * (1.0f / 16777216.0f);
}

#if defined(__HIPCC__)

// ---- 8-element chunks of fp16 -------------------------------------------------------
// Whole chunks move as 16-byte accesses, the ragged last chunk element by element.
__device__ __forceinline__ u32x4 load_bits8(const uint16_t* p, int base, int size, uint16_t fill)
{
    if (base + 8 <= size)
        return *reinterpret_cast<const u32x4*>(p + base);
    u32x4 v;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t lo = base + 2 * k < size ? p[base + 2 * k] : fill;
        const uint32_t hi = base + 2 * k + 1 < size ? p[base + 2 * k + 1] : fill;
        v[k] = lo | hi << 16;
    }
    return v;
}

__device__ __forceinline__ void store_half8(uint16_t* p, int base, int size, const uint16_t (&b)[8])
{
    if (base + 8 <= size) {
        u32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            v[k] = static_cast<uint32_t>(b[2 * k]) | (static_cast<uint32_t>(b[2 * k + 1]) << 16);
        *reinterpret_cast<u32x4*>(p + base) = v;
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (base + k < size)
                p[base + k] = b[k];
    }
}

__device__ __forceinline__ float half_of(const u32x4& v, int k)
{
    return half_bits_to_float(static_cast<uint16_t>(v[k >> 1] >> (16 * (k & 1))));
}

// ---- 1. exponentials (native/softmax_logits_kernel.cu:8-53) --------------------------
// p = expf(half(l / temperature) - max), stored as fp16; the sum takes the unrounded p.  A workgroup of 256
// threads computes the sums of 16 of the 1024 threads.  Division by a positive number and rounding keep the order,
// so the maximum of the quotients is the quotient of the maximum and costs one division instead of one per logit in
// every workgroup; for an infinite temperature, whose quotients of infinities are no numbers, it is taken the long way.
constexpr int kExpThreads = 256;
constexpr int kExpShare = 16; // threads of the 1024 per workgroup

template <int CH>
__global__ __launch_bounds__(kExpThreads) void sampler_exp_kernel(SampleArgs a)
{
    constexpr int N = CH * 8; // values per thread of the 1024
    __shared__ float red[kExpThreads / 64];
    __shared__ float val[kExpShare][N + 4];
    if (blockIdx.x == kSampBlock / kExpShare) { // one more workgroup in a decode step
        if (!a.state) {
            write_host_step_state(a.host, threadIdx.x);
            return;
        }
        const int next = a.state[kStatePos] + 1;
        if (threadIdx.x == 0) {
            a.s->go = next >= a.state[kStatePrompt] && next < a.state[kStateSlots];
            a.s->coin = sampler_coin(a.seed, next);
        }
        if (a.state[kStateAdvance] && threadIdx.x >= 64 && threadIdx.x < 64 + kRopeHeadSize / 2)
            write_rope_table(a.state, threadIdx.x - 64, next, a.theta); // for the next step
        return;
    }
    const h2_t lowest = {static_cast<_Float16>(-INFINITY), static_cast<_Float16>(-INFINITY)};
    h2_t m2 = lowest;
    float m = -INFINITY;
    const int whole = a.size >> 3;
    if (a.temperature <= 3.402823466e38f) {
        for (int c0 = threadIdx.x; c0 < whole; c0 += 16 * kExpThreads) {
            u32x4 v[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int c = c0 + i * kExpThreads;
                v[i] = reinterpret_cast<const u32x4*>(a.logits)[c < whole ? c : c0];
            }
#pragma unroll
            for (int i = 0; i < 16; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    m2 = __builtin_elementwise_max(m2, as_h2(v[i][k])); // a NaN loses, as in fmaxf
        }
        m = fmaxf(static_cast<float>(m2[0]), static_cast<float>(m2[1]));
        for (int i = whole * 8 + threadIdx.x; i < a.size; i += kExpThreads)
            m = fmaxf(m, half_bits_to_float(a.logits[i]));
    } else {
        for (int i = threadIdx.x; i < a.size; i += kExpThreads)
            m = fmaxf(m, half_bits_to_float(a.logits[i]) / a.temperature);
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    if (a.temperature <= 3.402823466e38f)
        m = half_bits_to_float(float_to_half_bits(m / a.temperature));
    // two values per thread and turn: thread u of 16 takes chunk i / 8 of its t
    const int u = threadIdx.x >> 4, t = blockIdx.x * kExpShare + u;
#pragma unroll
    for (int j = 0; j < N / 32; ++j) {
        const int i = j * 32 + (threadIdx.x & 15) * 2; // of the thread's N values
        const int at = (t + (i >> 3) * kSampBlock) * 8 + (i & 7);
        uint32_t out = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float v = 0.0f;
            if (at + e < a.size) {
                const float f = half_bits_to_float(float_to_half_bits(half_bits_to_float(a.logits[at + e]) / a.temperature));
                v = expf(f - m);
            }
            val[u][i + e] = v; // 0 where there is no logit: adding it changes no sum
            out |= static_cast<uint32_t>(float_to_half_bits(v)) << (16 * e);
        }
        *reinterpret_cast<uint32_t*>(a.s->exps + at) = out;
    }
    __syncthreads();
    if (threadIdx.x < kExpShare) {
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const float4 v = *reinterpret_cast<const float4*>(&val[threadIdx.x][i]);
            sum += v.x;
            sum += v.y;
            sum += v.z;
            sum += v.w;
        }
        a.s->sums[blockIdx.x * kExpShare + threadIdx.x] = sum;
    }
}

// ---- 2. probabilities, sorted tiles (native/sort_kernel.cu:13-37) ---------------------
// Stable descending order of fp16 keys (sign-flipped bit pattern; +0 before -0).
__device__ __forceinline__ uint32_t sort_rank(uint16_t k) // larger = sorts first
{
    return (k & 0x8000u) ? static_cast<uint32_t>(static_cast<uint16_t>(~k)) : static_cast<uint32_t>(k) | 0x8000u;
}
__device__ __forceinline__ uint16_t sort_key_of_rank(uint32_t rank)
{
    return static_cast<uint16_t>((rank & 0x8000u) ? rank ^ 0x8000u : ~rank);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xF, 0xF, true));
}

template <int MASK>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v)
{
    if constexpr (MASK == 1)
        return dpp_u32<DPP_QUAD_XOR1>(v);
    else if constexpr (MASK == 2)
        return dpp_u32<DPP_QUAD_XOR2>(v);
    else if constexpr (MASK == 3)
        return dpp_u32<DPP_QUAD_XOR3>(v);
    else if constexpr (MASK == 4)
        return dpp_u32<DPP_QUAD_XOR3>(dpp_u32<DPP_ROW_HALF_MIRROR>(v));
    else if constexpr (MASK == 7)
        return dpp_u32<DPP_ROW_HALF_MIRROR>(v);
    else if constexpr (MASK == 8)
        return dpp_u32<DPP_ROW_ROR8>(v);
    else if constexpr (MASK == 15)
        return dpp_u32<DPP_ROW_MIRROR>(v);
    else
        return static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), MASK, 64));
}

constexpr int kTileThreads = kSampTile / 4;

// One stage of a bitonic network over 1024 items, 4 consecutive ones per thread: thread t meets thread t ^ MASK and
// keeps the larger items if it is the lower one of the two.  FLIP: the order inside the four is reversed too (the
// first stage of a merge compares item e with e ^ (2^n - 1), so that all merges run in one direction).
template <int MASK, bool FLIP>
__device__ __forceinline__ void tile_stage(uint32_t (&it)[4], u32x4* lds)
{
    constexpr int kTopBit = MASK >= 128 ? 128 : MASK >= 64 ? 64 : MASK >= 32 ? 32 : MASK >= 16 ? 16 : MASK >= 8 ? 8
                            : MASK >= 4 ? 4 : MASK >= 2 ? 2 : 1;
    const bool lower = (threadIdx.x & kTopBit) == 0;
    uint32_t o[4];
    if constexpr (MASK >= 64) { // another wavefront
        __syncthreads();
        lds[threadIdx.x] = u32x4{it[0], it[1], it[2], it[3]};
        __syncthreads();
        const u32x4 v = lds[threadIdx.x ^ MASK];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            o[r] = v[FLIP ? 3 - r : r];
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            o[r] = lane_xor<MASK>(it[FLIP ? 3 - r : r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t hi = it[r] > o[r] ? it[r] : o[r], lo = it[r] > o[r] ? o[r] : it[r];
        it[r] = lower ? hi : lo;
    }
}

__device__ __forceinline__ void order_two(uint32_t& a, uint32_t& b)
{
    const uint32_t hi = a > b ? a : b, lo = a > b ? b : a;
    a = hi;
    b = lo;
}

__device__ __forceinline__ void tile_finish(uint32_t (&it)[4]) // distances 2 and 1
{
    order_two(it[0], it[2]);
    order_two(it[1], it[3]);
    order_two(it[0], it[1]);
    order_two(it[2], it[3]);
}

template <int HALF> // merges sorted runs of 4 HALF items (HALF threads) into runs twice as long
__device__ __forceinline__ void tile_merge(uint32_t (&it)[4], u32x4* lds)
{
    tile_stage<2 * HALF - 1, true>(it, lds);
    if constexpr (HALF >= 128) tile_stage<64, false>(it, lds);
    if constexpr (HALF >= 64) tile_stage<32, false>(it, lds);
    if constexpr (HALF >= 32) tile_stage<16, false>(it, lds);
    if constexpr (HALF >= 16) tile_stage<8, false>(it, lds);
    if constexpr (HALF >= 8) tile_stage<4, false>(it, lds);
    if constexpr (HALF >= 4) tile_stage<2, false>(it, lds);
    if constexpr (HALF >= 2) tile_stage<1, false>(it, lds);
    tile_finish(it);
}

// Items are distinct numbers (rank << 16) | (0xFFFF - position): the larger one sorts first, equal keys in input order.
__device__ __forceinline__ void sort_tile(uint32_t (&it)[4], u32x4* lds)
{
    order_two(it[0], it[1]);
    order_two(it[2], it[3]);
    order_two(it[0], it[3]);
    order_two(it[1], it[2]);
    order_two(it[0], it[1]);
    order_two(it[2], it[3]);
    tile_merge<1>(it, lds);
    tile_merge<2>(it, lds);
    tile_merge<4>(it, lds);
    tile_merge<8>(it, lds);
    tile_merge<16>(it, lds);
    tile_merge<32>(it, lds);
    tile_merge<64>(it, lds);
    tile_merge<128>(it, lds);
}

// Binade of a non-negative fp16 key: the exponent field for normal numbers, continued downwards
// through the subnormals by the position of the leading mantissa bit (zero: below all of them).
__device__ __forceinline__ int sort_head_binade(uint32_t rank)
{
    const int e = static_cast<int>((rank >> 10) & 31u);
    const uint32_t mant = rank & 0x3FFu;
    return e ? e : (mant ? 22 - __clz(mant) : -10); // mant in [2^k, 2^(k+1)): k - 9
}

// Buckets of the head: how many binades a probability lies below the largest one, 15 for all the rest.
__device__ __forceinline__ int sort_head_bucket(uint32_t rank, int emax)
{
    const int below = emax - sort_head_binade(rank);
    return (rank < 0x8000u || below > 15) ? 15 : below; // negative keys: last bucket
}

enum TileInput {
    TILE_KEYS, // llama2_sort: keys and values as they are
    TILE_EXPS  // the exponentials of sampler_exp_kernel
};

// `plain`, if not null, takes the probabilities in the order of the vocabulary (indices: 0, 1, 2 ...); head < 0: no sort.
template <TileInput IN>
__global__ __launch_bounds__(kTileThreads) void sampler_tile_kernel(SampleArgs a, const uint16_t* keys, const int* values,
                                                                    uint16_t* plain)
{
    __shared__ u32x4 lds[kTileThreads];
    SamplerScratch& s = *a.s;
    if (IN == TILE_EXPS && a.state && !s.go)
        return;
    const int first = blockIdx.x * kSampTile + threadIdx.x * 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint16_t key[4];
    float sum = 0.0f;
    if (IN == TILE_EXPS) {
        const u32x2 e = *reinterpret_cast<const u32x2*>(s.exps + first); // up to the end of the buffer
        float* red = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int w = 0; w < kSampWaves / 4; ++w) {
            const float v = wave_sum(s.sums[(wave + 4 * w) * 64 + lane]);
            if (lane == 0)
                red[wave + 4 * w] = v;
        }
        __syncthreads();
        sum = wave_sum(lane < kSampWaves ? red[lane] : 0.0f);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r)
            key[r] = float_to_half_bits(half_bits_to_float(static_cast<uint16_t>(e[r >> 1] >> (16 * (r & 1)))) / sum);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            key[r] = first + r < a.size ? keys[first + r] : static_cast<uint16_t>(0);
    }
    if (IN == TILE_EXPS) {
        if (plain) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (first + r < a.size) {
                    plain[first + r] = key[r];
                    a.indices[first + r] = first + r;
                }
        }
        if (a.head < 0)
            return;
    }
    if (IN == TILE_EXPS && a.head > 0) {
        // exact mass and number of the items in every bucket of the tile: columns of one lane, no two lanes in a bank
        uint32_t* col = reinterpret_cast<uint32_t*>(lds); // [16][64]
        const uint16_t top = float_to_half_bits(1.0f / sum); // the largest probability: its exponential is 1
        const int emax = sort_head_binade(sort_rank(top));
        if (blockIdx.x == 0 && threadIdx.x == 0)
            s.probabilities = sort_rank(top) >= 0x8000u && sort_rank(top) <= 0xBC00u; // false where the sum is no number
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
            for (int i = 0; i < kSampBuckets * 64 / kTileThreads; ++i)
                col[threadIdx.x + i * kTileThreads] = 0u;
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t rank = sort_rank(key[r]);
                const uint32_t e = (rank >> 10) & 31u, mant = rank & 0x3FFu;
                uint32_t units = e ? (0x400u | mant) << (e - 1) : mant; // value * 2^24, exact
                if (rank < 0x8000u || rank > 0xBC00u)
                    units = 0u;
                if (first + r < a.size)
                    __hip_atomic_fetch_add(&col[sort_head_bucket(rank, emax) * 64 + lane], pass ? 1u : units,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            __syncthreads();
            const u32x4 v = lds[threadIdx.x]; // bucket threadIdx.x / 16
            uint32_t n = v[0] + v[1] + v[2] + v[3];
            n += lane_xor<1>(n);
            n += lane_xor<2>(n);
            n += lane_xor<4>(n);
            n += lane_xor<8>(n);
            if ((threadIdx.x & 15) == 0)
                (pass ? s.count : s.mass)[blockIdx.x][threadIdx.x >> 4] = n;
            __syncthreads();
        }
    }
    uint32_t it[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) // behind the last key: smallest rank, last position
        it[r] = (first + r < a.size ? sort_rank(key[r]) << 16 : 0u) | static_cast<uint32_t>(0xFFFF - (first + r));
    sort_tile(it, lds);
    u32x4 items;
    u32x2 ranks;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        items[r] = it[r] ^ 0xFFFFu;
    ranks[0] = it[0] >> 16 | (it[1] & 0xFFFF0000u);
    ranks[1] = it[2] >> 16 | (it[3] & 0xFFFF0000u);
    *reinterpret_cast<u32x4*>(s.items + first) = items;
    *reinterpret_cast<u32x2*>(s.ranks + first) = ranks;
    if (IN == TILE_KEYS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = static_cast<int>(items[r] & 0xFFFFu);
            if (p < a.size)
                s.payload[first + r] = values[p];
        }
    }
}

// ---- the head of the sorted order ------------------------------------------------------
// The exact masses tell how many buckets it takes to reach top_p with a margin; the length of the head is the
// number of items in them, 0 when there is no such head within 15 binades and half of kSampHeadItems.  Prefix sums are
// rounded to fp16 (2^-11) after a blocked fp32 summation (a few 2^-24): a head whose exact mass is 1.004 top_p reaches
// top_p > coin * top_p in that arithmetic too.  Called by whole wavefronts, the same result in every lane.
struct Head {
    int n, last; // length, last bucket
};

__device__ __forceinline__ Head head_of(const SamplerScratch& s, int size, float top_p)
{
    const int lane = threadIdx.x & 63, tiles = (size + kSampTile - 1) / kSampTile;
    uint32_t mass = 0, count = 0;
    for (int t = lane >> 4; t < tiles; t += 4) { // bucket lane % 16
        mass += s.mass[t][lane & 15];
        count += s.count[t][lane & 15];
    }
    mass += lane_xor<16>(mass);
    mass += lane_xor<32>(mass);
    count += lane_xor<16>(count);
    count += lane_xor<32>(count);
    const float need = ceilf(top_p * 1.004f * 16777216.0f);
    float cum = 0.0f; // sums of integers below 2^25 in fp32 lose at most a unit or two: `need` carries a margin
    Head h{0, 0};
    bool found = false;
#pragma unroll
    for (int d = 0; d < kSampBuckets - 1; ++d) {
        cum += static_cast<float>(__builtin_amdgcn_readlane(static_cast<int>(mass), d));
        if (!found) {
            h.n += __builtin_amdgcn_readlane(static_cast<int>(count), d);
            h.last = d;
        }
        found |= cum >= need;
    }
    if (!s.probabilities || !found || h.n > kSampHeadItems / 2)
        h.n = 0;
    return h;
}

// ---- 3. places -------------------------------------------------------------------------
// The place of an item is its place in its own tile plus, for every other tile, the number of items there that sort
// in front of it (equal keys: those of the tiles before it): a binary search in the ranks, which all lie in LDS.  A
// workgroup places 128 neighbours of a sorted tile (neighbours take similar ways through the other tiles and meet
// in the same words), 8 threads share an item's searches.  128 KB of LDS at 65536 items, 64 KB at 32000.
template <int TILES>
__global__ __launch_bounds__(kSampBlock) void sampler_rank_kernel(SampleArgs a, uint16_t* keys, int* values, int identity)
{
    __shared__ __align__(16) uint16_t ranks[TILES * kSampTile];
    __shared__ int parts[8][kSampRun];
    const SamplerScratch& s = *a.s;
    if (a.state && !s.go)
        return;
    const int tiles = (a.size + kSampTile - 1) / kSampTile;
    const int i = threadIdx.x & (kSampRun - 1), sub = threadIdx.x / kSampRun;
    const int at = blockIdx.x * kSampRun + i, own = blockIdx.x * kSampRun / kSampTile;
    const uint32_t item = s.items[at];
    const uint32_t rank = item >> 16;
    int limit = a.size; // places beyond it are nobody's
    if (a.head > 0) {
        const Head h = head_of(s, a.size, a.top_p);
        if (h.n) {
            limit = h.n;
            int mine = 0; // items of this tile in the head: they are the first of it
            for (int d = 0; d <= h.last; ++d)
                mine += static_cast<int>(s.count[own][d]);
            if (static_cast<int>(blockIdx.x) * kSampRun - own * kSampTile >= mine)
                return;
        }
    }
    const u32x4* from = reinterpret_cast<const u32x4*>(s.ranks);
    u32x4* to = reinterpret_cast<u32x4*>(ranks);
    for (int p = threadIdx.x; p < tiles * (kSampTile / 8); p += kSampBlock)
        to[p] = from[p];
    __syncthreads();
    int before = 0;
    for (int t0 = sub; t0 < tiles; t0 += 32) { // four searches at a time: each is a chain of LDS reads
        const uint16_t* r[4];
        uint32_t least[4]; // smallest rank that sorts in front
        int n[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = t0 + u * 8;
            r[u] = ranks + (t < tiles ? t : own) * kSampTile;
            least[u] = t >= tiles || t == own ? 0x10000u : t < own ? rank : rank + 1;
            n[u] = 0;
        }
#pragma unroll
        for (int step = kSampTile / 2; step > 0; step >>= 1)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                n[u] += r[u][n[u] + step - 1] >= least[u] ? step : 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            before += n[u] + (r[u][n[u]] >= least[u] ? 1 : 0);
    }
    parts[sub][i] = before;
    __syncthreads();
    if (sub)
        return;
    int place = at % kSampTile;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        place += parts[k][i];
    const int position = static_cast<int>(item & 0xFFFFu);
    if (position >= a.size || place >= limit)
        return;
    keys[place] = sort_key_of_rank(rank);
    values[place] = identity ? position : s.payload[at];
}

// ---- 4. prefix sums and the pick -------------------------------------------------------
// native/cumulative_sum_kernel.cu:8-26: inclusive prefix sums in fp32, each rounded to fp16.  A thread sums its
// 8 CH consecutive values in order, the thread totals are scanned by doubling within a wavefront and in order over the
// wavefronts.  `piece(p)` gives the 16-byte piece p of the values; all = false: the sums of wavefront blockIdx.x alone are
// stored.  PICK, native/sample_top_p_kernel.cu:8-21: returns a thread's first position whose sum reaches the threshold,
// or the last position.
template <int CH, bool PICK, class F>
__device__ __forceinline__ int prefix_sums(const F& piece, int size, float threshold, bool all, uint16_t* out, float* total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first = threadIdx.x * 8 * CH;
    int best = size - 1;
    float f[CH][8];
    float run = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int p = threadIdx.x * CH + c;
        if (p * 8 < size) {
            const u32x4 v = piece(p);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                run += half_of(v, k);
                f[c][k] = run;
            }
        }
    }
    float inc = run;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float o = __shfl_up(inc, off, 64);
        if (lane >= off)
            inc += o;
    }
    if (lane == 63)
        total[wave] = inc;
    __syncthreads();
    float before = 0.0f; // total of the wavefronts in front of this one
#pragma unroll
    for (int w = 0; w < kSampWaves; ++w)
        before += w < wave ? total[w] : 0.0f;
    before = before + inc - run;
    // Probabilities are not negative (or all of them are NaN): a thread whose last sum does not reach the threshold
    // has none that does, so only those that have one look for the first.
    const bool hit = PICK && blockIdx.x == 0 && first < size &&
                     half_bits_to_float(float_to_half_bits(before + run)) >= threshold;
    const bool mine = all || wave == static_cast<int>(blockIdx.x);
    if (mine || hit) {
#pragma unroll
        for (int c = CH - 1; c >= 0; --c) {
            const int base = first + c * 8;
            if (base < size) {
                uint16_t b[8];
#pragma unroll
                for (int k = 7; k >= 0; --k) {
                    b[k] = float_to_half_bits(before + f[c][k]);
                    if (hit && base + k < size && half_bits_to_float(b[k]) >= threshold)
                        best = base + k;
                }
                if (mine)
                    store_half8(out, base, size, b);
            }
        }
    }
    return best;
}

// The lowest of the threads' positions; where its token goes.  go = false: a decode step that draws none.
__device__ __forceinline__ void finish_pick(const SampleArgs& a, int best, bool go, int* first_hit)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(best, off, 64);
        best = o < best ? o : best;
    }
    if ((threadIdx.x & 63) == 0)
        first_hit[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x != 0)
        return;
    for (int w = 1; w < kSampWaves; ++w)
        best = first_hit[w] < best ? first_hit[w] : best;
    if (!a.state) {
        const int token = a.indices[best];
        a.result[a.pos] = token;
        write_host_token(a.host, token);
        return;
    }
    const int next = a.state[kStatePos] + 1;
    if (go)
        a.tokens[next] = a.indices[best];
    if (a.state[kStateAdvance])
        a.state[kStatePos] = next;
}

// Every workgroup scans everything (64 KB from the L2) and stores the share of wavefront blockIdx.x, so that nothing has
// to be handed from one to the other; in a launch of one workgroup it stores everything and may work in place.  The
// first workgroup picks.
template <int CH, bool PICK>
__global__ __launch_bounds__(kSampBlock) void sampler_pick_kernel(SampleArgs a, const uint16_t* in)
{
    constexpr bool kStaged = PICK || CH > 4;
    __shared__ u32x4 chunk[CH * kSampBlock];
    __shared__ float total[kSampWaves];
    __shared__ int first_hit[kSampWaves];
    int size = a.size;
    float threshold = a.coin;
    bool go = true;
    if (PICK) {
        const SamplerScratch& s = *a.s;
        if (a.state) {
            go = s.go != 0;
            threshold = s.coin;
        }
        if (a.head >= 0)
            threshold *= a.top_p;
        if (a.head > 0 && go) {
            const Head h = head_of(s, a.size, a.top_p);
            size = h.n ? h.n : size;
        }
    }
    int best = size - 1;
    if (go) {
        // 16-byte pieces come in the order of memory; piece p lies at p ^ (p / 16 % CH), where the 16 threads that LDS
        // serves at a time find theirs, CH apart, in 16 different places.  Without a pick there is one workgroup, and up to
        // 32768 values its threads load their own pieces: 32000 values take 4.56 us, through LDS and its barrier 5.00 (1000:
        // 2.54 and 2.62).  65536 values take 9.4 us like that, for a thread's 8 pieces are 128 bytes apart from the next
        // one's, and 8.5 through LDS.
        if (kStaged) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int p = threadIdx.x + c * kSampBlock;
                if (p * 8 < size)
                    chunk[p ^ ((p >> 4) & (CH - 1))] = load_bits8(in, p * 8, size, 0);
            }
            __syncthreads();
        }
        best = prefix_sums<CH, PICK>(
            [&](int p) { return kStaged ? chunk[p ^ ((p >> 4) & (CH - 1))] : load_bits8(in, p * 8, size, 0); }, size,
            threshold, gridDim.x == 1, a.logits, total);
    }
    if (PICK && blockIdx.x == 0)
        finish_pick(a, best, go, first_hit);
}

// ---- 1, 2 and 4 in one workgroup ---------------------------------------------------------
// Without a sort the launches of the others cost more than one compute unit alone takes for a short vector: the
// probabilities of 1000 / 5000 / 8192 / 11264 logits take 5.8 / 6.6 / 6.7 / 6.5 us in two launches of many workgroups and
// 2.7 / 4.1 / 4.9 / 6.2 here, with the pick (and 2.5 us for the copy of the logits) 11.1 / 12.6 / 12.7 / 13.2 in three and 6.6 /
// 8.1 / 8.9 / 11.0 here.  Every 2048 logits more are another wavefront with a second piece on each SIMD and 0.5 us.
constexpr int kSampOneItems = 11 * 1024;

template <int PIECES, bool PICK> // PIECES: of 8 logits per thread
__global__ __launch_bounds__(kSampBlock) void sampler_one_kernel(SampleArgs a)
{
    constexpr int CH = 4; // pieces per thread of the prefix sums
    __shared__ u32x4 chunk[PICK ? PIECES * kSampBlock : 1];
    __shared__ float red[3][kSampWaves];
    __shared__ int first_hit[kSampWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float threshold = a.coin;
    bool go = true;
    if (PICK && a.state) { // read by every thread before the first one changes it, behind the barrier of finish_pick
        const int next = a.state[kStatePos] + 1;
        go = next >= a.state[kStatePrompt] && next < a.state[kStateSlots];
        threshold = sampler_coin(a.seed, next);
        if (a.state[kStateAdvance] && threadIdx.x >= 64 && threadIdx.x < 64 + kRopeHeadSize / 2)
            write_rope_table(a.state, threadIdx.x - 64, next, a.theta); // for the next step
    } else if (PICK && threadIdx.x >= 64) {
        write_host_step_state(a.host, threadIdx.x - 64);
    }
    int best = a.size - 1;
    if (go) {
        float f[PIECES][8];
        uint16_t b[PIECES][8];
        float m = -INFINITY;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
            const int base = (threadIdx.x + c * kSampBlock) * 8;
            if (base < a.size) {
                const u32x4 v = load_bits8(a.logits, base, a.size, 0xFC00u);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    f[c][k] = half_bits_to_float(float_to_half_bits(half_of(v, k) / a.temperature));
                    m = base + k < a.size ? fmaxf(m, f[c][k]) : m;
                }
            }
        }
        m = wave_max(m);
        if (lane == 0)
            red[0][wave] = m;
        __syncthreads();
        m = row16_max(red[0][lane & 15]);
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
            const int base = (threadIdx.x + c * kSampBlock) * 8;
            if (base < a.size) {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float e = base + k < a.size ? expf(f[c][k] - m) : 0.0f;
                    sum += e;
                    b[c][k] = float_to_half_bits(e);
                }
            }
        }
        sum = wave_sum(sum);
        if (lane == 0)
            red[1][wave] = sum;
        __syncthreads();
        sum = wave_sum(lane < kSampWaves ? red[1][lane] : 0.0f);
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
            const int p = threadIdx.x + c * kSampBlock, base = p * 8;
            if (base < a.size) {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    b[c][k] = float_to_half_bits(half_bits_to_float(b[c][k]) / sum);
                if (PICK) {
                    u32x4 v;
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        v[k] = b[c][2 * k] | static_cast<uint32_t>(b[c][2 * k + 1]) << 16;
                    chunk[p ^ ((p >> 4) & (CH - 1))] = v;
                } else {
                    store_half8(a.logits, base, a.size, b[c]);
                }
                if (base + 8 <= a.size) {
                    u32x4* to = reinterpret_cast<u32x4*>(a.indices + base);
                    const uint32_t i = base;
                    to[0] = u32x4{i, i + 1, i + 2, i + 3};
                    to[1] = u32x4{i + 4, i + 5, i + 6, i + 7};
                } else {
                    for (int i = base; i < a.size; ++i)
                        a.indices[i] = i;
                }
            }
        }
        if (PICK) {
            __syncthreads();
            best = prefix_sums<CH, true>([&](int p) { return chunk[p ^ ((p >> 4) & (CH - 1))]; }, a.size, threshold, true,
                                         a.logits, red[2]);
        }
    }
    if (PICK)
        finish_pick(a, best, go, first_hit);
}

// The pick alone, on any values.
template <int CH>
__global__ __launch_bounds__(kSampBlock) void sample_top_p_kernel(const uint16_t* logits, const int* indices, int size,
                                                                  float threshold, int* result, int pos)
{
    __shared__ int first_hit[kSampWaves];
    int best = size - 1;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int base = (threadIdx.x + c * kSampBlock) * 8;
        if (base < size) {
            const u32x4 v = load_bits8(logits, base, size, 0xFC00u);
#pragma unroll
            for (int k = 7; k >= 0; --k)
                if (base + k < size && half_of(v, k) >= threshold && base + k < best)
                    best = base + k;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_xor(best, off, 64);
        best = o < best ? o : best;
    }
    if ((threadIdx.x & 63) == 0)
        first_hit[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kSampWaves; ++w)
            best = first_hit[w] < best ? first_hit[w] : best;
        result[pos] = indices[best];
    }
}

#endif // __HIPCC__

} // namespace l2
