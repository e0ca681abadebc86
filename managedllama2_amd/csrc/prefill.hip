// The layers of Transformer.Forward (src/Transformer.cs:158-183) for many known tokens at once.
//
// A prompt's tokens are all there before the first step, and only their key and value rows matter to
// what follows (the step of the last prompt token, which produces the first logits anyone reads, is an
// ordinary decode step).  Taken one by one each token reads all the weights, 3.6 GB for Llama-2-7B; here up
// to kPrefillMaxRows tokens share one reading and the matrix products run on the matrix cores:
//   norm (+ embedding) | QKV + RoPE + cache rows | causal attention | o-proj + residual | norm |
//   SwiGLU | down-proj + residual: 7 launches per layer and batch, 8 where attention is split.
//
// Arithmetic, module by module as in the decode step: fp16 between the modules, exact integer weights
// (n - z) in fp16, fp32 sums of their products with the fp16 inputs over a quantisation group of 128,
// the group's scale applied in fp32, fp32 sums over the groups; scores rounded to fp16, softmax
// statistics in fp32, probabilities with all the bits of fp32.  The order of the sums is not that of the decode step.
//
// Measured, Llama-2-7B: 512 prompt tokens one by one 560 ms, 511 in one batch and the last as a step 10.7 ms;
// 13B, 74 tokens behind 600 rows: 151 -> 7 ms.
#include "int4_kernels.hpp"
#include "gemm_shape.hpp"
#include "prefill.hpp"

#include <cmath>
#include <cstdlib>
#include <type_traits>
#include <utility>

namespace l2 {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f16v_t __attribute__((ext_vector_type(16)));

constexpr int kGroup = 128;       // quantisation group along K
constexpr int kFragBytes = 1024;  // one operand fragment: 64 lanes of 16 bytes
constexpr int kBlockBytes = 8 * kFragBytes; // a token tile times a group

// Fragment order of an activation matrix [m][k]: the lane (k / 64 % 2) * 32 + m % 32 of fragment
// (m / 32, k / 128, k / 8 % 8) holds 8 consecutive k, in the order in which the weights' nibbles come out of
// a word (0 4 1 5 2 6 3 7).  The word of weights that goes with them is word k / 8 of its row, so a lane's 8
// words of a group are 32 contiguous bytes, and every fragment is one fully coalesced load.
__device__ __forceinline__ uint32_t frag_offset(int m, int k, int groups)
{
    return static_cast<uint32_t>(((m >> 5) * groups + (k >> 7)) * 8 + ((k >> 3) & 7)) * kFragBytes +
           ((((k >> 6) & 1) << 5) + (m & 31)) * 16;
}

__device__ __forceinline__ u32x4 frag_order(u32x4 v) // 8 consecutive values -> 0 4 1 5 2 6 3 7
{
    u32x4 o;
    o[0] = (v[0] & 0xFFFFu) | (v[2] << 16);
    o[1] = (v[0] >> 16) | (v[2] & 0xFFFF0000u);
    o[2] = (v[1] & 0xFFFFu) | (v[3] << 16);
    o[3] = (v[1] >> 16) | (v[3] & 0xFFFF0000u);
    return o;
}

// ---------------------------------------------------------------- RoPE angles
__global__ __launch_bounds__(256) void prefill_rope_kernel(float* tab, int position, int count, float theta)
{
    const int i = blockIdx.x * 256 + threadIdx.x, row = i >> 6;
    if (row >= count)
        return;
    float c, s;
    rope_cos_sin(c, s, i & 63, kRopeHeadSize, position + row, theta);
    tab[2 * i] = c;
    tab[2 * i + 1] = s;
}

// ---------------------------------------------------------------- RMSNorm into fragment order
struct NormArgs {
    uint16_t* x; // [rows][K]
    const uint16_t* gamma;
    uint16_t* xf;
    const uint16_t* embedding; // non-null: the row comes from the table and is also written to x
    const int* tokens;         // of the first row
    const float* parts; // non-null: x += the sum of n_parts fp32 results [part][part_rows][K] of the product before
    int n_parts, part_rows;
    int vocab, K;
    float eps;
};

// One row per workgroup of 256 threads; the same sums as the decode step's RMSNorm (block256_sum).  The
// residual product before it leaves fp32 sums over pieces of K; they are added here, in order, and
// rounded to fp16 once, so that product can be split over as many workgroups as the GPU holds.
template <int PIECES>
__global__ __launch_bounds__(256) void prefill_norm_kernel(NormArgs a)
{
    __shared__ float red4[4];
    const int m = blockIdx.x;
    uint16_t* row = a.x + static_cast<size_t>(m) * a.K;
    const uint16_t* src = row;
    if (a.embedding) {
        int token = a.tokens[m];
        token = token < 0 ? 0 : (token >= a.vocab ? a.vocab - 1 : token); // never read outside the table
        src = a.embedding + static_cast<size_t>(token) * a.K;
    }
    VecPieces<PIECES> p, g;
    p.load(src, a.K);
    g.load(a.gamma, a.K);
    if (a.parts) {
        // Four pieces are requested together: one after the other each waited for the one before (511 rows, four
        // pieces: 10.5 us, together 9.8; 74 rows of 13B with six 7.2 and 6.0).
        constexpr int kTogether = 4;
        float sum[PIECES][8] = {};
        for (int t0 = 0; t0 < a.n_parts; t0 += kTogether) {
            u32x4 q[kTogether][PIECES][2];
#pragma unroll
            for (int u = 0; u < kTogether; ++u) {
                // behind the last piece a buffer of no length, which reads as zero and moves no data
                const bool have = t0 + u < a.n_parts;
                const __amdgpu_buffer_rsrc_t r =
                    make_rsrc(a.parts + (static_cast<size_t>(have ? t0 + u : 0) * a.part_rows + m) * a.K, have ? a.K * 4 : 0);
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        q[u][i][e] = __builtin_amdgcn_raw_buffer_load_b128(r, (threadIdx.x + i * 256) * 32 + e * 16, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < kTogether; ++u)
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        sum[i][e] += __uint_as_float(q[u][i][e >> 2][e & 3]);
        }
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const h2_t x = as_h2(p.v[i][e]);
                p.v[i][e] = static_cast<uint32_t>(float_to_half_bits(sum[i][2 * e] + static_cast<float>(x[0]))) |
                            static_cast<uint32_t>(float_to_half_bits(sum[i][2 * e + 1] + static_cast<float>(x[1]))) << 16;
            }
    }
    if (a.embedding || a.parts) {
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(row, a.K * 2);
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
            __builtin_amdgcn_raw_buffer_store_b128(p.v[i], ro, (threadIdx.x + i * 256) * 16, 0, 0);
    }
    const float ss = block256_sum(p.sum_squares(), red4);
    p.scale(1.0f / sqrtf(ss / static_cast<float>(a.K) + a.eps), g);
    const int groups = a.K / kGroup;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        const int k = (threadIdx.x + i * 256) * 8;
        if (k < a.K)
            *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(a.xf) + frag_offset(m, k, groups)) = frag_order(p.v[i]);
    }
}

// ---------------------------------------------------------------- int4 matrix product
enum PrefillEpi { EPI_QKV, EPI_PARTIAL, EPI_SWIGLU };

struct GemmArgs {
    QW m[3];
    const uint16_t* xf;
    uint32_t xf_bytes;
    int groups, N, ws, ss, zs; // N: rows of one tensor
    int M, mblocks, pairs, nblocks, splits; // pairs of weight tiles, and blocks of them
    int first, mblocks2; // blocks of weights of one XCD that meet blocks of MT token tiles (the rest: MT2), and blocks of MT2
    uint16_t* out[3]; // QKV: q, key-cache rows, value-cache rows of this batch; SWIGLU: hf
    float* parts;     // PARTIAL: [splits][part_rows][N]
    int part_rows;
    int out_groups; // SWIGLU: groups of hf
    const float* rope;
};

// Pair k of the 8 nibbles of a word as fp16 n - z, exact: n sits in the mantissa of 1024 + n (bits 0-3 of a half) or
// 1024 + 16 n (bits 4-7).
__device__ __forceinline__ uint32_t dequant_pair(uint32_t w, int k, h2_t zlo /* 1024 + z */, h2_t zhi /* -(64 + z) */)
{
    const h2_t sixteenth = {static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
    uint32_t magic = 0x64006400u; // in a vector register: (w & mask) | magic is one instruction then
    asm("" : "+v"(magic));
    const uint32_t v = k >= 2 ? w >> 8 : w;
    return k & 1 ? as_u32(__builtin_elementwise_fma(as_h2((v & 0x00F000F0u) | magic), sixteenth, zhi))
                 : as_u32(as_h2((v & 0x000F000Fu) | magic) - zlo);
}

__device__ __forceinline__ f16v_t mfma(h8_t a, h8_t b, f16v_t c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// 64 lanes x 16 bytes from a buffer straight into LDS at `lds` + 16 lane (`lds`, `soff` uniform).  Written
// as assembly because the compiler, told that LDS is written, waits for it before any later LDS read,
// also of the other half of a ring; there is no destination register, and the caller waits (vmcnt)
// before the barrier that publishes the data.  The LDS address travels in M0, which the compiler writes in
// front of the assembly; a load that reads M0 needs one wait state after that write, and the compiler
// does not know that this is such a load: hence the s_nop (7B, 512 known tokens: 11.16 ms without, 11.11 with).
__device__ __forceinline__ void load_to_lds(u32x4 rsrc, uint32_t lds, int voff, int soff)
{
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "{m0}"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

// The same from an address per lane, 4 bytes to `lds` + 4 lane.
__device__ __forceinline__ void load_to_lds_x1(const void* p, uint32_t lds)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %1, off" : : "{m0}"(lds), "v"(p) : "memory");
}

// s_waitcnt vmcnt(n), the other counters free
constexpr int wait_vm(int n) { return 0x0F70 | (n & 15) | (n >> 4) << 14; }

template <typename F, int... I>
__device__ __forceinline__ void static_for(const F& f, std::integer_sequence<int, I...>) // f(0), f(1) ... with constant indices
{
    (f(std::integral_constant<int, I>{}), ...);
}

// A workgroup owns MT token tiles and WN pairs of weight tiles of 32 rows; the two tiles of a pair hold
// results that belong together (the two halves of a RoPE pair, gate and up, or neighbours).  8 wavefronts: one per
// weight tile and group, a step covers WK consecutive groups of K.  At the end the WK sums add up, and the tiles
// of a pair meet, through LDS.  The launch may split K further (EPI_PARTIAL).
//
// What bounds it: a step of four tiles is 1024 cycles of matrix products per wavefront, two wavefronts to a SIMD, and takes
// 2990, so that the matrix cores wait 940 of them (the barrier, LDS, vector work that no product covers); and the clock, which
// their power brings from 2.4 down to 1.6 .. 2.0 GHz (a loop of nothing but these products on random numbers, with
// their LDS reads, runs at 1.8 and reaches 1.65 PFLOP/s).  7B, 511 rows, QKV: 1.08 PFLOP/s over the steps; a library product of
// 8192^3 reaches 1.14.  Around the steps there are 3.5 us to the first and 4 us behind the last one, and rounds of
// workgroups that do not fill the card.  So the vector work and the loads stay out of the way:
// - Vector work runs beside the matrix products only where it stands between them (5 instructions for one product
//   of 32 cycles cost nothing, 8 cost 12 cycles); left to the compiler the unpacking and the scaled sums came after the
//   products of their step, 5000 cycles for four tiles.
// - A compute unit looks up one cache address per cycle and 64 contiguous bytes.  A lane that reads its own row's
//   weights costs 64 lookups per load (13.2 ms instead of 11.9 for the 512-token prompt).  Everything
//   comes through LDS, requested in the order of memory; LDS delivers 256 bytes per cycle where 16 neighbouring
//   lanes meet all banks, hence the swizzle of the weight rows.
// - One barrier per step, LDS for three: activations are requested two steps ahead, weights three, because
//   they are unpacked into registers a step ahead.
// - Results leave in pieces of 16 bytes after one exchange of all tiles through LDS, their RoPE angles requested
//   before it: stored as they lie in the registers, 2 bytes per lane and tile by tile, they took 25 us of the 72 of QKV.
// 7B, 511 rows: QKV 76 -> 62 us; the whole 512-token prompt 11.25 -> 10.75 ms.
template <int MT, int WN, int WK>
struct GemmLds {
    static constexpr int kXStage = WK * MT * kBlockBytes;  // activations of a step
    static constexpr int kWRow = WK * 64;                  // bytes of a weight row per step
    static constexpr int kWStage = WN * 2 * kTile * kWRow; // weights of a step
    static constexpr int kZStage = 8 * 256;                // a word with the scale and one with the zero point per row and group
    static constexpr int kWAt = 3 * kXStage, kZAt = kWAt + 3 * kWStage, kAll = kZAt + 3 * kZStage;
    static constexpr int kRedRow = kTile + 4, kRed = 8 * MT * kTile * kRedRow * 4;
    static constexpr int kBytes = kAll > kRed ? kAll : kRed;
    static_assert(kBytes <= 160 * 1024, "LDS of a compute unit");
};

// Block `unit` of weights (and piece of K) with block `mb` of MT token tiles.
template <int MT, int WN, int WK, int EPI>
__device__ __forceinline__ void gemm_block(const GemmArgs& a, char* lds, int unit, int mb)
{
    static_assert(WN * WK == 4, "8 wavefronts");
    using Lds = GemmLds<MT, WN, WK>;
    constexpr int kXStage = Lds::kXStage, kWRow = Lds::kWRow, kWStage = Lds::kWStage, kZStage = Lds::kZStage;
    constexpr int kWAt = Lds::kWAt, kZAt = Lds::kZAt, kRedRow = Lds::kRedRow;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = wave & 1, wn = (wave >> 1) % WN, wk = (wave >> 1) / WN;
    const int h = lane >> 5, l31 = lane & 31;
    const int nb = unit / a.splits, split = unit - nb * a.splits;
    // tensor and first row of a tile; the last block may have pairs to spare, which repeat the last one
    auto tile_of = [&](int pair, int tile, int& tensor, int& row) {
        pair = pair < a.pairs ? pair : a.pairs - 1;
        if (EPI == EPI_QKV) {
            const int per = a.N >> 6, r = pair % per;
            tensor = pair / per;
            row = (r >> 1) * kRopeHeadSize + (r & 1) * kTile + tile * 64;
        } else if (EPI == EPI_SWIGLU) {
            tensor = tile;
            row = pair * kTile;
        } else {
            tensor = 0;
            row = (pair * 2 + tile) * kTile;
        }
    };
    // by value: a choice among the arguments themselves puts them into scratch memory
    auto choose = [](int i, auto first, auto second, auto third) { return i == 0 ? first : (i == 1 ? second : third); };
    auto tensor_of = [&](int i) {
        return QW{choose(i, a.m[0].w, a.m[1].w, a.m[2].w), choose(i, a.m[0].z, a.m[1].z, a.m[2].z),
                  choose(i, a.m[0].s, a.m[1].s, a.m[2].s)};
    };
    auto rsrc_of = [](const void* p, uint32_t bytes) {
        const unsigned long long v = reinterpret_cast<unsigned long long>(p);
        return u32x4{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v))),
                     static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32))), bytes, 0x00020000u};
    };
    const int mt0 = mb * MT, last_tile = (a.M - 1) / kTile;
    const int g_begin = a.groups * split / a.splits, g_end = a.groups * (split + 1) / a.splits;
    const int steps = (g_end - g_begin + WK - 1) / WK;
    // what does not exist is loaded as the last one that does, and not used
    auto base_of = [&](int step) { return g_begin + (step < steps ? step : steps - 1) * WK; };
    auto group_of = [&](int step) {
        const int g = g_begin + step * WK + wk;
        return g < g_end ? g : g_end - 1;
    };
    const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
        static_cast<int>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)));

    // Activations: the fragments of this wavefront's group are shared by its 2 WN wavefronts.
    const u32x4 rx = rsrc_of(a.xf, a.xf_bytes);
    constexpr int kXPer = 8 / (2 * WN);
    auto load_x = [&](int step, int at) {
        const int g = group_of(step);
        const uint32_t dst = lds_base + at * kXStage + wk * MT * kBlockBytes;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int tile = mt0 + mt <= last_tile ? mt0 + mt : last_tile; // the last block may have tiles to spare
#pragma unroll
            for (int j = 0; j < kXPer; ++j) {
                const int f = (wave % (2 * WN)) * kXPer + j;
                load_to_lds(rx, dst + mt * kBlockBytes + f * kFragBytes, lane * 16,
                            (tile * a.groups + g) * kBlockBytes + f * kFragBytes);
            }
        }
    };
    // Weights: this wavefront fetches 2 KB of the step, RPI rows per load.  Piece c of 16 bytes of row r lies in
    // place c ^ swizzle(r) of the row: 16 neighbouring rows put the same piece into 16 different 16-byte columns.
    // Reads past the end of a tensor return 0; those past the end of a row (K not a multiple of 128) meet
    // zeros of the input.
    constexpr int LPR = WK * 4, RPI = 64 / LPR;
    auto swizzle = [](int r) { return (r / (256 / kWRow)) & (LPR - 1); };
    const int wr0 = wave * 2 * RPI; // first row of the block this wavefront fetches
    int wt, wrow;
    tile_of(nb * WN + wr0 / 64, (wr0 / kTile) & 1, wt, wrow);
    wrow += wr0 & (kTile - 1);
    const u32x4 rw = rsrc_of(tensor_of(wt).w, static_cast<uint32_t>(a.N) * a.ws * 4);
    int wvoff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = i * RPI + lane / LPR, row = wrow + r < a.N ? wrow + r : a.N - 1;
        wvoff[i] = row * a.ws * 4 + ((lane % LPR) ^ swizzle(wr0 + r)) * 16;
    }
    // Scales and zero points of this wavefront's tile and group, by the two halves of the lanes.  Scales need not be
    // aligned to more than their 2 bytes: the word that holds one is fetched.
    int tensor, r0;
    tile_of(nb * WN + wn, t, tensor, r0);
    const int row = r0 + l31 < a.N ? r0 + l31 : a.N - 1;
    const QW q = tensor_of(tensor);
    const int s_odd = static_cast<int>(reinterpret_cast<uintptr_t>(q.s) & 2) + row * a.ss * 2; // from the first word
    const char* zs_base = h ? reinterpret_cast<const char*>(q.z + static_cast<size_t>(row) * a.zs)
                            : reinterpret_cast<const char*>(reinterpret_cast<uintptr_t>(q.s) & ~static_cast<uintptr_t>(2));
    auto load_w = [&](int step, int at) {
        const int gb = base_of(step), g = group_of(step);
        const uint32_t dst = lds_base + kWAt + at * kWStage + wr0 * kWRow;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            load_to_lds(rw, dst + i * kFragBytes, wvoff[i], gb * 64);
        load_to_lds_x1(zs_base + (h ? (g >> 3) * 4 : (s_odd + 2 * g) & ~3), lds_base + kZAt + at * kZStage + wave * 256);
    };

    // The products of a step are one sequence, tile by tile and fragment by fragment; every product is a slot that also
    // holds a share of the vector work, pinned there by scheduling fences: the activations of three slots later, the
    // next step's weights, and the scaled sum of the tile before (whose last product needs two slots to finish).
    constexpr int N = MT * 8, kAhead = 3, kRing = kAhead + 1, kFirstPair = 3;
    f16v_t acc[MT], p[2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
        acc[mt] = f16v_t{};
    p[0] = p[1] = f16v_t{};
    u32x4 raw[2];
    u32x4 wf[2][8]; // weights of this step's group and of the next one's, n - z in fp16
    h2_t zlo, zhi;
    float sc = 0.0f, sc_next = 0.0f, sc_pending = 0.0f; // scales of this group, the next, and of the sums still in p
    uint32_t zword;
    uint16_t sbits;
    auto read_w = [&](int step, int at) { // what it reads is used later than the slots before
        const int r = (wn * 2 + t) * kTile + l31, g = group_of(step);
        const char* from = lds + kWAt + at * kWStage + r * kWRow;
        const char* sz = lds + kZAt + at * kZStage + wave * 256 + l31 * 4;
        sbits = *reinterpret_cast<const uint16_t*>(sz + ((s_odd + 2 * g) & 2));
        zword = *reinterpret_cast<const uint32_t*>(sz + 128);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            raw[i] = *reinterpret_cast<const u32x4*>(from + ((wk * 4 + h * 2 + i) ^ swizzle(r)) * 16);
    };
    auto unpack_sz = [&](int step) {
        sc_next = half_bits_to_float(sbits);
        asm("" : "+v"(sc_next)); // a float from here on: the multiply-adds take it as one
        const float z = static_cast<float>((zword >> ((group_of(step) & 7) * 4)) & 0xFu);
        const _Float16 lo = static_cast<_Float16>(1024.0f + z), hi = static_cast<_Float16>(-64.0f - z);
        zlo = h2_t{lo, lo}, zhi = h2_t{hi, hi};
    };
    constexpr int kLoads = MT * kXPer + 3; // of a step
    auto wait_all_but = [](auto n) {
        __builtin_amdgcn_s_waitcnt(wait_vm(decltype(n)::value));
        asm volatile("" ::: "memory");
    };
    load_w(0, 0);
    load_x(0, 0);
    load_w(1, 1);
    load_x(1, 1);
    load_w(2, 2);
    wait_all_but(std::integral_constant<int, 2 * kLoads>{});
    __syncthreads();
    read_w(0, 0);
    unpack_sz(0);
#pragma unroll
    for (int k = 0; k < 32; ++k)
        wf[0][k >> 2][k & 3] = dequant_pair(raw[k >> 4][(k >> 2) & 3], k & 3, zlo, zhi);
    int s0 = 0, s1 = 1, s2 = 2; // LDS of this step, the next and the one after it
    auto flush = [&](int tile, int sum, int from, int to) { // results from .. to - 1 of p[sum] into a tile's sums
#pragma unroll
        for (int i = from; i < to; ++i)
            acc[tile][i] = __builtin_fmaf(p[sum][i], sc_pending, acc[tile][i]);
    };
    auto body = [&](auto parity, int step) {
        constexpr int P = decltype(parity)::value;
        constexpr int kFirst = P * MT & 1; // the sums' register of the first tile; the other one holds the last tile before
        // this step's activations and the next one's weights; every wavefront is through with the step before
        wait_all_but(std::integral_constant<int, kLoads>{});
        __syncthreads();
        const char* xs = lds + s0 * kXStage + wk * MT * kBlockBytes + lane * 16;
        h8_t xa[kRing];
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
            xa[i] = *reinterpret_cast<const h8_t*>(xs + (i >> 3) * kBlockBytes + (i & 7) * kFragBytes);
        read_w(step + 1, s1);
        load_x(step + 2, s2);
        load_w(step + 3, s0);
        sc = sc_next;
        if (WK == 1 || g_begin + step * WK + wk < g_end) {
            static_for([&](auto slot) {
                constexpr int i = decltype(slot)::value, mt = i >> 3, j = i & 7;
                if constexpr (i + kAhead < N) {
                    constexpr int n = i + kAhead;
                    xa[n % kRing] = *reinterpret_cast<const h8_t*>(xs + (n >> 3) * kBlockBytes + (n & 7) * kFragBytes);
                }
                f16v_t& q = p[(kFirst + mt) & 1];
                q = mfma(xa[i % kRing], __builtin_bit_cast(h8_t, wf[P][j]), j == 0 ? f16v_t{} : q);
                if (i == 2)
                    unpack_sz(step + 1);
                if constexpr (j >= 2) // 16 results over the slots 2 .. 7
                    flush(mt == 0 ? MT - 1 : mt - 1, (kFirst + mt + 1) & 1, (j - 2) * 8 / 3, (j - 1) * 8 / 3);
                if (j == 7)
                    sc_pending = sc;
                if constexpr (i >= kFirstPair) {
                    constexpr int from = (i - kFirstPair) * 32 / (N - kFirstPair), to = (i - kFirstPair + 1) * 32 / (N - kFirstPair);
#pragma unroll
                    for (int k = from; k < to; ++k)
                        wf[P ^ 1][k >> 2][k & 3] = dequant_pair(raw[k >> 4][(k >> 2) & 3], k & 3, zlo, zhi);
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, N>{});
        } else { // the last step of a piece that has no group for this wavefront
            flush(MT - 1, (kFirst + 1) & 1, 0, 16);
            sc_pending = 0.0f;
            p[0] = p[1] = f16v_t{};
        }
        const int s = s0;
        s0 = s1, s1 = s2, s2 = s;
    };
    int step = 0;
    for (; step + 1 < steps; step += 2) {
        body(std::integral_constant<int, 0>{}, step);
        body(std::integral_constant<int, 1>{}, step + 1);
    }
    if (step < steps) {
        body(std::integral_constant<int, 0>{}, step);
        flush(MT - 1, (MT - 1) & 1, 0, 16);
    } else {
        flush(MT - 1, (2 * MT - 1) & 1, 0, 16);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing may still write LDS
    __syncthreads();

    // Rows of 32 results lie kRedRow floats apart; a thread takes 8 neighbours of both tiles of the pair.
    const bool mine = nb * WN + wn < a.pairs;
    int tensor0, row_a, row_b;
    tile_of(nb * WN + wn, 1, tensor0, row_b);
    tile_of(nb * WN + wn, 0, tensor0, row_a);
    constexpr int kPasses = (MT + WK - 1) / WK; // 128 WK threads for MT x 128 such pieces
    const int piece = (wk * 2 + t) * 64 + lane;
    auto row_of = [&](int pass) { return (piece + pass * 128 * WK) >> 2; };
    const int n8 = (piece & 3) * 8;
    float4 angles[EPI == EPI_QKV ? kPasses : 1][4];
    if (EPI == EPI_QKV && tensor0 < 2) { // requested together, before the results are exchanged
#pragma unroll
        for (int pass = 0; pass < kPasses; ++pass) {
            const int m = mt0 * kTile + row_of(pass);
            const float* cs = a.rope + (static_cast<size_t>(m < a.M ? m : a.M - 1) * 64 + (row_a & 63) + n8) * 2;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                angles[pass][k] = reinterpret_cast<const float4*>(cs)[k];
        }
    }
    float* red = reinterpret_cast<float*>(lds);
    auto red_at = [&](int w, int tile, int row) { return red + (((w * WN + wn) * 2 + tile) * MT * kTile + row) * kRedRow; };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            red_at(wk, t, mt * kTile + 8 * (i >> 2) + 4 * h + (i & 3))[l31] = acc[mt][i];
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) {
        const int row = row_of(pass), m = mt0 * kTile + row;
        if (row >= MT * kTile || m >= a.M || !mine)
            continue;
        float v0[8] = {}, v1[8] = {};
#pragma unroll
        for (int w = 0; w < WK; ++w)
#pragma unroll
            for (int k = 0; k < 8; k += 4) {
                const float4 r0 = *reinterpret_cast<const float4*>(red_at(w, 0, row) + n8 + k);
                const float4 r1 = *reinterpret_cast<const float4*>(red_at(w, 1, row) + n8 + k);
                v0[k] += r0.x, v0[k + 1] += r0.y, v0[k + 2] += r0.z, v0[k + 3] += r0.w;
                v1[k] += r1.x, v1[k + 1] += r1.y, v1[k + 2] += r1.z, v1[k + 3] += r1.w;
            }
        if (EPI == EPI_QKV) {
            // q and k are rounded to fp16 before RoPE reads them (native/rope_kernel.cu:14-26)
            u32x4 oa, ob;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                uint16_t b0 = float_to_half_bits(v0[k]), b1 = float_to_half_bits(v1[k]);
                if (tensor0 < 2) {
                    const float4 cs = angles[pass][k >> 1];
                    rope_rotate(b0, b1, half_bits_to_float(b0), half_bits_to_float(b1), k & 1 ? cs.z : cs.x,
                                k & 1 ? cs.w : cs.y);
                }
                oa[k >> 1] = k & 1 ? oa[k >> 1] | static_cast<uint32_t>(b0) << 16 : b0;
                ob[k >> 1] = k & 1 ? ob[k >> 1] | static_cast<uint32_t>(b1) << 16 : b1;
            }
            uint16_t* o = choose(tensor0, a.out[0], a.out[1], a.out[2]) + static_cast<size_t>(m) * a.N + n8;
            *reinterpret_cast<u32x4*>(o + row_a) = oa;
            *reinterpret_cast<u32x4*>(o + row_b) = ob;
        } else if (EPI == EPI_PARTIAL) {
            float* o = a.parts + (static_cast<size_t>(split) * a.part_rows + m) * a.N + n8;
#pragma unroll
            for (int k = 0; k < 8; k += 4) {
                *reinterpret_cast<float4*>(o + row_a + k) = make_float4(v0[k], v0[k + 1], v0[k + 2], v0[k + 3]);
                *reinterpret_cast<float4*>(o + row_b + k) = make_float4(v1[k], v1[k + 1], v1[k + 2], v1[k + 3]);
            }
        } else {
            const int n = row_a + n8; // N is a multiple of 8
            if (n < a.N) {
                u32x4 o;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    float v = v0[k];
                    v *= 1.0f / (1.0f + expf(-v)); // native/mat_vec_kernel.cu:219-221
                    v *= v1[k];
                    const uint32_t bits = float_to_half_bits(v);
                    o[k >> 1] = k & 1 ? o[k >> 1] | bits << 16 : bits;
                }
                *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(a.out[0]) + frag_offset(m, n, a.out_groups)) = frag_order(o);
            }
        }
    }
}

// The token blocks of one block of weights run on one XCD, next to each other in time: its L2 serves the weights to all but the
// first.  With MT2 other than MT the first blocks of weights of every XCD are taken with MT token tiles, in rounds that
// fill its compute units, the others with MT2: what would be a last round of few workgroups that take as long as the others becomes one of
// more and shorter ones.
template <int MT, int MT2, int WN, int WK, int EPI>
__global__ __launch_bounds__(512, 2) void prefill_gemm_kernel(GemmArgs a)
{
    constexpr int kBytes = GemmLds<MT, WN, WK>::kBytes, kBytes2 = GemmLds<MT2, WN, WK>::kBytes;
    __shared__ __align__(1024) char lds[kBytes > kBytes2 ? kBytes : kBytes2];
    int slot = blockIdx.x >> 3, mblocks = a.mblocks, row = 0; // row: of 8 blocks of weights, one to an XCD
    const bool second = MT2 != MT && slot >= a.first * a.mblocks;
    if (second)
        slot -= a.first * a.mblocks, mblocks = a.mblocks2, row = a.first;
    const int unit = (row + slot / mblocks) * 8 + (blockIdx.x & 7), mb = slot % mblocks;
    if (unit >= a.nblocks * a.splits)
        return;
    if constexpr (MT2 != MT) {
        if (second) {
            gemm_block<MT2, WN, WK, EPI>(a, lds, unit, mb);
            return;
        }
    }
    gemm_block<MT, WN, WK, EPI>(a, lds, unit, mb);
}

static GemmShape gemm_shape(int tiles, int pairs, int groups, bool may_split)
{
    return gemm_shape(tiles, pairs, groups, may_split, ctx().num_cus > 0 ? ctx().num_cus : 256);
}

static GemmShape residual_shape(int M, int N, int groups) { return gemm_shape(ceil_div(M, kTile), N / 64, groups, true); }

template <int MT, int WN, int EPI, int MT2 = MT>
void launch_gemm_as(GemmArgs& a)
{
    a.mblocks = ceil_div(a.M, MT * kTile);
    a.mblocks2 = ceil_div(a.M, MT2 * kTile);
    a.nblocks = ceil_div(a.pairs, WN);
    const int rows = ceil_div(a.nblocks * a.splits, 8);
    if (MT2 == MT)
        a.first = rows;
    const dim3 grid(8 * (a.first * a.mblocks + (rows - a.first) * a.mblocks2));
    hipLaunchKernelGGL((prefill_gemm_kernel<MT, MT2, WN, 4 / WN, EPI>), grid, dim3(512), 0, ctx().stream, a);
}

template <int EPI>
int launch_gemm(const char* name, GemmArgs a, int pairs)
{
    const GemmShape s = gemm_shape(ceil_div(a.M, kTile), pairs, a.groups, EPI == EPI_PARTIAL);
    a.pairs = pairs;
    a.splits = s.splits;
    a.first = s.first;
    if constexpr (EPI != EPI_PARTIAL) {
        if (s.mt2 != s.mt) {
            if (s.mt == 4 && s.mt2 == 3)
                launch_gemm_as<4, 4, EPI, 3>(a);
            else if (s.mt == 4)
                launch_gemm_as<4, 4, EPI, 2>(a);
            else
                launch_gemm_as<3, 4, EPI, 2>(a);
            L2_LAUNCH_CHECK(name);
            return LLAMA2_OK;
        }
    }
    switch (s.wn * 10 + s.mt) {
    case 44: launch_gemm_as<4, 4, EPI>(a); break;
    case 43: launch_gemm_as<3, 4, EPI>(a); break;
    case 42: launch_gemm_as<2, 4, EPI>(a); break;
    case 41: launch_gemm_as<1, 4, EPI>(a); break;
    case 22: launch_gemm_as<2, 2, EPI>(a); break;
    case 21: launch_gemm_as<1, 2, EPI>(a); break;
    default: launch_gemm_as<1, 1, EPI>(a); break;
    }
    L2_LAUNCH_CHECK(name);
    return LLAMA2_OK;
}

// ---------------------------------------------------------------- causal attention
struct PrefillAttnArgs {
    const uint16_t* q; // [rows][dim], rotated
    const uint16_t* kcache;
    const uint16_t* vcache; // layer base, rows of `dim`
    uint16_t* xf;
    float* parts; // SPLIT: [splits][n_heads][part_rows][128] sums, then (maximum, sum) of every row
    int position, M, dim, n_heads, splits, part_rows;
    float scale;
};

constexpr int kAttnT = 64;        // timesteps per pass
constexpr int kKStride = 256 + 16; // bytes of a key row in LDS: 8 lanes x 16 bytes of consecutive rows hit all banks
constexpr int kVStride = 128 + 16; // bytes of a row of 64 timesteps of one output element
constexpr float kProbScale = 16384.0f; // 2^14: the largest probability, 1, fits into fp16
constexpr float kRestScale = 8192.0f;  // 2^13: what rounding to fp16 leaves of a scaled probability, at most 4, too

__device__ __forceinline__ int v_row_offset(int d) { return d * kVStride + (d >> 3) * 16; }

// A probability as fp16 numbers: p = (hi + (mid + lo) / 2^13) / 2^14, all 24 bits of it down to 2^-28, below that to
// the nearest multiple of 2^-51.
struct ProbParts {
    h8_t hi, mid, lo;
    __device__ __forceinline__ void set(int i, float p)
    {
        const float ps = p * kProbScale;
        hi[i] = static_cast<_Float16>(ps);
        const float rest = (ps - static_cast<float>(hi[i])) * kRestScale;
        mid[i] = static_cast<_Float16>(rest);
        lo[i] = static_cast<_Float16>(rest - static_cast<float>(mid[i]));
    }
};

// The 16 timesteps t0 .. t0 + 15 of one operand step, one product each, kept only by the queries that
// attend it (lane half u / 8 holds timestep t0 + u % 8 / 4 * 8 + u / 8 * 4 + u % 4 as element u % 8).
__device__ __forceinline__ void one_by_one(f16v_t (&o)[4], const ProbParts& p, const char* v, int l31, int hl, int t0, int limit)
{
    for (int u = 0; u < 16; ++u) {
        const bool keep = t0 + ((u & 7) >> 2) * 8 + (u >> 3) * 4 + (u & 3) <= limit;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            u32x4 w = *reinterpret_cast<const u32x4*>(v + v_row_offset(d * 32 + l31));
#pragma unroll
            for (int k = 0; k < 4; ++k)
                w[k] &= hl == (u >> 3) && k == ((u & 7) >> 1) ? ((u & 1) ? 0xFFFF0000u : 0x0000FFFFu) : 0u;
            const h8_t vf = __builtin_bit_cast(h8_t, w);
            const f16v_t c = mfma(vf, p.hi, f16v_t{});
            f16v_t r = mfma(vf, p.mid, f16v_t{});
            r = mfma(vf, p.lo, r);
#pragma unroll
            for (int i = 0; i < 16; ++i)
                o[d][i] = keep ? o[d][i] + __builtin_fmaf(r[i], 1.0f / kRestScale, c[i]) : o[d][i];
        }
    }
}

// One wavefront per tile of 32 queries of a head, NW tiles per workgroup share the key and value rows in
// LDS.  Scores are computed transposed (rows: timesteps, columns: queries), so that a lane holds 32
// timesteps of ONE query and its probabilities are already the second operand of the product with the
// transposed values.  Probabilities keep fp32's precision (ProbParts): three fp16 numbers that go through the
// matrix cores one after the other, the two small ones, scaled up, into sums of their own for each pass.  Two
// numbers of 22 bits, with nothing below 2^-39, took the same time (7B, 512 tokens 11.65 ms, three 11.61; 1003 + 24
// tokens 46.35, 46.46): a pass is bound by its chain, not by the matrix cores.  An infinite value that a query attends may
// reach its sum as NaN (infinity times a part that is 0): no output can tell, the norm behind it makes
// NaN of the whole row either way.
//
// What bounds it: a pass of 64 timesteps is a chain (LDS filled, scores, maximum, probabilities, output) of 4 us
// when its compute unit holds little else, and a tile walks all its passes.  SPLIT: gridDim.z workgroups share the
// passes of a tile, and prefill_attn_merge_kernel adds up their fp32 sums, which lie in the L2 in between.
// 7B, whole prompt in front of the first token, unsplit -> split: 75 tokens behind 3500 rows 12.9 -> 6.8 ms, behind
// 600 rows 6.57 -> 5.75; 9 tokens behind 3500 rows 11.1 -> 4.7; 512 tokens 11.8 -> 11.6.
template <int NW, bool SPLIT>
__global__ __launch_bounds__(NW * 64) void prefill_attn_kernel(PrefillAttnArgs a)
{
    __shared__ __align__(16) char ks[kAttnT * kKStride];
    __shared__ __align__(16) char vs[kRopeHeadSize * kVStride + 16 * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hl = lane >> 5, l31 = lane & 31;
    const int head = blockIdx.y;
    const int qb = gridDim.x - 1 - blockIdx.x; // the longest blocks first
    const int tile = qb * NW + wave;
    const int m = tile * kTile + l31;
    const int rows = a.position + a.M; // valid cache rows
    const int last_q = (qb * NW + NW) * kTile < a.M ? (qb * NW + NW) * kTile : a.M;
    const int t_end = a.position + last_q; // timesteps any query of the workgroup attends
    const int limit = a.position + m;      // last timestep of this lane's query
    const int wave_limit = a.position + tile * kTile + kTile - 1;

    h8_t qf[8];
    {
        const int mq = m < a.M ? m : a.M - 1;
        const uint16_t* q = a.q + static_cast<size_t>(mq) * a.dim + head * kRopeHeadSize + hl * 64;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            qf[j] = *reinterpret_cast<const h8_t*>(q + j * 8);
    }
    const uint32_t cache_bytes = static_cast<uint32_t>(rows) * a.dim * 2; // < 2^31: checked on the host
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.kcache, cache_bytes), rv = make_rsrc(a.vcache, cache_bytes);

    f16v_t o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
        o[d] = f16v_t{};
    float mx = -INFINITY, sum = 0.0f;

    constexpr int KP = kAttnT * 16 / (NW * 64); // 16-byte pieces of the key rows per thread
    constexpr int VP = 256 / (NW * 64);         // blocks of 4 timesteps x 8 elements per thread
    u32x4 kr[KP], vr[VP][4];
    auto request = [&](int tb) {
#pragma unroll
        for (int i = 0; i < KP; ++i) {
            const int e = threadIdx.x + i * NW * 64;
            kr[i] = __builtin_amdgcn_raw_buffer_load_b128(
                rk, ((tb + (e >> 4)) * a.dim + head * kRopeHeadSize + (e & 15) * 8) * 2, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int e = threadIdx.x + i * NW * 64, u = e >> 4;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                vr[i][r] = __builtin_amdgcn_raw_buffer_load_b128(
                    rv, ((tb + 4 * u + r) * a.dim + head * kRopeHeadSize + (e & 15) * 8) * 2, 0, 0);
        }
    };
    const int passes = (t_end + kAttnT - 1) / kAttnT;
    const int t_first = SPLIT ? passes * static_cast<int>(blockIdx.z) / a.splits * kAttnT : 0;
    const int t_last = SPLIT ? passes * (static_cast<int>(blockIdx.z) + 1) / a.splits * kAttnT : passes * kAttnT;
    if (t_first < t_last)
        request(t_first);
    for (int tb = t_first; tb < t_last; tb += kAttnT) {
        __syncthreads(); // the previous pass has been read
#pragma unroll
        for (int i = 0; i < KP; ++i) {
            const int e = threadIdx.x + i * NW * 64;
            *reinterpret_cast<u32x4*>(ks + (e >> 4) * kKStride + (e & 15) * 16) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < VP; ++i) {
            const int e = threadIdx.x + i * NW * 64, u = e >> 4, d0 = (e & 15) * 8;
            // unit u: timesteps 4u .. 4u + 3, i.e. block a = (u >> 1) & 3 and half u & 1 of tile u >> 3
            const int at = (u >> 3) * 64 + (u & 1) * 32 + ((u >> 1) & 3) * 8;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t a0 = vr[i][0][k], a1 = vr[i][1][k], a2 = vr[i][2][k], a3 = vr[i][3][k];
                const u32x2 even = {(a0 & 0xFFFFu) | (a1 << 16), (a2 & 0xFFFFu) | (a3 << 16)};
                const u32x2 odd = {(a0 >> 16) | (a1 & 0xFFFF0000u), (a2 >> 16) | (a3 & 0xFFFF0000u)};
                *reinterpret_cast<u32x2*>(vs + v_row_offset(d0 + 2 * k) + at) = even;
                *reinterpret_cast<u32x2*>(vs + v_row_offset(d0 + 2 * k + 1) + at) = odd;
            }
        }
        __syncthreads();
        if (tb + kAttnT < t_last)
            request(tb + kAttnT);
        if (tb > wave_limit)
            continue; // this tile attends nothing here (the barriers are the same for all wavefronts)

        // Where some queries do not attend some of these timesteps, an infinite or NaN value must not reach
        // them through a probability of 0.
        bool careful = false;
        if (tb + kAttnT - 1 > a.position + tile * kTile) {
            uint32_t bad = 0;
            for (int d = 0; d < 4; ++d)
                for (int u = 0; u < 4; ++u) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(vs + v_row_offset(d * 32 + l31) + (u >> 1) * 64 +
                                                                    hl * 32 + (u & 1) * 16);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        bad |= (v[k] & 0x7C007C00u) + 0x04000400u; // bits 15 and 31: all exponent bits set
                }
            careful = __any((bad & 0x80008000u) != 0);
        }

        f16v_t s[2] = {};
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const h8_t kf = *reinterpret_cast<const h8_t*>(ks + (tt * 32 + l31) * kKStride + hl * 128 + j * 16);
                s[tt] = mfma(kf, qf[j], s[tt]);
            }
        float bm = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = tb + tt * 32 + 8 * (i >> 2) + 4 * hl + (i & 3);
                const float v = half_bits_to_float(float_to_half_bits(s[tt][i] * a.scale)); // native/mat_vec_kernel.cu:71-74
                s[tt][i] = t <= limit ? v : -INFINITY;
                bm = fmaxf(bm, s[tt][i]);
            }
        bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
        const float nm = fmaxf(mx, bm);
        // no score above -infinity so far (a SPLIT whose timesteps the query does not attend, or scores below
        // fp16's range): probabilities are 0, not NaN; if none follows, the quotient by their sum is NaN
        const float base = nm == -INFINITY ? 0.0f : nm;
        const float alpha = expf(mx - base);
        mx = nm;
        sum *= alpha;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                o[d][i] *= alpha;
        ProbParts p[4]; // of the operand steps of 16 timesteps
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float pr = expf(s[u >> 1][8 * (u & 1) + i] - base);
                sum += pr;
                p[u].set(i, pr);
            }
        auto values = [&](int u) { return vs + (u >> 1) * 64 + hl * 32 + (u & 1) * 16; };
        if (careful) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                one_by_one(o, p[u], values(u), l31, hl, tb + u * 16, limit);
            continue;
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            f16v_t r = {};
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const h8_t vf = *reinterpret_cast<const h8_t*>(values(u) + v_row_offset(d * 32 + l31));
                o[d] = mfma(vf, p[u].hi, o[d]);
                r = mfma(vf, p[u].mid, r);
                r = mfma(vf, p[u].lo, r);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i)
                o[d][i] = __builtin_fmaf(r[i], 1.0f / kRestScale, o[d][i]);
        }
    }
    sum += __shfl_xor(sum, 32, 64);
    const float inv = 1.0f / kProbScale;
    if (tile * kTile >= a.M) // the whole wavefront
        return;
    if constexpr (SPLIT) {
        const size_t row = (static_cast<size_t>(blockIdx.z) * a.n_heads + head) * a.part_rows + m;
        float* out = a.parts + row * kRopeHeadSize + 4 * hl;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                *reinterpret_cast<float4*>(out + d * 32 + 8 * k) =
                    float4{o[d][4 * k] * inv, o[d][4 * k + 1] * inv, o[d][4 * k + 2] * inv, o[d][4 * k + 3] * inv};
        float* stats = a.parts + static_cast<size_t>(a.splits) * a.n_heads * a.part_rows * kRopeHeadSize;
        if (hl == 0)
            *reinterpret_cast<float2*>(stats + row * 2) = float2{mx, sum};
        return;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int p = 0; p < 2; ++p) { // blocks of 8 outputs, two at a time: the lower half of the lanes stores the first
            uint32_t w[2][2];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int i = (2 * p + b) * 4 + 2 * k;
                    w[b][k] = static_cast<uint32_t>(float_to_half_bits(o[d][i] * inv / sum)) |
                              static_cast<uint32_t>(float_to_half_bits(o[d][i + 1] * inv / sum)) << 16;
                }
            uint32_t lo[2], hi[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t got = __shfl_xor(static_cast<int>(hl ? w[0][k] : w[1][k]), 32, 64);
                lo[k] = hl ? got : w[0][k];
                hi[k] = hl ? w[1][k] : got;
            }
            const u32x4 out = {(lo[0] & 0xFFFFu) | (hi[0] << 16), (lo[0] >> 16) | (hi[0] & 0xFFFF0000u),
                               (lo[1] & 0xFFFFu) | (hi[1] << 16), (lo[1] >> 16) | (hi[1] & 0xFFFF0000u)};
            const int k0 = head * kRopeHeadSize + (d * 4 + 2 * p + hl) * 8;
            if (m < a.M)
                *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(a.xf) + frag_offset(m, k0, a.n_heads)) = out;
        }
}

// Adds up the pieces of a split attention, 16 lanes of 8 outputs per row and head.
__global__ __launch_bounds__(256) void prefill_attn_merge_kernel(PrefillAttnArgs a)
{
    const int m = blockIdx.x * 16 + (threadIdx.x >> 4), head = blockIdx.y, k = (threadIdx.x & 15) * 8;
    if (m >= a.M)
        return;
    const size_t step = static_cast<size_t>(a.n_heads) * a.part_rows, row = static_cast<size_t>(head) * a.part_rows + m;
    const float2* stats = reinterpret_cast<const float2*>(a.parts + a.splits * step * kRopeHeadSize) + row;
    float mx = -INFINITY;
    for (int i = 0; i < a.splits; ++i)
        mx = fmaxf(mx, stats[i * step].x);
    float o[8] = {}, sum = 0.0f;
    for (int i = 0; i < a.splits; ++i) { // in order: deterministic
        const float2 st = stats[i * step];
        const float w = st.x == -INFINITY ? 0.0f : expf(st.x - mx); // a piece the row does not attend
        const float4* p = reinterpret_cast<const float4*>(a.parts + (i * step + row) * kRopeHeadSize + k);
        const float4 p0 = p[0], p1 = p[1];
        sum = fmaf(w, st.y, sum);
        o[0] = fmaf(w, p0.x, o[0]), o[1] = fmaf(w, p0.y, o[1]), o[2] = fmaf(w, p0.z, o[2]), o[3] = fmaf(w, p0.w, o[3]);
        o[4] = fmaf(w, p1.x, o[4]), o[5] = fmaf(w, p1.y, o[5]), o[6] = fmaf(w, p1.z, o[6]), o[7] = fmaf(w, p1.w, o[7]);
    }
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        v[e] = static_cast<uint32_t>(float_to_half_bits(o[2 * e] / sum)) |
               static_cast<uint32_t>(float_to_half_bits(o[2 * e + 1] / sum)) << 16;
    *reinterpret_cast<u32x4*>(reinterpret_cast<char*>(a.xf) + frag_offset(m, head * kRopeHeadSize + k, a.n_heads)) =
        frag_order(v);
}

struct PrefillAttnShape {
    int waves, splits;
};

constexpr int kMaxAttnSplits = 32;

// Tiles share key and value rows (waves) as long as every compute unit has a workgroup.  Passes are split until there
// are 4 wavefronts per compute unit; more only costs the merge (7B: 512 tokens, 1024 wavefronts 11.62 ms, 2048
// 11.91; 1003 tokens, 1024 wavefronts 19.3, 2048 19.6; 400 behind 3500 rows, 416 wavefronts 18.7, 832 15.0).
// A piece may be a single pass: 20 tokens behind 200 rows 3.55 ms, with two passes at least 3.65, unsplit 3.89.
static PrefillAttnShape prefill_attn_shape(int M, int rows, int n_heads)
{
    const int tiles = ceil_div(M, kTile), passes = ceil_div(rows, kAttnT);
    const int cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    const int waves = ceil_div(tiles, 4) * n_heads >= cus ? 4 : ceil_div(tiles, 2) * n_heads >= cus ? 2 : 1;
    int splits = 4 * cus / (tiles * n_heads);
    splits = splits < passes ? splits : passes;
    splits = splits < kMaxAttnSplits ? splits : kMaxAttnSplits;
    return PrefillAttnShape{waves, splits > 1 ? splits : 1};
}

static size_t attn_part_floats(int M, int splits, int n_heads)
{
    return splits > 1 ? static_cast<size_t>(splits) * n_heads * ceil_div(M, kTile) * kTile * (kRopeHeadSize + 2) : 0;
}

template <int NW>
static void launch_prefill_attn_as(const PrefillAttnArgs& a)
{
    const dim3 grid(ceil_div(ceil_div(a.M, kTile), NW), a.n_heads, a.splits), block(NW * 64);
    if (a.splits > 1)
        hipLaunchKernelGGL((prefill_attn_kernel<NW, true>), grid, block, 0, ctx().stream, a);
    else
        hipLaunchKernelGGL((prefill_attn_kernel<NW, false>), grid, block, 0, ctx().stream, a);
}

int launch_prefill_attn(PrefillAttnArgs a)
{
    const PrefillAttnShape shape = prefill_attn_shape(a.M, a.position + a.M, a.n_heads);
    a.splits = shape.splits;
    a.part_rows = ceil_div(a.M, kTile) * kTile;
    switch (shape.waves) {
    case 4: launch_prefill_attn_as<4>(a); break;
    case 2: launch_prefill_attn_as<2>(a); break;
    default: launch_prefill_attn_as<1>(a); break;
    }
    L2_LAUNCH_CHECK("prefill attention");
    if (a.splits > 1) {
        hipLaunchKernelGGL(prefill_attn_merge_kernel, dim3(ceil_div(a.M, 16), a.n_heads), dim3(256), 0, ctx().stream, a);
        L2_LAUNCH_CHECK("prefill attention merge");
    }
    return LLAMA2_OK;
}

int launch_prefill_norm(const NormArgs& a, int M)
{
    const dim3 grid(M), block(256);
    const hipStream_t st = ctx().stream;
    switch (ceil_div(a.K, 2048)) {
    case 1: hipLaunchKernelGGL((prefill_norm_kernel<1>), grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL((prefill_norm_kernel<2>), grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL((prefill_norm_kernel<3>), grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL((prefill_norm_kernel<4>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((prefill_norm_kernel<8>), grid, block, 0, st, a); break;
    }
    L2_LAUNCH_CHECK("prefill norm");
    return LLAMA2_OK;
}

static size_t up256(size_t n) { return (n + 255) / 256 * 256; }

struct PrefillSizes {
    size_t vec, hid, rope, parts;
    size_t total() const { return 3 * vec + hid + rope + parts; }
};

static PrefillSizes prefill_sizes(const llama2_config& cfg, int rows)
{
    PrefillSizes z;
    z.vec = up256(static_cast<size_t>(rows) * cfg.dim * 2);
    z.hid = up256(static_cast<size_t>(rows) * ceil_div(cfg.hidden_dim, kGroup) * kGroup * 2);
    z.rope = up256(static_cast<size_t>(rows) * 128 * sizeof(float));
    size_t parts = 0; // the largest [splits][rows][dim] any batch needs
    for (int m = kTile; m <= rows; m += kTile)
        for (int k : {cfg.dim, cfg.hidden_dim}) {
            const size_t n = static_cast<size_t>(residual_shape(m, cfg.dim, ceil_div(k, kGroup)).splits) * m;
            parts = n > parts ? n : parts;
        }
    parts *= cfg.dim;
    for (int m = kTile; m <= rows; m += kTile) { // attention's pieces, gone before the next product writes its own
        const size_t n = attn_part_floats(m, prefill_attn_shape(m, cfg.seq_len, cfg.n_heads).splits, cfg.n_heads);
        parts = n > parts ? n : parts;
    }
    z.parts = parts * sizeof(float);
    return z;
}

int prefill_create(PrefillWorkspace& ws, const llama2_config& cfg)
{
    // A host may have given nearly all of the memory to its caches (the reference's run state leaves 8 MiB): at
    // most half of what is free is taken, with smaller batches where that is too little, and without any room
    // the decoder goes step by step.
    size_t limit = 0, total_memory = 0;
    L2_HIP(hipMemGetInfo(&limit, &total_memory));
    limit /= 2;
    if (const char* mib = getenv("LLAMA2_PREFILL_MIB")) {
        const size_t wanted = static_cast<size_t>(strtoull(mib, nullptr, 10)) << 20;
        limit = wanted < limit ? wanted : limit;
    }
    int rows = ceil_div(cfg.seq_len < kPrefillMaxRows ? cfg.seq_len : kPrefillMaxRows, kTile) * kTile;
    PrefillSizes z{};
    for (;; rows = ceil_div(rows / 2, kTile) * kTile) {
        z = prefill_sizes(cfg, rows);
        if (z.total() <= limit) {
            const hipError_t e = hipMalloc(&ws.base, z.total());
            if (e == hipSuccess)
                break;
            if (e != hipErrorOutOfMemory)
                return hip_fail(e, "prefill workspace");
            (void)hipGetLastError();
            ws.base = nullptr;
        }
        if (rows == kTile)
            return LLAMA2_OK;
    }
    char* p = static_cast<char*>(ws.base);
    ws.x = reinterpret_cast<uint16_t*>(p);
    ws.q = reinterpret_cast<uint16_t*>(p + z.vec);
    ws.xf = reinterpret_cast<uint16_t*>(p + 2 * z.vec);
    ws.hf = reinterpret_cast<uint16_t*>(p + 3 * z.vec);
    ws.rope = reinterpret_cast<float*>(p + 3 * z.vec + z.hid);
    ws.parts = reinterpret_cast<float*>(p + 3 * z.vec + z.hid + z.rope);
    ws.rows = rows;
    // hf beyond hidden_dim is never written and must read as zero
    L2_HIP(hipMemsetAsync(ws.base, 0, z.total(), ctx().stream));
    L2_HIP(hipStreamSynchronize(ctx().stream));
    return LLAMA2_OK;
}

void prefill_destroy(PrefillWorkspace& ws)
{
    if (ws.base)
        (void)hipFree(ws.base);
    ws = PrefillWorkspace{};
}

#define L2_TRY(expr)          \
    do {                      \
        int rc_ = (expr);     \
        if (rc_ != LLAMA2_OK) \
            return rc_;       \
    } while (0)

static int prefill_batch(const PrefillWorkspace& ws, const llama2_config& c, const llama2_layer_weights* layers,
                         const llama2_transformer_weights& w, const llama2_run_state& s, int position, int M)
{
    const int dim = c.dim, hidden = c.hidden_dim;
    const int ss = ceil_div(dim, 128), wsz = ceil_div(dim, 32) * 4, zs = ceil_div(ss, 8);
    const int hss = ceil_div(hidden, 128), hws = ceil_div(hidden, 32) * 4, hzs = ceil_div(hss, 8);
    const uint32_t xf_bytes = static_cast<uint32_t>(ws.rows) * ss * kGroup * 2;
    const uint32_t hf_bytes = static_cast<uint32_t>(ws.rows) * hss * kGroup * 2;
    const int part_rows = ceil_div(M, kTile) * kTile;
    const int o_splits = residual_shape(M, dim, ss).splits, down_splits = residual_shape(M, dim, hss).splits;
    auto qw = [](const llama2_qweight& q) { return QW{q.weight, q.zeros, q.scales}; };
    hipLaunchKernelGGL(prefill_rope_kernel, dim3(ceil_div(M * 64, 256)), dim3(256), 0, ctx().stream, ws.rope, position,
                       M, c.rope_theta);
    L2_LAUNCH_CHECK("prefill rope");
    for (int i = 0; i < c.n_layers; ++i) {
        const llama2_layer_weights& L = layers[i];
        const size_t layer_offset = static_cast<size_t>(i) * c.seq_len * dim;
        const size_t row = layer_offset + static_cast<size_t>(position) * dim;
        NormArgs n{};
        n.x = ws.x, n.gamma = L.rms_attention, n.xf = ws.xf, n.K = dim, n.eps = 1e-5f;
        n.part_rows = part_rows;
        if (i > 0)
            n.parts = ws.parts, n.n_parts = down_splits;
        else
            n.embedding = w.token_embedding_table, n.tokens = s.tokens + position, n.vocab = c.vocab_size;
        L2_TRY(launch_prefill_norm(n, M));
        {
            GemmArgs a{};
            a.m[0] = qw(L.query), a.m[1] = qw(L.key), a.m[2] = qw(L.value);
            a.out[0] = ws.q, a.out[1] = s.key_cache + row, a.out[2] = s.value_cache + row;
            a.xf = ws.xf, a.xf_bytes = xf_bytes, a.groups = ss, a.N = dim, a.ws = wsz, a.ss = ss, a.zs = zs, a.M = M;
            a.rope = ws.rope;
            L2_TRY(launch_gemm<EPI_QKV>("prefill qkv", a, 3 * (dim / 64)));
        }
        if (i == c.n_layers - 1)
            break; // the batch's tokens leave nothing but their cache rows
        {
            PrefillAttnArgs a{};
            a.q = ws.q, a.kcache = s.key_cache + layer_offset, a.vcache = s.value_cache + layer_offset, a.xf = ws.xf;
            a.parts = ws.parts, a.position = position, a.M = M, a.dim = dim, a.n_heads = c.n_heads;
            a.scale = 1.0f / sqrtf(static_cast<float>(kRopeHeadSize));
            L2_TRY(launch_prefill_attn(a));
        }
        {
            GemmArgs a{};
            a.m[0] = qw(L.output), a.parts = ws.parts, a.part_rows = part_rows, a.xf = ws.xf, a.xf_bytes = xf_bytes;
            a.groups = ss, a.N = dim, a.ws = wsz, a.ss = ss, a.zs = zs, a.M = M;
            L2_TRY(launch_gemm<EPI_PARTIAL>("prefill o-proj", a, dim / 64));
        }
        n.gamma = L.rms_feed_forward, n.embedding = nullptr, n.parts = ws.parts, n.n_parts = o_splits;
        L2_TRY(launch_prefill_norm(n, M));
        {
            GemmArgs a{};
            a.m[0] = qw(L.gate), a.m[1] = qw(L.up), a.out[0] = ws.hf, a.xf = ws.xf, a.xf_bytes = xf_bytes;
            a.groups = ss, a.N = hidden, a.ws = wsz, a.ss = ss, a.zs = zs, a.M = M;
            a.out_groups = hss;
            L2_TRY(launch_gemm<EPI_SWIGLU>("prefill swiglu", a, ceil_div(hidden, kTile)));
        }
        {
            GemmArgs a{};
            a.m[0] = qw(L.down), a.parts = ws.parts, a.part_rows = part_rows, a.xf = ws.hf, a.xf_bytes = hf_bytes;
            a.groups = hss, a.N = dim, a.ws = hws, a.ss = hss, a.zs = hzs, a.M = M;
            L2_TRY(launch_gemm<EPI_PARTIAL>("prefill down-proj", a, dim / 64));
        }
    }
    return LLAMA2_OK;
}

int prefill_run(const PrefillWorkspace& ws, const llama2_config& cfg, const llama2_layer_weights* layers,
                const llama2_transformer_weights& w, const llama2_run_state& s, int position, int count)
{
    const int batches = ceil_div(count, ws.rows), rows = ceil_div(count, batches);
    for (int done = 0; done < count; done += rows)
        L2_TRY(prefill_batch(ws, cfg, layers, w, s, position + done, rows < count - done ? rows : count - done));
    return LLAMA2_OK;
}

} // namespace l2
