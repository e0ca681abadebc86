// Shared host/device helpers of libllama2_hip.so (gfx950 only).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <mutex>

#include "../../include/llama2_hip.h"

namespace l2 {

// ------------------------------------------------------------------ host side
constexpr int kMaxRetiredPartials = 32;

struct SamplerScratch;
struct HostStep;

struct Context {
    bool ready = false;
    int device = -1;
    hipStream_t stream = nullptr;
    int num_cus = 0;
    bool capturing = false; // between llama2_graph_begin_capture and _end_capture
    // A/B switches of the int4 mat-vec launches: LLAMA2_INT4_NARROW=1 one row per item for every
    // shape, LLAMA2_INT4_BLOCKS=1 blocks of rows for every shape (default: by row length)
    // LLAMA2_INT4_NO_SPAN=1: never the span kernel (the shapes it does not take always go this way)
    bool int4_narrow = false;
    bool int4_blocks = false;
    bool int4_no_span = false;
    int attn_waves = 0; // LLAMA2_ATTN_WAVES: block size of the attention entry points, for sweeps (0: by length)
    // fp32 partial sums of the sequence-split attention kernels
    float* attn_partials = nullptr;
    size_t attn_partials_bytes = 0;
    // earlier, smaller buffers: a graph captured by the caller may still hold their address,
    // so they stay allocated until llama2_shutdown
    float* retired_partials[kMaxRetiredPartials] = {};
    int n_retired_partials = 0;
    // per-head arrival counters of llama2_multi_head_attention (zero between launches)
    unsigned* attn_counters = nullptr;
    SamplerScratch* sampler = nullptr; // between the sampler modules' launches (sampler_kernels.hpp)
    // Pinned: where a kernel leaves the token that the call behind it returns (a copy of 4 bytes is a launch of 4.3 us)
    int* host_token = nullptr;
};

constexpr int kMaxAttnHeads = 1024;

Context& ctx();
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int hip_fail(hipError_t e, const char* what);
int ensure_attn_partials(size_t bytes);
// Device address of llama2_vec_mat_static's scratch array on `device` (current), asked for once at llama2_init.
int resolve_vec_mat_static_scratch(int device);
// Sampler.Sample's stochastic branch (sampler.hip).  token_only: the caller reads the
// token alone, so the sort may stop at the head of the distribution that holds top_p of the mass.
int sample_launch(const char* fn, SamplerScratch* scratch, uint16_t* logits, int* indices, int size, float temperature,
                  float top_p, float coin, int* result, int pos, bool token_only, const HostStep* host = nullptr);

// HIP's current device is a per-thread setting: a host thread other than the one that called
// llama2_init (a thread-pool worker of the managed host, say) is bound to the library's device on
// its first call.
int bind_thread();

// Every entry point runs under one recursive lock (entry points call each other): host threads
// that share the library -- one Transformer per connection, say -- take turns.  The GPU work is in
// order on one stream either way; what the lock protects is the stream-capture state and the lazily
// captured graphs.  llama2_graph_begin_capture keeps the lock until llama2_graph_end_capture.
std::recursive_mutex& api_mutex();

#define L2_REQUIRE_INIT()                                                          \
    std::lock_guard<std::recursive_mutex> l2_api_lock_(::l2::api_mutex());         \
    do {                                                                           \
        if (!::l2::ctx().ready)                                                    \
            return ::l2::fail(LLAMA2_ERR_NOT_INITIALIZED, "%s: llama2_init has not been called", __func__); \
        if (int rc_bind_ = ::l2::bind_thread())                                    \
            return rc_bind_;                                                       \
    } while (0)

#define L2_CHECK(cond, ...)                                                        \
    do {                                                                           \
        if (!(cond))                                                               \
            return ::l2::fail(LLAMA2_ERR_INVALID_ARGUMENT, __VA_ARGS__);           \
    } while (0)

#define L2_HIP(expr)                                                               \
    do {                                                                           \
        hipError_t e_ = (expr);                                                    \
        if (e_ != hipSuccess)                                                      \
            return ::l2::hip_fail(e_, #expr);                                      \
    } while (0)

#define L2_LAUNCH_CHECK(name)                                                      \
    do {                                                                           \
        hipError_t e_ = hipGetLastError();                                         \
        if (e_ != hipSuccess)                                                      \
            return ::l2::hip_fail(e_, name);                                       \
    } while (0)

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }
inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
inline bool overlap(const void* a, size_t na, const void* b, size_t nb)
{
    auto pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return pa < pb + nb && pb < pa + na;
}

// ---------------------------------------------------------------- device side
#if defined(__HIPCC__)

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2_t as_h2(uint32_t v) { return __builtin_bit_cast(h2_t, v); }
__device__ __forceinline__ uint32_t as_u32(h2_t v) { return __builtin_bit_cast(uint32_t, v); }

// fp32 += a.x*b.x + a.y*b.y  (v_dot2_f32_f16: fp16 products, fp32 accumulate)
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float acc)
{
    return __builtin_amdgcn_fdot2(as_h2(a), as_h2(b), acc, false);
}

__device__ __forceinline__ float half_bits_to_float(uint16_t h)
{
    return static_cast<float>(__builtin_bit_cast(_Float16, h));
}
__device__ __forceinline__ uint16_t float_to_half_bits(float f)
{
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(f)); // v_cvt_f16_f32, RNE
}

// The rotation of native/rope_kernel.cu:14-26, rounded the way the reference rounds it: the fp32
// value first, then __float2half of it.  The multiply-adds are spelled out and the fp32 results are
// made opaque before the conversion, so that every kernel that inlines this produces the same bits:
// left alone, the compiler fuses some of these multiply-adds with the conversion (v_fma_mixlo_f16,
// ONE rounding straight to fp16) and not others, depending on the surrounding code, and a value
// near an fp16 tie then rounds differently from kernel to kernel.
__device__ __forceinline__ void rope_rotate(uint16_t& b0, uint16_t& b1, float v0, float v1, float fcr, float fci)
{
    float o0 = __builtin_fmaf(v0, fcr, -(v1 * fci));
    float o1 = __builtin_fmaf(v0, fci, v1 * fcr);
    asm volatile("" : "+v"(o0), "+v"(o1));
    b0 = float_to_half_bits(o0);
    b1 = float_to_half_bits(o1);
}

// DPP controls (GCN3/CDNA encoding)
constexpr int DPP_QUAD_XOR1 = 0xB1;        // quad_perm:[1,0,3,2]
constexpr int DPP_QUAD_XOR2 = 0x4E;        // quad_perm:[2,3,0,1]
constexpr int DPP_QUAD_XOR3 = 0x1B;        // quad_perm:[3,2,1,0]
constexpr int DPP_ROW_ROR8 = 0x128;        // lane i <- lane (i + 8) % 16
constexpr int DPP_ROW_HALF_MIRROR = 0x141; // lane i <- lane 7-i within 8
constexpr int DPP_ROW_MIRROR = 0x140;      // lane i <- lane 15-i within 16
constexpr int DPP_ROW_BCAST15 = 0x142;     // lane 15 of each row -> next row
constexpr int DPP_ROW_BCAST31 = 0x143;     // lane 31 -> rows 2,3
constexpr int DPP_ROW_NEWBCAST = 0x150;    // + i: lane i of each row of 16 -> the whole row

template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_f32(float v)
{
    // lanes whose row is masked out (or whose source is invalid) read 0
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, false));
}

// Sum over each 16-lane row, the sums of neighbouring lanes in front of it; every lane of the row ends with a total.
__device__ __forceinline__ float row16_sum_of_pairs(float v)
{
    v += dpp_f32<DPP_QUAD_XOR2>(v);
    v += dpp_f32<DPP_ROW_HALF_MIRROR>(v);
    v += dpp_f32<DPP_ROW_MIRROR>(v);
    return v;
}

// Sum over each 16-lane row; every lane of the row ends with the row total.
__device__ __forceinline__ float row16_sum(float v)
{
    v += dpp_f32<DPP_QUAD_XOR1>(v);
    return row16_sum_of_pairs(v);
}

// Denominator of merged blocks of timesteps: sum of w * l over each 16-lane row, block i in lane i; the total is that of
// the row's first lane.  The fused multiply-add of the first level is written out: left to the compiler it came and went
// with the code around it, and the three kernels that merge (attention, o-projection, persistent step) owe each other
// the same bits.
__device__ __forceinline__ float row16_dot(float w, float l)
{
    return row16_sum_of_pairs(__builtin_fmaf(w, l, dpp_f32<DPP_QUAD_XOR1>(w * l)));
}

// Largest value of each 16-lane row, in every lane of it.
__device__ __forceinline__ float row16_max(float v)
{
    v = fmaxf(v, dpp_f32<DPP_QUAD_XOR1>(v));
    v = fmaxf(v, dpp_f32<DPP_QUAD_XOR2>(v));
    v = fmaxf(v, dpp_f32<DPP_ROW_HALF_MIRROR>(v));
    v = fmaxf(v, dpp_f32<DPP_ROW_MIRROR>(v));
    return v;
}

// Sum of the four row totals (lane 15 of each row), returned in every lane (as a scalar).
__device__ __forceinline__ float wave_sum_of_rows(float v)
{
    v += dpp_f32<DPP_ROW_BCAST15, 0xA>(v);
    v += dpp_f32<DPP_ROW_BCAST31, 0xC>(v);
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Sum over the 64-lane wavefront, returned in every lane (as a scalar).
__device__ __forceinline__ float wave_sum(float v) { return wave_sum_of_rows(row16_sum(v)); }

// The denominator of up to 64 blocks; up to 16 blocks it has the bits of row16_dot's first lane (lanes 0 and 15 of a
// row add up the same terms in the same order, and the other rows are zero).
__device__ __forceinline__ float wave_dot(float w, float l) { return wave_sum_of_rows(row16_dot(w, l)); }

// Largest value of the 64-lane wavefront, in every lane; all lanes take part.  By row operations and lane reads: six
// shuffles are six round trips through LDS (softmax of 300 scores 3.28 -> 3.08 us, a decode step of 7B at 700 rows
// 1147 -> 1138).
__device__ __forceinline__ float wave_max(float v)
{
    const int m = __builtin_bit_cast(int, row16_max(v));
    float rows[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        rows[r] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(m, 16 * r));
    return fmaxf(fmaxf(rows[0], rows[1]), fmaxf(rows[2], rows[3]));
}

// The sum of a lane's value and that of the lane 16 (32) further on or back.
__device__ __forceinline__ float add_xor16(float v)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_xor32(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Data handed from one workgroup to another INSIDE a kernel (attention partials,
// arrival counters) moves through agent-scope accesses: the store is written
// through to the level every XCD sees, the load bypasses this XCD's possibly
// stale L2 lines.  That replaces __threadfence(), whose L2 write-back +
// invalidate costs tens of microseconds on this part.  Ordering: a producer
// calls wait_agent_stores() before it announces its data with an atomic.
__device__ __forceinline__ void store_agent(float* p, float v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_agent(const float* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_agent(unsigned* p, unsigned v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned add_agent(unsigned* p, unsigned v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void wait_agent_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Sum over a 256-thread workgroup (4 wavefronts), identical in every thread and
// independent of which kernel calls it: RMSNorm is evaluated both by the
// stand-alone module and inside the fused mat-vec kernels, and the two must
// agree bit for bit.  `lds4` holds 4 floats.
__device__ __forceinline__ float block256_sum(float v, float* lds4)
{
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0)
        lds4[threadIdx.x >> 6] = v;
    __syncthreads();
    const float t = (lds4[0] + lds4[1]) + (lds4[2] + lds4[3]);
    __syncthreads();
    return t;
}

// Cache-policy bits of the raw buffer load/store builtins on gfx94x/gfx950.
constexpr int kAuxNonTemporal = 2; // "nt": streamed once, do not keep
constexpr int kAuxAgent = 16;      // "sc1": coherent at agent scope (sees other workgroups' sc1 stores)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes)
{
    // raw buffer, 32-bit elements; out-of-range reads return 0
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}

// One thread's share of a K-element fp16 vector read 16 bytes at a time by a
// 256-thread workgroup: piece i covers elements 8*(tid + 256 i) .. +7.
template <int PIECES>
struct VecPieces {
    u32x4 v[PIECES];
    __device__ __forceinline__ void load(const uint16_t* p, int K)
    {
        const __amdgpu_buffer_rsrc_t r = make_rsrc(p, K * 2);
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
            v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, (threadIdx.x + i * 256) * 16, 0, 0);
    }
    __device__ __forceinline__ float sum_squares() const
    {
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const h2_t p = as_h2(v[i][k]);
                const float a = static_cast<float>(p[0]), b = static_cast<float>(p[1]);
                ss += a * a;
                ss += b * b;
            }
        return ss;
    }
    // v <- half(rms * gamma * v), the product order of native/rmsnorm_kernel.cu:34
    __device__ __forceinline__ void scale(float rms, const VecPieces& gamma)
    {
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const h2_t x = as_h2(v[i][k]), g = as_h2(gamma.v[i][k]);
                h2_t o;
                o[0] = static_cast<_Float16>(rms * static_cast<float>(g[0]) * static_cast<float>(x[0]));
                o[1] = static_cast<_Float16>(rms * static_cast<float>(g[1]) * static_cast<float>(x[1]));
                v[i][k] = as_u32(o);
            }
    }
};

// Largest fp16 value of x[0..size), lowest index among equals, by a workgroup of 1024 threads;
// valid in thread 0 (0 when every entry is NaN).  The value first, then the lowest index that holds it: both are
// independent of any order (no race, unlike native/argmax_kernel.cu:32-36).  `sv`: 16 entries of LDS, `si`: one.
//
// One compute unit, so latency and issue bound it: all loads of up to 32768 elements are requested together, and the
// elements of a thread take one packed maximum per two; only a thread that holds the largest value looks for its
// index.  Carrying (value, index) pairs through every comparison, loads one by one, the kernels of the decode step and of
// a host's loop took 5.3 and 5.4 us for 32000 logits (profiler), now 4.5 and 4.0; for 1000 logits 4.6 -> 4.2.
__device__ __forceinline__ h2_t max_h2(h2_t a, h2_t b) { return __builtin_elementwise_max(a, b); } // NaN: the other one

__device__ __forceinline__ int first_equal(u32x4 v, float m, int first) // index of the first of 8 that equals m
{
    int at = 0x7FFFFFFF;
#pragma unroll
    for (int k = 7; k >= 0; --k)
        at = half_bits_to_float(static_cast<uint16_t>(v[k >> 1] >> (16 * (k & 1)))) == m ? first + k : at;
    return at;
}

struct Nothing {
    __device__ __forceinline__ void operator()() const {}
};

// `meanwhile` runs while the elements are on their way.
template <class F = Nothing>
__device__ __forceinline__ int block1024_argmax(const uint16_t* x, int size, float* sv, int* si, F meanwhile = F())
{
    constexpr int kPieces = 4; // of 8 elements per thread, held in registers
    constexpr uint32_t kLeast = 0xFC00FC00u;
    // 16 bytes per load while whole groups of 8 remain (when x is 16-byte aligned), the rest one by one
    const int n8 = (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? size >> 3 : 0;
    const u32x4* x8 = reinterpret_cast<const u32x4*>(x);
    const int t = threadIdx.x;
    if (t == 0)
        si[0] = 0x7FFFFFFF;
    u32x4 v[kPieces];
    h2_t m2 = as_h2(kLeast);
    // Beyond the end the last group once more; without groups the buffer is empty and reads as zero.
    const __amdgpu_buffer_rsrc_t r = make_rsrc(x, min(n8, kPieces * 1024) * 16);
#pragma unroll
    for (int p = 0; p < kPieces; ++p)
        v[p] = __builtin_amdgcn_raw_buffer_load_b128(r, min(t + p * 1024, n8 - 1) * 16, 0, 0);
    meanwhile();
    if (n8 > 0) {
#pragma unroll
        for (int p = 0; p < kPieces; ++p)
            asm volatile("" : "+v"(v[p])); // nothing that needs the elements moves in front of `meanwhile`
#pragma unroll
        for (int p = 0; p < kPieces; ++p)
            m2 = max_h2(m2, max_h2(max_h2(as_h2(v[p][0]), as_h2(v[p][1])), max_h2(as_h2(v[p][2]), as_h2(v[p][3]))));
    }
    for (int g = t + kPieces * 1024; g < n8; g += 1024) {
        const u32x4 w = x8[g];
        m2 = max_h2(m2, max_h2(max_h2(as_h2(w[0]), as_h2(w[1])), max_h2(as_h2(w[2]), as_h2(w[3]))));
    }
    float m = fmaxf(static_cast<float>(m2[0]), static_cast<float>(m2[1]));
    for (int i = n8 * 8 + t; i < size; i += 1024)
        m = fmaxf(m, half_bits_to_float(x[i]));

    const float wave = wave_max(m);
    if ((t & 63) == 0)
        sv[t >> 6] = wave;
    __syncthreads();
    const float most = row16_max(sv[t & 15]);
    if (m == most) {
        int at = 0x7FFFFFFF;
        for (int i = n8 * 8 + t; i < size; i += 1024)
            if (half_bits_to_float(x[i]) == most) {
                at = i;
                break;
            }
        for (int g = t + kPieces * 1024; g < n8; g += 1024)
            at = min(at, first_equal(x8[g], most, g * 8));
        if (n8 > 0) {
#pragma unroll
            for (int p = 0; p < kPieces; ++p)
                at = min(at, first_equal(v[p], most, min(t + p * 1024, n8 - 1) * 8));
        }
        if (at != 0x7FFFFFFF)
            atomicMin(si, at);
    }
    __syncthreads();
    const int best = si[0];
    return best == 0x7FFFFFFF ? 0 : best;
}

#endif // __HIPCC__


} // namespace l2
