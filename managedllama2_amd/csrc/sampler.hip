// The stochastic sampler's modules (src/SoftmaxLogits.cs, Sort.cs,
// CumulativeSum.cs, SampleTopP.cs; kernels native/softmax_logits_kernel.cu,
// sort_kernel.cu, cumulative_sum_kernel.cu, sample_top_p_kernel.cu) and the
// whole stochastic branch of Sampler.Sample (src/Sampler.cs:48-67).
#include "sampler_kernels.hpp"

namespace l2 {

int check_sampler_size(const char* fn, int size)
{
    L2_CHECK(size > 0, "%s: size=%d must be positive", fn, size);
    if (size > LLAMA2_MAX_SAMPLER_SIZE)
        return fail(LLAMA2_ERR_UNSUPPORTED, "%s: size=%d exceeds %d", fn, size, LLAMA2_MAX_SAMPLER_SIZE);
    return LLAMA2_OK;
}

int check_temperature(const char* fn, float temperature)
{
    L2_CHECK(temperature > 0.0f, "%s: temperature=%g must be positive (temperature 0 is the argmax branch)", fn,
             static_cast<double>(temperature));
    return LLAMA2_OK;
}

static void launch_exp(const SampleArgs& a)
{
    const dim3 grid(kSampBlock / kExpShare + (a.state || a.host.state ? 1 : 0));
    if (sampler_chunks(a.size) == 4)
        hipLaunchKernelGGL(sampler_exp_kernel<4>, grid, dim3(kExpThreads), 0, ctx().stream, a);
    else
        hipLaunchKernelGGL(sampler_exp_kernel<8>, grid, dim3(kExpThreads), 0, ctx().stream, a);
}

static void launch_rank(const SampleArgs& a, uint16_t* keys, int* values, bool identity)
{
    const int tiles = ceil_div(a.size, kSampTile);
    const dim3 grid(tiles * (kSampTile / kSampRun));
    if (tiles <= kSampTiles / 2)
        hipLaunchKernelGGL(sampler_rank_kernel<kSampTiles / 2>, grid, dim3(kSampBlock), 0, ctx().stream, a, keys, values,
                           identity ? 1 : 0);
    else
        hipLaunchKernelGGL(sampler_rank_kernel<kSampTiles>, grid, dim3(kSampBlock), 0, ctx().stream, a, keys, values,
                           identity ? 1 : 0);
}

template <bool PICK>
static void launch_pick(const SampleArgs& a, const uint16_t* in, bool in_place)
{
    const int ch = sampler_chunks(a.size);
    const dim3 grid(in_place ? 1 : ceil_div(a.size, 64 * 8 * ch));
    if (ch == 4)
        hipLaunchKernelGGL((sampler_pick_kernel<4, PICK>), grid, dim3(kSampBlock), 0, ctx().stream, a, in);
    else
        hipLaunchKernelGGL((sampler_pick_kernel<8, PICK>), grid, dim3(kSampBlock), 0, ctx().stream, a, in);
}

template <bool PICK>
static void launch_one(const SampleArgs& a)
{
    if (a.size <= 8 * kSampBlock)
        hipLaunchKernelGGL((sampler_one_kernel<1, PICK>), dim3(1), dim3(kSampBlock), 0, ctx().stream, a);
    else
        hipLaunchKernelGGL((sampler_one_kernel<2, PICK>), dim3(1), dim3(kSampBlock), 0, ctx().stream, a);
}

int sample_enqueue(const char* name, const SampleArgs& args)
{
    if (!sample_sorts(args.top_p) && args.size <= kSampOneItems) {
        launch_one<true>(args);
        L2_LAUNCH_CHECK(name);
        return LLAMA2_OK;
    }
    SampleArgs a = args;
    SamplerScratch* s = a.s;
    if (!sample_sorts(a.top_p))
        a.head = -1;
    else if (a.size > kSampHeadItems)
        a.head = 0;
    launch_exp(a);
    hipLaunchKernelGGL(sampler_tile_kernel<TILE_EXPS>, dim3(ceil_div(a.size, kSampTile)), dim3(kTileThreads), 0,
                       ctx().stream, a, static_cast<const uint16_t*>(nullptr), static_cast<const int*>(nullptr),
                       a.head < 0 ? s->keys : a.head > 0 ? a.logits : nullptr);
    if (a.head >= 0)
        launch_rank(a, s->keys, a.indices, true);
    launch_pick<true>(a, s->keys, false);
    L2_LAUNCH_CHECK(name);
    return LLAMA2_OK;
}

} // namespace l2

using namespace l2;

#define L2_TRY(expr)          \
    do {                      \
        int rc_ = (expr);     \
        if (rc_ != LLAMA2_OK) \
            return rc_;       \
    } while (0)

extern "C" {

int llama2_softmax_logits(llama2_half* logits, int size, float temperature, int* indices)
{
    L2_REQUIRE_INIT();
    const char* fn = "llama2_softmax_logits";
    L2_CHECK(logits && indices, "%s: null pointer", fn);
    L2_TRY(check_sampler_size(fn, size));
    L2_TRY(check_temperature(fn, temperature));
    L2_CHECK(aligned(logits, 16) && aligned(indices, 16), "%s: logits and indices must be 16-byte aligned", fn);
    SampleArgs a{};
    a.logits = logits, a.indices = indices, a.size = size, a.temperature = temperature, a.s = ctx().sampler, a.head = -1;
    if (size <= kSampOneItems) {
        launch_one<false>(a);
        L2_LAUNCH_CHECK(fn);
        return LLAMA2_OK;
    }
    launch_exp(a);
    hipLaunchKernelGGL(sampler_tile_kernel<TILE_EXPS>, dim3(ceil_div(size, kSampTile)), dim3(kTileThreads), 0, ctx().stream,
                       a, static_cast<const uint16_t*>(nullptr), static_cast<const int*>(nullptr), logits);
    L2_LAUNCH_CHECK(fn);
    return LLAMA2_OK;
}

int llama2_sort(llama2_half* keys, int* values, int size)
{
    L2_REQUIRE_INIT();
    const char* fn = "llama2_sort";
    L2_CHECK(keys && values, "%s: null pointer", fn);
    L2_TRY(check_sampler_size(fn, size));
    L2_CHECK(aligned(keys, 16) && aligned(values, 16), "%s: keys and values must be 16-byte aligned", fn);
    SampleArgs a{};
    a.size = size, a.s = ctx().sampler;
    hipLaunchKernelGGL(sampler_tile_kernel<TILE_KEYS>, dim3(ceil_div(size, kSampTile)), dim3(kTileThreads), 0, ctx().stream,
                       a, keys, values, static_cast<uint16_t*>(nullptr));
    launch_rank(a, keys, values, false);
    L2_LAUNCH_CHECK(fn);
    return LLAMA2_OK;
}

int llama2_cumulative_sum(llama2_half* values, int size)
{
    L2_REQUIRE_INIT();
    const char* fn = "llama2_cumulative_sum";
    L2_CHECK(values, "%s: null pointer", fn);
    L2_TRY(check_sampler_size(fn, size));
    L2_CHECK(aligned(values, 16), "%s: values must be 16-byte aligned", fn);
    SampleArgs a{};
    a.logits = values, a.size = size;
    launch_pick<false>(a, values, true);
    L2_LAUNCH_CHECK(fn);
    return LLAMA2_OK;
}

int llama2_sample_top_p(const llama2_half* logits, const int* indices, int size, float threshold, int* result, int pos)
{
    L2_REQUIRE_INIT();
    const char* fn = "llama2_sample_top_p";
    L2_CHECK(logits && indices && result, "%s: null pointer", fn);
    L2_TRY(check_sampler_size(fn, size));
    L2_CHECK(pos >= 0, "%s: pos=%d is negative", fn, pos);
    L2_CHECK(aligned(logits, 16), "%s: logits must be 16-byte aligned", fn);
    if (sampler_chunks(size) == 4)
        hipLaunchKernelGGL(sample_top_p_kernel<4>, dim3(1), dim3(kSampBlock), 0, ctx().stream, logits, indices, size,
                           threshold, result, pos);
    else
        hipLaunchKernelGGL(sample_top_p_kernel<8>, dim3(1), dim3(kSampBlock), 0, ctx().stream, logits, indices, size,
                           threshold, result, pos);
    L2_LAUNCH_CHECK(fn);
    return LLAMA2_OK;
}

int llama2_sample(llama2_half* logits, int* indices, int size, float temperature, float top_p, float coin,
                  int* result, int pos)
{
    L2_REQUIRE_INIT();
    return sample_launch("llama2_sample", ctx().sampler, logits, indices, size, temperature, top_p, coin, result, pos,
                         false);
}

} // extern "C"

namespace l2 {

int sample_launch(const char* fn, SamplerScratch* scratch, uint16_t* logits, int* indices, int size, float temperature,
                  float top_p, float coin, int* result, int pos, bool token_only, const HostStep* host)
{
    L2_CHECK(logits && indices && result, "%s: null pointer", fn);
    L2_TRY(check_sampler_size(fn, size));
    L2_TRY(check_temperature(fn, temperature));
    L2_CHECK(pos >= 0, "%s: pos=%d is negative", fn, pos);
    L2_CHECK(aligned(logits, 16) && aligned(indices, 16), "%s: logits and indices must be 16-byte aligned", fn);
    SampleArgs a{};
    a.logits = logits, a.indices = indices, a.size = size, a.s = scratch;
    a.temperature = temperature, a.top_p = top_p, a.coin = coin, a.result = result, a.pos = pos;
    a.head = token_only ? 1 : 0;
    if (host)
        a.host = *host;
    return sample_enqueue(fn, a);
}

} // namespace l2
