// The Euler sampler around the DiT on the device (src/model/sampler.cpp and
// the latent preparation of src/core/engine.cpp of the reference): the
// condition latent, the 33-channel DiT input, classifier-free guidance with
// the standard-deviation rescale, and the Euler / v-lerp update.  Latents are
// fp32 [C][T][H][W] arrays; every operation is elementwise, in fp32 with the
// reference's operation order and no fused multiply-add, so the outputs equal
// the reference's bit for bit (the guidance rescale factor comes from double
// sums whose order differs from the reference's, within an ulp of it).
#include "sv2_internal.h"

#include <cmath>

// Every float expression here is evaluated as written: no contraction into
// fused multiply-adds, on the device and on the host.
#pragma clang fp contract(off)

namespace sv2
{
namespace
{

constexpr int kThreads = 256;
constexpr int kSumThreads = 1024;   // of the guidance with statistics and of the rescale
constexpr int kReduceBlocks = 1024; // at most: partial sums of the guidance statistics
constexpr int kScaleBlocks = 512;   // at most: blocks of the rescale, two per CU
static_assert(kReduceBlocks <= kSumThreads, "a thread of the rescale takes one block's partials");
static_assert(kSumThreads == 1024, "16 waves of four sums are one value a lane");

unsigned blocks_for(long long n)
{
    return static_cast<unsigned>((n + kThreads - 1) / kThreads);
}

int launch_status(const char* what)
{
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? SV2_OK : hip_error(err, what);
}

// engine.cpp:106-122: (1 - ratio) * encoded + ratio * noise
__global__ __launch_bounds__(kThreads) void condition_kernel(const float* a, const float* b, float* out,
                                                             long long count, float ratio)
{
    const long long i = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= count)
        return;
    const float wa = 1.0f - ratio;
    const float left = wa * a[i];
    const float right = ratio * b[i];
    out[i] = left + right;
}

// Four consecutive fp32 elements of an array of any float alignment.
typedef __attribute__((ext_vector_type(4), aligned(4))) float f4;

// A thread takes four consecutive elements: the arrays stream in 16-byte
// accesses, and a launch's blocks fall to a quarter.
unsigned blocks_for_quads(long long n)
{
    return blocks_for((n + 3) / 4);
}

// engine.cpp:125-149: channels 0-15 the latent, 16-31 the condition, 32 ones.
// Channel-major ([16][tokens] sources into [33][tokens], the CPU engine): the
// output is the latent, the condition and a channel of ones one after the
// other, copied in quads (no channel index: with one 64-bit division an
// element the 720p clip's input took 7.5 us).
__global__ __launch_bounds__(kThreads) void dit_input_kernel(const float* latent, const float* condition, float* out,
                                                             long long tokens)
{
    const long long i = 4 * (static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x);
    const long long n = 16 * tokens; // a multiple of four: no quad crosses a source
    if (i < 2 * n)
    {
        const float* src = i < n ? latent + i : condition + (i - n);
        *reinterpret_cast<f4*>(out + i) = *reinterpret_cast<const f4*>(src);
        return;
    }
    for (long long k = i; k < min(i + 4, 33 * tokens); k++)
        out[k] = 1.0f;
}

// Token-major: [tokens][16] sources into [tokens][33] (sampler.cpp:337-357).
__global__ __launch_bounds__(kThreads) void dit_input_tokens_kernel(const float* latent, const float* condition,
                                                                    float* out, long long tokens)
{
    const long long i = static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= 33 * tokens)
        return;
    const long long t = i / 33;
    const long long c = i - t * 33;
    out[i] = c < 16 ? latent[t * 16 + c] : (c < 32 ? condition[t * 16 + c - 16] : 1.0f);
}

// sampler.cpp:217-218: neg + scale * (pos - neg)
__device__ inline float guide(float p, float n, float scale)
{
    const float diff = p - n;
    const float scaled = scale * diff;
    return n + scaled;
}

// Grid-stride: a launch holds at most 2^32 threads, counts are not bounded by it.
__global__ __launch_bounds__(kThreads) void cfg_kernel(const float* pos, const float* neg, float* out,
                                                       long long count, float scale)
{
    const long long stride = 4LL * gridDim.x * kThreads;
    for (long long i = 4 * (static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x); i < count; i += stride)
    {
        if (i + 4 <= count)
        {
            const f4 p = *reinterpret_cast<const f4*>(pos + i);
            const f4 n = *reinterpret_cast<const f4*>(neg + i);
            f4 o;
            for (int e = 0; e < 4; e++)
                o[e] = guide(p[e], n[e], scale);
            *reinterpret_cast<f4*>(out + i) = o;
            continue;
        }
        for (long long k = i; k < count; k++)
            out[k] = guide(pos[k], neg[k], scale);
    }
}

// Lane l of the wave gets the sum over its lanes of v[l % 4]: two halving
// exchanges, then four of one value (a sum of each value by itself takes 24).
__device__ inline double wave_sum4(const double (&v)[4], int lane)
{
    const bool odd = lane & 1;
    const bool high = lane & 2;
    const double a = (odd ? v[1] : v[0]) + __shfl_xor(odd ? v[0] : v[1], 1);
    const double b = (odd ? v[3] : v[2]) + __shfl_xor(odd ? v[2] : v[3], 1);
    double s = (high ? b : a) + __shfl_xor(high ? a : b, 2);
#pragma unroll
    for (int d = 4; d < 64; d <<= 1)
        s += __shfl_xor(s, d);
    return s;
}

// The same over a block of kSumThreads, in every wave: 16 waves of 4 sums are
// one value a lane.
__device__ inline double block_sum4(const double (&v)[4], double* red)
{
    const int lane = threadIdx.x & 63;
    const double s = wave_sum4(v, lane);
    if (lane < 4)
        red[4 * (threadIdx.x >> 6) + lane] = s;
    __syncthreads();
    double t = red[lane];
#pragma unroll
    for (int d = 4; d < 64; d <<= 1)
        t += __shfl_xor(t, d);
    return t;
}

// With the rescale each block also writes its double sums of pos, pos^2, out,
// out^2 (grid-stride over the quads, fixed order).  Blocks of 1024: a quad a
// thread fills a CU and leaves few partials for the next kernel to add (338 at
// the 720p clip, where blocks of 256 left the most there may be, 1024).
__global__ __launch_bounds__(kSumThreads) void cfg_sums_kernel(const float* pos, const float* neg, float* out,
                                                               long long count, float scale, double* partial)
{
    __shared__ double red[64];
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    auto add = [&](float p, float o) {
        v[0] += p;
        v[1] += static_cast<double>(p) * p;
        v[2] += o;
        v[3] += static_cast<double>(o) * o;
    };
    const long long stride = 4LL * gridDim.x * kSumThreads;
    for (long long i = 4 * (static_cast<long long>(blockIdx.x) * kSumThreads + threadIdx.x); i < count; i += stride)
    {
        if (i + 4 <= count)
        {
            const f4 p = *reinterpret_cast<const f4*>(pos + i);
            const f4 n = *reinterpret_cast<const f4*>(neg + i);
            f4 o;
            for (int e = 0; e < 4; e++)
            {
                o[e] = guide(p[e], n[e], scale);
                add(p[e], o[e]);
            }
            *reinterpret_cast<f4*>(out + i) = o;
            continue;
        }
        for (long long k = i; k < count; k++)
        {
            const float p = pos[k];
            const float o = guide(p, neg[k], scale);
            out[k] = o;
            add(p, o);
        }
    }
    const double s = block_sum4(v, red);
    if (threadIdx.x < 4)
        partial[static_cast<long long>(blockIdx.x) * 4 + threadIdx.x] = s;
}

// sampler.cpp:41-62 (unbiased standard deviation from the sums) and :219-235:
// factor = rescale * std(pos) / std(out) + (1 - rescale) when std(out) > 0,
// then the outputs times it.  Every block forms the factor itself: thread t
// takes the partials of block t (at most kReduceBlocks of them), the sums
// follow in a fixed order, so the factor is the same in all blocks and does not
// depend on scheduling.  A thread's first quad is requested before that.
//
// Bound by launch and the chain partials - sums - factor - product.  Guidance
// and rescale together, in a graph: 9.8 us at the 720p clip, 6.0 at the
// smallest.  With 256 blocks of 256 threads, each adding 1024 partials through
// an eight-level tree of barriers before it streamed, 12.8 and 6.3; with 5400
// blocks and a launch of its own for the factor, 11.7 and 7.3.
__global__ __launch_bounds__(kSumThreads) void cfg_scale_kernel(const double* partial, int nblocks, float* out,
                                                                long long count, float rescale)
{
    __shared__ double red[64];
    __shared__ float factor[2];
    const int tid = threadIdx.x;
    long long i = 4 * (static_cast<long long>(blockIdx.x) * kSumThreads + tid);
    f4 o = {0.f, 0.f, 0.f, 0.f};
    if (i + 4 <= count)
        o = *reinterpret_cast<const f4*>(out + i);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (tid < nblocks)
        for (int k = 0; k < 4; k++)
            v[k] = partial[4 * tid + k];
    const double s = block_sum4(v, red);
    if (tid < 64)
    {
        const double sp = __shfl(s, 0), spp = __shfl(s, 1), so = __shfl(s, 2), soo = __shfl(s, 3);
        double std_pos = 0.0, std_out = 0.0;
        if (count > 1)
        {
            const double n = static_cast<double>(count);
            std_pos = sqrt(fmax(0.0, (spp - sp * sp / n) / (n - 1)));
            std_out = sqrt(fmax(0.0, (soo - so * so / n) / (n - 1)));
        }
        if (tid == 0)
        {
            const bool apply = std_out > 0.0;
            factor[0] = apply ? static_cast<float>(static_cast<double>(rescale) * std_pos / std_out +
                                                   static_cast<double>(1.0f - rescale))
                              : 1.0f;
            factor[1] = apply ? 1.0f : 0.0f;
        }
    }
    __syncthreads();
    if (factor[1] == 0.0f)
        return;
    const float f = factor[0];
    const long long stride = 4LL * gridDim.x * kSumThreads;
    for (; i + 4 <= count; i += stride)
    {
        for (int e = 0; e < 4; e++)
            o[e] *= f;
        *reinterpret_cast<f4*>(out + i) = o;
        if (i + stride + 4 <= count)
            o = *reinterpret_cast<const f4*>(out + i + stride);
    }
    for (long long k = i; k < count; k++)
        out[k] *= f;
}

// sampler.cpp:253-263: x0 = x - bt * pred, xT = x + at * pred,
// out = as * x0 + bs * xT (endpoint: bs = 0, as = 1 gives out = x0 exactly).
__device__ inline float euler(float p, float x, float bt, float at, float as, float bs, int endpoint)
{
    const float x0 = x - bt * p;
    if (endpoint)
        return x0;
    const float xT = x + at * p;
    const float left = as * x0;
    const float right = bs * xT;
    return left + right;
}

__global__ __launch_bounds__(kThreads) void euler_kernel(const float* pred, const float* cur, float* out,
                                                         long long count, float bt, float at, float as, float bs,
                                                         int endpoint)
{
    const long long i = 4 * (static_cast<long long>(blockIdx.x) * kThreads + threadIdx.x);
    if (i + 4 <= count)
    {
        const f4 p = *reinterpret_cast<const f4*>(pred + i);
        const f4 x = *reinterpret_cast<const f4*>(cur + i);
        f4 o;
        for (int e = 0; e < 4; e++)
            o[e] = euler(p[e], x[e], bt, at, as, bs, endpoint);
        *reinterpret_cast<f4*>(out + i) = o;
        return;
    }
    for (long long k = i; k < count; k++)
        out[k] = euler(pred[k], cur[k], bt, at, as, bs, endpoint);
}

int check_count(long long count, const char* what)
{
    if (count < 0 || count / kThreads >= (1LL << 31))
        return set_error(SV2_EINVAL, std::string(what) + ": bad element count");
    return SV2_OK;
}

} // namespace
} // namespace sv2

extern "C" {

int sv2_euler_timesteps(int steps, float* out)
try
{
    if (!out)
        return sv2::set_error(SV2_EINVAL, "sv2_euler_timesteps: null output");
    // EulerSampler::EulerSampler (sampler.cpp:181-187): at least one step
    const int n = steps < 1 ? 1 : steps;
    for (int i = 0; i < n; i++)
        out[i] = 1000.0f * (1.0f - static_cast<float>(i) / n);
    return n;
}
catch (...)
{
    return sv2::caught_exception("sv2_euler_timesteps");
}

float sv2_condition_ratio(float noise_scale, int frames, int height, int width)
{
    // transformed_condition_timestep (engine.cpp:79-92) over the encoded
    // latent's [T][H][W], divided by 1000 as make_condition_latent does
    // (engine.cpp:110): the resolution-dependent shift of the noise level.
    const float timestep = noise_scale * 1000.0f;
    if (timestep == 0.0f)
        return 0.0f;
    const float f = static_cast<float>((frames - 1) * 4 + 1);
    const float h = static_cast<float>(height * 8);
    const float w = static_cast<float>(width * 8);
    const float x1 = 256.0f * 256.0f * 37.0f;
    const float x2 = 1280.0f * 720.0f * 145.0f;
    const float shift = 1.0f + (h * w * f - x1) * (5.0f - 1.0f) / (x2 - x1);
    const float normalized = timestep / 1000.0f;
    return 1000.0f * shift * normalized / (1.0f + (shift - 1.0f) * normalized) / 1000.0f;
}

int sv2_make_condition(const float* encoded, const float* noise, float* out, int64_t count, float ratio,
                       void* stream)
try
{
    using namespace sv2;
    int rc = check_count(count, "sv2_make_condition");
    if (rc != SV2_OK)
        return rc;
    if (count == 0)
        return SV2_OK;
    if (!encoded || !noise || !out)
        return set_error(SV2_EINVAL, "sv2_make_condition: null pointer");
    hipLaunchKernelGGL(condition_kernel, dim3(blocks_for(count)), dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                       encoded, noise, out, static_cast<long long>(count), ratio);
    return launch_status("condition_kernel launch");
}
catch (...)
{
    return sv2::caught_exception("sv2_make_condition");
}

int sv2_make_dit_input(const float* latent, const float* condition, float* out, int64_t tokens, int channel_major,
                       void* stream)
try
{
    using namespace sv2;
    int rc = check_count(33 * tokens, "sv2_make_dit_input");
    if (rc != SV2_OK)
        return rc;
    if (tokens == 0)
        return SV2_OK;
    if (!latent || !condition || !out)
        return set_error(SV2_EINVAL, "sv2_make_dit_input: null pointer");
    if (channel_major)
        hipLaunchKernelGGL(dit_input_kernel, dim3(blocks_for_quads(33 * tokens)), dim3(kThreads), 0,
                           static_cast<hipStream_t>(stream), latent, condition, out, static_cast<long long>(tokens));
    else
        hipLaunchKernelGGL(dit_input_tokens_kernel, dim3(blocks_for(33 * tokens)), dim3(kThreads), 0,
                           static_cast<hipStream_t>(stream), latent, condition, out, static_cast<long long>(tokens));
    return launch_status("dit_input_kernel launch");
}
catch (...)
{
    return sv2::caught_exception("sv2_make_dit_input");
}

int64_t sv2_cfg_workspace_size(int64_t count)
try
{
    (void)count;
    // partial sums of every reduction block (and 256 bytes kept from when the
    // factor had a place of its own)
    return static_cast<int64_t>(sv2::kReduceBlocks) * 4 * sizeof(double) + 256;
}
catch (...)
{
    return sv2::caught_exception("sv2_cfg_workspace_size");
}

int sv2_apply_cfg(const float* positive, const float* negative, float* out, int64_t count, float scale,
                  float rescale, void* workspace, size_t workspace_bytes, void* stream_ptr)
try
{
    using namespace sv2;
    int rc = check_count(count, "sv2_apply_cfg");
    if (rc != SV2_OK)
        return rc;
    if (count == 0)
        return SV2_OK;
    if (!positive || !negative || !out)
        return set_error(SV2_EINVAL, "sv2_apply_cfg: null pointer");
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    if (rescale == 0.0f)
    {
        const int nb = static_cast<int>(std::min<long long>(((count + 3) / 4 + kThreads - 1) / kThreads, 1LL << 20));
        hipLaunchKernelGGL(cfg_kernel, dim3(nb), dim3(kThreads), 0, stream, positive, negative, out,
                           static_cast<long long>(count), scale);
        return launch_status("cfg_kernel launch");
    }
    if (!workspace || static_cast<int64_t>(workspace_bytes) < sv2_cfg_workspace_size(count))
        return set_error(SV2_EINVAL, "sv2_apply_cfg: the rescale needs sv2_cfg_workspace_size bytes of workspace");
    double* partial = static_cast<double*>(workspace);
    const long long blocks = ((count + 3) / 4 + kSumThreads - 1) / kSumThreads;
    const int nb = static_cast<int>(std::min<long long>(blocks, kReduceBlocks));
    hipLaunchKernelGGL(cfg_sums_kernel, dim3(nb), dim3(kSumThreads), 0, stream, positive, negative, out,
                       static_cast<long long>(count), scale, partial);
    if ((rc = launch_status("cfg_sums_kernel launch")) != SV2_OK)
        return rc;
    const int ns = static_cast<int>(std::min<long long>(blocks, kScaleBlocks));
    hipLaunchKernelGGL(cfg_scale_kernel, dim3(ns), dim3(kSumThreads), 0, stream, partial, nb, out,
                       static_cast<long long>(count), rescale);
    return launch_status("cfg_scale_kernel launch");
}
catch (...)
{
    return sv2::caught_exception("sv2_apply_cfg");
}

int sv2_euler_step(const float* prediction, const float* current, float* out, int64_t count, float timestep,
                   float next_timestep, void* stream)
try
{
    using namespace sv2;
    int rc = check_count(count, "sv2_euler_step");
    if (rc != SV2_OK)
        return rc;
    if (count == 0)
        return SV2_OK;
    if (!prediction || !current || !out)
        return set_error(SV2_EINVAL, "sv2_euler_step: null pointer");
    // EulerSampler::step_to (sampler.cpp:253-256)
    const float bt = timestep / 1000.0f;
    const float at = 1.0f - bt;
    const float bs = std::fmin(std::fmax(next_timestep / 1000.0f, 0.0f), 1.0f);
    const float as = 1.0f - bs;
    hipLaunchKernelGGL(euler_kernel, dim3(blocks_for_quads(count)), dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                       prediction, current, out, static_cast<long long>(count), bt, at, as, bs, 0);
    return launch_status("euler_kernel launch");
}
catch (...)
{
    return sv2::caught_exception("sv2_euler_step");
}

int sv2_euler_endpoint(const float* prediction, const float* current, float* out, int64_t count, float timestep,
                       void* stream)
try
{
    using namespace sv2;
    int rc = check_count(count, "sv2_euler_endpoint");
    if (rc != SV2_OK)
        return rc;
    if (count == 0)
        return SV2_OK;
    if (!prediction || !current || !out)
        return set_error(SV2_EINVAL, "sv2_euler_endpoint: null pointer");
    // EulerSampler::endpoint (sampler.cpp:280-282)
    const float bt = timestep / 1000.0f;
    hipLaunchKernelGGL(euler_kernel, dim3(blocks_for_quads(count)), dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                       prediction, current, out, static_cast<long long>(count), bt, 0.0f, 1.0f, 0.0f, 1);
    return launch_status("euler_kernel launch");
}
catch (...)
{
    return sv2::caught_exception("sv2_euler_endpoint");
}

} // extern "C"
