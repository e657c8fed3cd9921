// The fp32 InnerProduct of the parity mode: y = float(sum_i double(x_i) *
// double(w_i) + double(b)), every output's products added one after another
// in increasing i, then the bias, then one rounding to float.
//
// The products of two floats are exact in double, so each step rounds only
// the running sum, and the result is the same bit for bit as any evaluation
// that adds the same exact products in the same order and rounds the same
// way: the CPU oracle's double-accumulated y = W x + b, W [out][in] row-major.
// The reference's InnerProduct is ncnn's (seedvr2_dit_block.cpp:28-56 creates
// it), which accumulates in float in an order not known here (ncnn is not in
// the reference tree): against it this product is pinned by the closed form
// y = W x + b only, not bit for bit.
//
// Two forms of the same arithmetic:
//   * tiled (rows > 16): v_mfma_f64_16x16x4_f64.  The instruction adds its
//     four products to an accumulator one after another in increasing k, each
//     a fused multiply-add with its own rounding (tests/test_gpu_exact.py
//     pins the product bit for bit), so it is the same sum as a chain of
//     scalar ones.  A lane supplies two doubles for 16 multiply-adds where
//     the VALU form, an 8 x 4 block a thread, read 12 doubles of LDS for 32:
//     LDS reads bounded that one at 25 TFLOP/s;
//   * few rows (rows <= 16, e.g. the DiT's one-row time MLP): one one-wave
//     workgroup per 16 output columns and one such MFMA tile, so a wide
//     product spreads over many CUs; chunks of 64 k, four of them in flight.
#include "sv2_internal.h"

namespace sv2
{
namespace
{

typedef __attribute__((ext_vector_type(4))) double d4;

constexpr int kBN = 64;        // output columns per workgroup
constexpr int kBK = 32;        // k per LDS stage
constexpr int kStride = 36;    // floats per staged row: 32 + 4, 16 consecutive rows on distinct banks
constexpr int kFill = 1024;    // workgroups of 64 rows from which 64-row tiles are taken

// One workgroup of four waves per BM x 64 tile of y, wave (r, c) = (wave / 2,
// wave % 2) a (BM / 2) x 32 block.  A stage of 32 k is held in LDS as fp32 in
// the order an MFMA lane consumes it: lane group q = lane / 16 multiplies k =
// 4 s + q at step s, so k sits at position 8 (k % 4) + k / 4 of its row and a
// lane's eight steps are two 16-byte reads.  The next stage is loaded into
// registers while the current one is multiplied.
//
// Bound by the fp64 matrix rate (45 to 47 TFLOP/s measured with nothing but
// this instruction, two waves or more per SIMD; one wave per SIMD gives 34,
// hence the small tiles).
template <int BM>
__global__ __launch_bounds__(256) void gemm_f32_exact_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ y,
                                                             int rows, int in, int out)
{
    constexpr int kMT = BM / 32;       // 16-row tiles per wave
    constexpr int kXQ = BM * kBK / 4 / 256; // float4 of x per thread and stage
    constexpr int kWQ = kBN * kBK / 4 / 256;
    __shared__ __attribute__((aligned(16))) float xs[2][BM * kStride];
    __shared__ __attribute__((aligned(16))) float ws[2][kBN * kStride];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int lr = lane & 15;
    const int lq = lane >> 4;
    // the row bands of one column tile run side by side and share its W rows
    const long long id = static_cast<long long>(blockIdx.y) * gridDim.x + blockIdx.x;
    const long long row0 = id % gridDim.y * BM;
    const long long col0 = id / gridDim.y * kBN;
    const bool quads = (in & 3) == 0 && ((reinterpret_cast<size_t>(x) | reinterpret_cast<size_t>(w)) & 15) == 0;

    // thread: k 4 (tid % 8) .. + 3 of rows tid / 8 + 32 i.  Values past the
    // edges are zero (their products are +0 and leave the sums unchanged)
    const int kq = tid & 7;
    const int sr = tid >> 3;
    float4 xv[kXQ], wv[kWQ];
    auto load1 = [&](const float* base, long long row, long long limit, int k) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < limit && k < in)
        {
            const float* p = base + row * in + k;
            if (quads)
                return *reinterpret_cast<const float4*>(p);
            v.x = p[0];
            v.y = k + 1 < in ? p[1] : 0.f;
            v.z = k + 2 < in ? p[2] : 0.f;
            v.w = k + 3 < in ? p[3] : 0.f;
        }
        return v;
    };
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kXQ; i++)
            xv[i] = load1(x, row0 + sr + 32 * i, rows, k0 + 4 * kq);
#pragma unroll
        for (int i = 0; i < kWQ; i++)
            wv[i] = load1(w, col0 + sr + 32 * i, out, k0 + 4 * kq);
    };
    auto put = [&](float* dst, const float4& v) {
        dst[0] = v.x;
        dst[8] = v.y;
        dst[16] = v.z;
        dst[24] = v.w;
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kXQ; i++)
            put(&xs[buf][(sr + 32 * i) * kStride + kq], xv[i]);
#pragma unroll
        for (int i = 0; i < kWQ; i++)
            put(&ws[buf][(sr + 32 * i) * kStride + kq], wv[i]);
    };

    const int wr = (wave >> 1) * (BM / 2);
    const int wc = (wave & 1) * 32;
    d4 acc[kMT][2];
#pragma unroll
    for (int i = 0; i < kMT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
            acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

    const int nk = (in + kBK - 1) / kBK;
    load(0);
    store(0);
    __syncthreads();
    for (int s = 0; s < nk; s++)
    {
        const int buf = s & 1;
        if (s + 1 < nk)
            load((s + 1) * kBK);
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            float4 a[kMT], b[2];
#pragma unroll
            for (int i = 0; i < kMT; i++)
                a[i] = *reinterpret_cast<const float4*>(&xs[buf][(wr + 16 * i + lr) * kStride + 8 * lq + 4 * h]);
#pragma unroll
            for (int j = 0; j < 2; j++)
                b[j] = *reinterpret_cast<const float4*>(&ws[buf][(wc + 16 * j + lr) * kStride + 8 * lq + 4 * h]);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < kMT; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            static_cast<double>((&a[i].x)[e]), static_cast<double>((&b[j].x)[e]), acc[i][j], 0, 0, 0);
        }
        // the other buffer's readers passed the last barrier
        if (s + 1 < nk)
            store(buf ^ 1);
        __syncthreads();
    }

    // register e of a tile: row 4 e + lane / 16, column lane % 16
#pragma unroll
    for (int j = 0; j < 2; j++)
    {
        const long long c = col0 + wc + 16 * j + lr;
        if (c >= out)
            continue;
        const double bv = bias ? static_cast<double>(bias[c]) : 0.0;
#pragma unroll
        for (int i = 0; i < kMT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++)
            {
                const long long r = row0 + wr + 16 * i + 4 * e + lq;
                if (r < rows)
                    y[r * out + c] = static_cast<float>(acc[i][j][e] + bv);
            }
    }
}

constexpr int kRowsSmall = 16; // the few-rows form handles up to this many rows
constexpr int kCols = 16;      // output columns per few-rows workgroup (one wave)
constexpr int kChunk = 64;     // k per chunk of the few-rows form
constexpr int kAhead = 4;      // chunks in flight
constexpr int kChunkStride = kChunk + 4;

// One wave: one 16 x 16 MFMA tile, rows of x by 16 output columns.  Lane l
// loads k 16 (l % 4) .. + 15 of row l / 4 of a chunk, four chunks ahead, into
// registers; a chunk goes through the wave's LDS into the lane order of the
// MFMA (k at position 16 (k % 4) + k / 4 of its row).  A workgroup is one
// wave, whose LDS operations complete in order: no barrier.
//
// An output's 2560 sums are one chain of 640 dependent MFMAs, which bounds the
// DiT's square time product (2560 -> 2560, one row); the wide one (2560 ->
// 15360) is the stream of its 157 MB of weights.
__global__ __launch_bounds__(64) void gemv_f32_exact_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ bias, float* __restrict__ y,
                                                            int rows, int in, int out)
{
    __shared__ __attribute__((aligned(16))) float wt[kCols * kChunkStride];
    __shared__ __attribute__((aligned(16))) float xt[kRowsSmall * kChunkStride];
    const int lane = threadIdx.x;
    const int lr = lane & 15;
    const int lq = lane >> 4;
    const int col0 = blockIdx.x * kCols;
    const int sr = lane >> 2;
    const int sk = (lane & 3) * 16;
    const bool w_ok = col0 + sr < out;
    const bool x_ok = sr < rows;
    const float* wp = w + static_cast<long long>(w_ok ? col0 + sr : 0) * in;
    const float* xp = x + static_cast<long long>(x_ok ? sr : 0) * in;
    const bool quads = (in & 3) == 0 && ((reinterpret_cast<size_t>(x) | reinterpret_cast<size_t>(w)) & 15) == 0;

    // values past the edges are zero: their products are +0 and the running
    // sums, which start at +0, stay what they were
    auto load = [&](const float* p, bool ok, int k0, float4 (&v)[4]) {
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            const int k = k0 + sk + 4 * e;
            v[e] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!ok || k >= in)
                continue;
            if (quads)
            {
                v[e] = *reinterpret_cast<const float4*>(p + k);
                continue;
            }
            v[e].x = p[k];
            v[e].y = k + 1 < in ? p[k + 1] : 0.f;
            v[e].z = k + 2 < in ? p[k + 2] : 0.f;
            v[e].w = k + 3 < in ? p[k + 3] : 0.f;
        }
    };
    auto put = [&](float* dst, const float4 (&v)[4]) {
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            float* d = dst + (sk >> 2) + e;
            d[0] = v[e].x;
            d[16] = v[e].y;
            d[32] = v[e].z;
            d[48] = v[e].w;
        }
    };

    d4 acc = {0.0, 0.0, 0.0, 0.0};
    float4 wv[kAhead][4], xv[kAhead][4];
#pragma unroll
    for (int a = 0; a < kAhead; a++)
    {
        load(wp, w_ok, a * kChunk, wv[a]);
        load(xp, x_ok, a * kChunk, xv[a]);
    }
    for (int k0 = 0; k0 < in; k0 += kAhead * kChunk)
    {
#pragma unroll
        for (int a = 0; a < kAhead; a++)
        {
            // chunks past the last are zero: their products change nothing
            put(&wt[sr * kChunkStride], wv[a]);
            put(&xt[sr * kChunkStride], xv[a]);
            __builtin_amdgcn_wave_barrier();
            load(wp, w_ok, k0 + (a + kAhead) * kChunk, wv[a]);
            load(xp, x_ok, k0 + (a + kAhead) * kChunk, xv[a]);
            float4 wf[4], xf[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
            {
                wf[e] = *reinterpret_cast<const float4*>(&wt[lr * kChunkStride + 16 * lq + 4 * e]);
                xf[e] = *reinterpret_cast<const float4*>(&xt[lr * kChunkStride + 16 * lq + 4 * e]);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < 16; s++)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>((&xf[s >> 2].x)[s & 3]),
                                                           static_cast<double>((&wf[s >> 2].x)[s & 3]), acc, 0, 0, 0);
        }
    }
    const int c = col0 + lr;
    if (c >= out)
        return;
    const double bv = bias ? static_cast<double>(bias[c]) : 0.0;
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        const int r = 4 * e + lq;
        if (r < rows)
            y[static_cast<long long>(r) * out + c] = static_cast<float>(acc[e] + bv);
    }
}

} // namespace

int gemm_f32_exact(hipStream_t stream, int rows, int in, int out, const float* x, const float* w, const float* bias,
                   float* y)
{
    if (rows < 0 || in <= 0 || out <= 0)
        return set_error(SV2_EINVAL, "inner product (fp32): bad shape");
    if (rows == 0)
        return SV2_OK;
    if (!x || !w || !y)
        return set_error(SV2_EINVAL, "inner product (fp32): null pointer");
    if (rows <= kRowsSmall)
    {
        hipLaunchKernelGGL(gemv_f32_exact_kernel, dim3(static_cast<unsigned>((out + kCols - 1) / kCols)), dim3(64), 0,
                           stream, x, w, bias, y, rows, in, out);
        const hipError_t err = hipGetLastError();
        return err == hipSuccess ? SV2_OK : hip_error(err, "gemv_f32_exact_kernel launch");
    }
    const unsigned bands = (static_cast<unsigned>(rows) + 63u) / 64u;
    const unsigned cols = (static_cast<unsigned>(out) + kBN - 1) / kBN;
    if (bands > 65535u)
        return set_error(SV2_EUNSUPPORTED, "inner product (fp32): too many rows");
    // 32-row tiles where 64-row ones would give few workgroups per CU
    if (static_cast<long long>(bands) * cols >= kFill)
        hipLaunchKernelGGL(gemm_f32_exact_kernel<64>, dim3(cols, bands), dim3(256), 0, stream, x, w, bias, y, rows,
                           in, out);
    else
        hipLaunchKernelGGL(gemm_f32_exact_kernel<32>, dim3(cols, (static_cast<unsigned>(rows) + 31u) / 32u), dim3(256),
                           0, stream, x, w, bias, y, rows, in, out);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? SV2_OK : hip_error(err, "gemm_f32_exact_kernel launch");
}

} // namespace sv2

extern "C" int sv2_inner_product_f32(const float* x, const float* w, const float* bias, float* y, int rows, int in,
                                     int out, void* stream)
try
{
    return sv2::gemm_f32_exact(static_cast<hipStream_t>(stream), rows, in, out, x, w, bias, y);
}
catch (...)
{
    return sv2::caught_exception("sv2_inner_product_f32");
}
