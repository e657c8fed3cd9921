// fp16 InnerProducts of many rows on gfx950 MFMA, with the passes that follow
// them in the block folded in (the reference runs ncnn InnerProduct,
// seedvr2_dit_block.cpp:28-56 and :668-674, then separate SwiGLU and
// ada-residual passes, :1093-1112 and :807-825).
//
//   Y[m][n] = epilogue(sum_k X[m][k] * W[n][k])      X [M][K], W [N][K] fp16
//
// A 512-thread workgroup (8 waves, two per SIMD) computes tiles of MH x 128
// rows by NH x 128 columns on v_mfma_f32_16x16x32_f16; a wave's part of the
// 256 x 256 tile is 64 columns of each W half by 32 rows of each X half, 128
// fp32 accumulators a lane.  The product is computed transposed (W as the A
// operand), so a lane holds four consecutive columns of one output row.
//
// Fetch.  K moves in stages of 64 (whole 128-byte lines) through a ring of
// LDS slots (two 64 KB, three 48 KB or four 32 KB ones), by
// global_load_lds_dwordx4 alone: no register is held by a fetch.  A half-tile
// of a slot is refilled as soon as the phase after the one that read it, so
// fetches run 1.5 (256 x 256) to 3 stages ahead, and waits name the exact
// number of younger fetches.  16-byte chunk c of row r sits in slot
// c ^ ((r >> 1) & 7): the 16 rows an operand read takes fall on 16 different
// bank groups.
//
// Phases.  A stage is walked in quadrants (W half x X half), each a memory
// part (operand reads, fetches, waits) and 16 MFMAs, with a barrier after
// each.  The two waves of a SIMD belong to different groups, one slot apart:
// one group multiplies while the other one reads.
//
// Workgroups are persistent (one per CU) and take tiles in XCD-contiguous
// runs; the ring runs on across tiles, so a tile's first stages are in flight
// during the epilogue of the one before.  Outputs leave with non-temporal
// stores: written through the L2 they evict the operand panels (128 KB a tile
// and CU is the whole L2 of an XCD), and qkv at 21658 rows takes an eighth
// longer.
//
// What bounds it, 21658 rows in a block (MI355X, kernel trace, us; the library
// beside it, its separate SwiGLU pass after the +):
//   qkv 2560 -> 7680                   609 (1.40 PFLOP/s)   606
//   proj 2560 -> 2560 + residual       282                  281
//   gate/in 2560 -> 2 x 6912 + SwiGLU  1109                 1076 + 135
//   out 6912 -> 2560 + residual        620                  629
// The matrix cores are busy 71 to 77% of the cycles of a 256 x 256 launch, at
// 1.7 GHz: with all-zero operands, alone and back to back, the four take 434 /
// 215 / 773 / 512 us, with random ones 594 / 250 / 1062 / 605, where the clock
// drops under the matrix cores' power.  The rest is LDS bandwidth (192 KB of
// operand reads and 64 KB of fetch a 256 x 256 stage, 2048 cycles at 128
// B/clk, as many as its MFMAs take).  A 128 x 128 tile reads three bytes of LDS
// where the large one reads two, and runs at 0.39 us a stage against 0.24 us
// for a quarter of the large one's; it is there for the products that would
// leave CUs idle.  `KS` is the 128 x 128 tile with a 64 x 64 part per wave: the
// two groups take one k-step of each stage each and add their sums at the end
// (reads a third less LDS than 64 x 32 parts do).
//
// Epilogues, in fp32 from the accumulators:
//   kGemmStore     Y = fp16(acc)
//   kGemmResidual  Y = fp16(acc * gate + R + bias), one rounding; `rounded`:
//                  fp16((fp16(acc) + bias) * gate + R), the unfused passes'
//                  order (gate and bias optional)
//   kGemmSwiGLU    two weight matrices, gate W and value W2, both [N][K]: the
//                  W halves of a tile are the gate and value rows of the same
//                  128 columns, Y = fp16(g / (1 + exp(-g)) * u); `rounded`: g
//                  and u rounded to fp16 first, as the separate products are
#include "sv2_internal.h"
#include <algorithm>
#include <climits>
#include <type_traits>

#pragma clang fp contract(off)

namespace sv2
{
namespace
{

typedef __attribute__((ext_vector_type(8))) _Float16 h8;
typedef __attribute__((ext_vector_type(4))) _Float16 h4;
typedef __attribute__((ext_vector_type(4))) float f4;
typedef __attribute__((ext_vector_type(4), aligned(4))) float f4u; // gate and bias: any float alignment
typedef __attribute__((ext_vector_type(4))) unsigned u4;

constexpr int kThreads = 512;      // 8 waves, two per SIMD
constexpr int kHalf = 128;         // rows of one operand half-tile
constexpr int kBK = 64;            // K per stage: whole 128-byte lines of every row
constexpr int kRowBytes = kBK * 2; // 128
constexpr int kHalfBytes = kHalf * kRowBytes; // 16 KB
constexpr int kEpiWave = 16 * 128; // bytes of one wave's epilogue staging: 16 rows of 64 fp16
constexpr int kEpiBytes = 8 * kEpiWave;
constexpr int kMaxLds = 160 * 1024;
constexpr int kCus = 256;            // compute units of one MI355X
constexpr int kPreferRows = 256;    // fewer rows go to the library
constexpr int kTouchAhead = 3;      // stages before a tile's end
constexpr float kLog2e = 1.4426950408889634f;

struct TileArgs
{
    const _Float16* x;  // [M][K]
    const _Float16* w;  // [N][K]
    const _Float16* w2; // SwiGLU: the value projection [N][K]
    _Float16* y;        // [M][N]
    const _Float16* r;  // residual [M][N]
    const float* bias;  // [N] or null
    const float* gate;  // [N] or null
    int m, n, k;
    int rounded;        // the product is rounded to fp16 before the epilogue
    int tiles_m;        // row bands
    int tiles_n;        // column tiles
    int total;          // tiles_m * tiles_n
    int group_m;        // row bands per tile group
};

// Stages an operand tile of MH (X) + NH (W) halves takes, and how many of
// them fit in LDS beside the epilogue staging.
template <int MH, int NH>
struct Shape
{
    static constexpr int kStageBytes = (MH + NH) * kHalfBytes;
    static constexpr int kFit = (kMaxLds - kEpiBytes) / kStageBytes;
    static constexpr int kSlots = kFit > 4 ? 4 : kFit;
    static constexpr int kLds = kSlots * kStageBytes + kEpiBytes;
    static_assert(kSlots >= 2 && kLds <= kMaxLds, "LDS of one gfx950 CU");
};

// 16 bytes per lane from global memory (uniform base + 32-bit lane offset)
// straight into LDS at lds + 16 * lane (lds wave-uniform, in M0; one wait
// state between the write of M0 and its use).  The compiler does not count
// these loads in its vmcnt waits; the loop waits for them itself.
__device__ inline void dma16(const char* base, unsigned voff, unsigned lds)
{
    const unsigned long long b = reinterpret_cast<unsigned long long>(base);
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(b));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(b >> 32));
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(static_cast<unsigned long long>(hi) << 32 | lo)
                 : "memory", "m0");
}

// The same with 4 bytes per lane, for its effect on the L2 alone: lds is a
// 256-byte sink.
__device__ inline void touch(const void* p, unsigned lds)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(p)
                 : "memory", "m0");
}

template <int N>
__device__ inline void wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt holds 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ inline void wait_lds()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// A wave's LDS operations complete in order; this keeps the compiler from
// reordering them.
__device__ inline void lds_order()
{
    asm volatile("" ::: "memory");
}

// A workgroup barrier without the waits of __syncthreads (the fetches in
// flight stay in flight); nothing is scheduled across it.
__device__ inline void bar()
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

__device__ inline float h2f(_Float16 v)
{
    return static_cast<float>(v);
}

__device__ inline float round16(float v)
{
    return static_cast<float>(static_cast<_Float16>(v));
}

// Tile id -> (row band, column tile): groups of group_m row bands, the bands
// of one column of tiles first.
__device__ inline void tile_at(const TileArgs& a, int id, int* tm, int* tn)
{
    const int per = a.group_m * a.tiles_n;
    const int grp = id / per;
    const int first = grp * a.group_m;
    const int rows = min(a.group_m, a.tiles_m - first);
    const int in = id - grp * per;
    *tn = in / rows;
    *tm = first + (in - *tn * rows);
}

// Waits until at most n fetches are outstanding; n one of the counts the
// pipeline's start and end meet (any other waits for all of them).
__device__ inline void wait_younger(int n)
{
    switch (n)
    {
    case 12: wait_vm<12>(); break;
    case 8: wait_vm<8>(); break;
    case 6: wait_vm<6>(); break;
    case 4: wait_vm<4>(); break;
    default: wait_vm<0>(); break;
    }
}

// Rounds and stores one wave's part of a tile: for W half h and X half j the
// lane holds rows row0 + 128 j + 16 b + lane % 16, columns col0 + 128 h +
// 16 t + 4 (lane / 16) .. + 3 of acc[h][j][t][b].  16 rows x 64 columns at a
// time go through `mine` (2 KB of LDS, this wave's own), 16-byte chunk c of
// row r in slot c ^ (r & 7), so that residual rows are read and output rows
// written as whole 128-byte lines.
//
// SwiGLU's silu: with `ROUNDED` expf and an IEEE divide, 2.5 fp32 ulps at most
// in all; else exp2 and the reciprocal, as the separate 16-bit pass has them
// (up to 8 ulps where the gate is large and negative: the fp32 rounding of the
// exponent, below the fp16 roundings of g and u that this form leaves out).
// Two bodies, not a branch per element: the first costs gate/in at 21658 rows
// 1166 us where the second takes 1107.
template <int MH, int NH, int EPI, bool ROUNDED>
__device__ __forceinline__ void epilogue(const TileArgs& a, f4 (&acc)[NH][MH][4][2], char* mine, int row0, int col0, int lane)
{
    constexpr bool kSw = EPI == kGemmSwiGLU;
    const int lr = lane & 15;
    const int lq = lane >> 4;
    const int rr = lane >> 3; // rows rr, rr + 8 of the line accesses
    const int cc = lane & 7;
    char* line[2];
    char* quad[4];
#pragma unroll
    for (int s = 0; s < 2; s++)
        line[s] = mine + (rr + 8 * s) * 128 + ((cc ^ (rr & 7)) << 4);
#pragma unroll
    for (int t = 0; t < 4; t++)
        quad[t] = mine + lr * 128 + (((2 * t + (lq >> 1)) ^ (lr & 7)) << 4) + 8 * (lq & 1);
#pragma unroll
    for (int h = 0; h < (kSw ? 1 : NH); h++)
    {
        const int col = col0 + kHalf * h;
        f4 gate[4], bias[4];
        u4 res[MH][2][2];
        if constexpr (EPI == kGemmResidual)
        {
#pragma unroll
            for (int j = 0; j < MH; j++)
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int s = 0; s < 2; s++)
                    {
                        const int row = min(row0 + kHalf * j + 16 * b + rr + 8 * s, a.m - 1);
                        res[j][b][s] = __builtin_nontemporal_load(
                            reinterpret_cast<const u4*>(a.r + static_cast<long long>(row) * a.n + col + 8 * cc));
                    }
#pragma unroll
            for (int t = 0; t < 4; t++)
            {
                gate[t] = f4{1.f, 1.f, 1.f, 1.f};
                bias[t] = f4{0.f, 0.f, 0.f, 0.f};
                if (a.gate)
                    gate[t] = *reinterpret_cast<const f4u*>(a.gate + col + 16 * t + 4 * lq);
                if (a.bias)
                    bias[t] = *reinterpret_cast<const f4u*>(a.bias + col + 16 * t + 4 * lq);
            }
        }
#pragma unroll
        for (int j = 0; j < MH; j++)
        {
#pragma unroll
            for (int b = 0; b < 2; b++)
            {
                h4 old[4];
                if constexpr (EPI == kGemmResidual)
                {
                    *reinterpret_cast<u4*>(line[0]) = res[j][b][0];
                    *reinterpret_cast<u4*>(line[1]) = res[j][b][1];
                    lds_order();
#pragma unroll
                    for (int t = 0; t < 4; t++)
                        old[t] = *reinterpret_cast<const h4*>(quad[t]);
                    lds_order();
                }
#pragma unroll
                for (int t = 0; t < 4; t++)
                {
                    h4 o;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                    {
                        float v = acc[h][j][t][b][e];
                        if constexpr (kSw)
                        {
                            float u = acc[NH - 1][j][t][b][e];
                            if constexpr (ROUNDED)
                            {
                                v = round16(v);
                                u = round16(u);
                                const float den = 1.f + expf(-v);
                                v = (v / den) * u;
                            }
                            else
                            {
                                const float den = 1.f + __builtin_amdgcn_exp2f(v * -kLog2e);
                                v = v * __builtin_amdgcn_rcpf(den) * u;
                            }
                        }
                        if constexpr (EPI == kGemmResidual)
                        {
                            const float r = h2f(old[t][e]);
                            if (!a.rounded)
                            {
                                v = v * gate[t][e] + r + bias[t][e];
                            }
                            else
                            {
                                v = round16(v);
                                if (a.bias)
                                    v = v + bias[t][e];
                                if (a.gate)
                                    v = v * gate[t][e];
                                v = v + r;
                            }
                        }
                        o[e] = static_cast<_Float16>(v);
                    }
                    *reinterpret_cast<h4*>(quad[t]) = o;
                }
                lds_order();
#pragma unroll
                for (int s = 0; s < 2; s++)
                {
                    const int row = row0 + kHalf * j + 16 * b + rr + 8 * s;
                    const u4 v = *reinterpret_cast<const u4*>(line[s]);
                    if (row < a.m)
                        __builtin_nontemporal_store(v, reinterpret_cast<u4*>(a.y + static_cast<long long>(row) * a.n + col + 8 * cc));
                }
                lds_order();
            }
        }
    }
}

template <int MH, int NH, int EPI, bool KS>
__global__ __launch_bounds__(kThreads) void gemm_tile_kernel(TileArgs a)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    using S = Shape<MH, NH>;
    constexpr int kSlots = S::kSlots;
    constexpr int kFour = MH == 2 && NH == 2; // four phases a stage
    static_assert(!KS || MH + NH == 2, "the K-split form is the 128 x 128 one");
    constexpr int kSteps = KS ? 1 : 2; // k-steps of 32 a wave multiplies per stage
    constexpr int kXT = KS ? 4 : 2;    // 16-row X tiles of a wave and half
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2; // the two groups alternate
    // rows of the wave's part in each W half and X half.  KS: the groups share
    // a 64 x 64 part and take one k-step of a stage each
    const int wrow = KS ? 64 * (wave & 1) : 64 * grp;
    const int xrow = KS ? 64 * ((wave >> 1) & 1) : 32 * (wave & 3);
    const int lr = lane & 15;
    const int lq = lane >> 4;
    const int nk = a.k / kBK;
    const unsigned k2 = 2u * static_cast<unsigned>(a.k);

    // tile list of this workgroup: round r gives XCD x the contiguous ids
    // [r G + x G/8, + G/8), the last round an even share of what is left
    const int G = static_cast<int>(gridDim.x);
    const int per_xcd = G >> 3;
    const int xcd = blockIdx.x & 7;
    const int local = blockIdx.x >> 3;
    const int full = a.total / G;
    const int left = a.total - full * G;
    const int left_per = (left + 7) >> 3;
    const int left_id = xcd * left_per + local;
    const bool has_left = local < left_per && left_id < left;
    const int ntiles = full + (has_left ? 1 : 0);
    if (ntiles == 0)
        return;
    auto tile_of = [&](int i, int* m0, int* n0) {
        const int id = i < full ? i * G + xcd * per_xcd + local : full * G + left_id;
        int tm, tn;
        tile_at(a, id, &tm, &tn);
        *m0 = tm * (kHalf * MH);
        *n0 = tn * (EPI == kGemmSwiGLU ? kHalf : kHalf * NH);
    };

    // fetch side: this wave fetches rows 16 wave + 8 i + lane / 8 of every
    // half-tile; the lane's LDS slot lane & 7 of the row holds chunk
    // (lane & 7) ^ ((row >> 1) & 7)
    const unsigned frow = 16u * wave + (lane >> 3);
    const unsigned chunk0 = 16u * ((lane & 7) ^ (lane >> 4));
    const unsigned vw0 = frow * k2 + chunk0;
    const unsigned vw1 = (frow + 8) * k2 + (chunk0 ^ 64u);
    unsigned vx[MH][2];
    const char* fx = nullptr;       // X rows of the tile being fetched, at the stage being fetched
    const char* fw[NH];
    int f_tile = -1;                // tile being fetched
    int f_kt = nk;                  // next stage to fetch of it (nk: open the next tile)
    unsigned f_slot = 0;
    auto open_tile = [&]() {
        f_tile++;
        f_kt = 0;
        int m0, n0;
        tile_of(f_tile, &m0, &n0);
        fx = reinterpret_cast<const char*>(a.x) + static_cast<unsigned long long>(m0) * k2;
        const int lastrow = a.m - 1 - m0;
#pragma unroll
        for (int j = 0; j < MH; j++)
        {
            // rows past M repeat the last one; their sums are never stored
            vx[j][0] = static_cast<unsigned>(min(static_cast<int>(kHalf * j + frow), lastrow)) * k2 + chunk0;
            vx[j][1] = static_cast<unsigned>(min(static_cast<int>(kHalf * j + frow + 8), lastrow)) * k2 + (chunk0 ^ 64u);
        }
#pragma unroll
        for (int h = 0; h < NH; h++)
        {
            const _Float16* src = (EPI == kGemmSwiGLU && h == 1) ? a.w2 : a.w;
            const int row = (EPI == kGemmSwiGLU) ? n0 : n0 + kHalf * h;
            fw[h] = reinterpret_cast<const char*>(src) + static_cast<unsigned long long>(row) * k2;
        }
    };
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<size_t>(smem));
    const unsigned lds_wave = lds0 + 16u * wave * kRowBytes;
    auto fetch_w = [&](int h) {
        const unsigned d = lds_wave + f_slot + h * kHalfBytes;
        dma16(fw[h], vw0, d);
        dma16(fw[h], vw1, d + 8 * kRowBytes);
    };
    auto fetch_x = [&](int j) {
        const unsigned d = lds_wave + f_slot + (NH + j) * kHalfBytes;
        dma16(fx, vx[j][0], d);
        dma16(fx, vx[j][1], d + 8 * kRowBytes);
    };
    // moves the fetch side to the next stage (of the next tile when needed)
    auto fetch_next = [&]() {
        f_kt++;
        f_slot = f_slot + S::kStageBytes == kSlots * S::kStageBytes ? 0u : f_slot + S::kStageBytes;
        fx += kRowBytes;
#pragma unroll
        for (int h = 0; h < NH; h++)
            fw[h] += kRowBytes;
        if (f_kt == nk && f_tile + 1 < ntiles)
            open_tile();
    };

    // operand reads: row wrow + 16 t + lr (W) / xrow + 16 b + lr (X) of a
    // half, chunk 4 ks + lq, in slot chunk ^ ((row >> 1) & 7)
    const unsigned swz = (lr >> 1) & 7;
    unsigned ow[kSteps], ox[kSteps];
#pragma unroll
    for (int ks = 0; ks < kSteps; ks++)
    {
        const unsigned c = ((4 * (KS ? grp : ks) + lq) ^ swz) << 4;
        ow[ks] = (wrow + lr) * kRowBytes + c;
        ox[ks] = NH * kHalfBytes + (xrow + lr) * kRowBytes + c;
    }
    h8 rw[kSteps][4];
    h8 rx[MH][kSteps][kXT];
    f4 acc[NH][MH][4][kXT];
    unsigned r_slot = 0;
    auto read_w = [&](int h) {
        const char* st = smem + r_slot + h * kHalfBytes;
#pragma unroll
        for (int ks = 0; ks < kSteps; ks++)
#pragma unroll
            for (int t = 0; t < 4; t++)
                rw[ks][t] = *reinterpret_cast<const h8*>(st + ow[ks] + t * 16 * kRowBytes);
    };
    auto read_x = [&](int j) {
        const char* st = smem + r_slot + j * kHalfBytes;
#pragma unroll
        for (int ks = 0; ks < kSteps; ks++)
#pragma unroll
            for (int b = 0; b < kXT; b++)
                rx[j][ks][b] = *reinterpret_cast<const h8*>(st + ox[ks] + b * 16 * kRowBytes);
    };
    auto mma = [&](int h, int j) {
#pragma unroll
        for (int ks = 0; ks < kSteps; ks++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int b = 0; b < kXT; b++)
                    acc[h][j][t][b] =
                        __builtin_amdgcn_mfma_f32_16x16x32_f16(rw[ks][t], rx[j][ks][b], acc[h][j][t][b], 0, 0, 0);
    };

    auto read_slot_next = [&]() {
        r_slot = r_slot + S::kStageBytes == kSlots * S::kStageBytes ? 0u : r_slot + S::kStageBytes;
    };
    auto clear = [&]() {
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
            for (int j = 0; j < MH; j++)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int b = 0; b < kXT; b++)
                        acc[h][j][t][b] = f4{0.f, 0.f, 0.f, 0.f};
    };

    // the first kSlots stages
    const int stages = ntiles * nk;
    open_tile();
#pragma unroll
    for (int s = 0; s < kSlots; s++)
        if (s < stages)
        {
            fetch_w(0);
            fetch_x(0);
            if constexpr (MH == 2)
                fetch_x(1);
            if constexpr (NH == 2)
                fetch_w(1);
            fetch_next();
        }
    // stage 0 has landed once only the younger stages' fetches are outstanding
    constexpr int kPer = 2 * (MH + NH); // fetches per wave and stage
    wait_younger(min(stages - 1, kSlots - 1) * kPer);
    bar();
    if (grp == 1)
        bar(); // the second group runs one slot behind
    clear();

    // One stage.  kSteady: every fetch below exists (the loop's body then has
    // no branch but the tile switch: scalar work between the barriers costs
    // MFMA time); else g is one of the last kSlots stages.
    auto stage = [&](auto steady, int g) __attribute__((always_inline)) {
        constexpr bool kSteady = decltype(steady)::value;
        const int rem = stages - 1 - g; // stages after this one
        if constexpr (kFour)
        {
            // phase 0: W0 X0; X1(g) next
            read_w(0);
            read_x(0);
            if (kSteady || rem >= 1)
                wait_vm<10>();
            else
                wait_vm<2>();
            wait_lds();
            bar();
            mma(0, 0);
            bar();
            // phase 1: W0 X1; W0 X0 of stage g + 2; W1(g) next
            read_x(1);
            if constexpr (kSteady)
            {
                fetch_w(0);
                fetch_x(0);
                wait_vm<12>();
            }
            else if (rem >= 1)
                wait_vm<8>();
            else
                wait_vm<0>();
            wait_lds();
            bar();
            mma(0, 1);
            bar();
            // phase 2: W1 X1; X1 of stage g + 2
            read_w(1);
            if constexpr (kSteady)
                fetch_x(1);
            wait_lds();
            bar();
            mma(1, 1);
            bar();
            // phase 3: W1 X0; W1 of stage g + 2; W0 X0 of stage g + 1 next
            if constexpr (kSteady)
            {
                fetch_w(1);
                fetch_next();
                wait_vm<12>();
            }
            else
                wait_vm<4>();
            bar();
            mma(1, 0);
            bar();
        }
        else if constexpr (MH + NH == 3)
        {
            // phase 0: W0 X0; the rest of stage g - 1 + kSlots; X1 / W1 of this stage next
            read_w(0);
            read_x(0);
            if (g > 0 && (kSteady || rem >= kSlots - 1))
            {
                if constexpr (MH == 2)
                    fetch_x(1);
                else
                    fetch_w(1);
                fetch_next();
            }
            if constexpr (kSteady)
                wait_vm<(kSlots - 1) * 6>();
            else
                wait_younger(min(rem, kSlots - 1) * 6);
            wait_lds();
            bar();
            mma(0, 0);
            bar();
            // phase 1: X1 or W1; W0 X0 of stage g + kSlots; W0 X0 of stage g + 1 next
            if constexpr (MH == 2)
                read_x(1);
            else
                read_w(1);
            if constexpr (kSteady)
            {
                fetch_w(0);
                fetch_x(0);
                wait_vm<2 + 6 * (kSlots - 2) + 4>();
            }
            else if (rem >= 2)
                wait_younger(2 + 6 * (rem - 1));
            else
                wait_vm<2>();
            wait_lds();
            bar();
            if constexpr (MH == 2)
                mma(0, 1);
            else
                mma(1, 0);
            bar();
        }
        else
        {
            read_w(0);
            read_x(0);
            if (g > 0 && (kSteady || rem >= kSlots - 1))
            {
                fetch_w(0);
                fetch_x(0);
                fetch_next();
            }
            if constexpr (kSteady)
                wait_vm<(kSlots - 2) * 4>();
            else
                wait_younger(max(0, min(rem, kSlots - 1) - 1) * 4);
            wait_lds();
            bar();
            mma(0, 0);
            bar();
        }
        read_slot_next();
    };
    int g = 0;
    for (int tile = 0; tile < ntiles; tile++)
    {
        const int steady = min(max(stages - kSlots - g, 0), nk);
        int m0, n0;
        tile_of(tile, &m0, &n0);
        int i = 0;
        if constexpr (EPI == kGemmResidual && MH == 2)
        {
            // the tile's residual lines move into the L2 while its last stages
            // run (not for the 128 x 128 forms, whose waves have half a
            // touch's rows each)
#pragma nounroll
            for (; i < steady - kTouchAhead; i++)
                stage(std::true_type{}, g++);
            // lane: line lane & (lines - 1) of row lane / lines of the wave's rows
            constexpr int kLines = 2 * NH;            // 128-byte lines of a tile row
            constexpr int kPerTouch = 64 / kLines;    // rows per instruction
            constexpr int kRows = kHalf * MH / 8;     // rows of this wave
#pragma unroll
            for (int u = 0; u < kRows / kPerTouch; u++)
            {
                const int row = min(m0 + kRows * wave + kPerTouch * u + lane / kLines, a.m - 1);
                touch(a.r + static_cast<long long>(row) * a.n + n0 + 64 * (lane % kLines),
                      lds0 + kSlots * S::kStageBytes + wave * kEpiWave);
            }
        }
#pragma nounroll
        for (; i < steady; i++)
            stage(std::true_type{}, g++);
#pragma nounroll
        for (; i < nk; i++)
            stage(std::false_type{}, g++);
        char* mine = smem + kSlots * S::kStageBytes + wave * kEpiWave;
        if constexpr (KS)
        {
            // one tile per workgroup: the stage slots are free once both
            // groups are done.  Each wave hands half of its sums to the wave
            // that holds the same part for the other k-steps, and finishes
            // the other half: group 0 X tiles 0, 1, group 1 X tiles 2, 3
            if (grp == 0)
                bar();
            f4* give = reinterpret_cast<f4*>(smem) + wave * 8 * 64 + lane;
            const f4* take = reinterpret_cast<const f4*>(smem) + (wave ^ 4) * 8 * 64 + lane;
            f4 sum[1][1][4][2];
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int b = 0; b < 2; b++)
                {
                    give[(2 * t + b) * 64] = grp == 0 ? acc[0][0][t][2 + b] : acc[0][0][t][b];
                    sum[0][0][t][b] = grp == 0 ? acc[0][0][t][b] : acc[0][0][t][2 + b];
                }
            wait_lds();
            bar();
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int b = 0; b < 2; b++)
                    sum[0][0][t][b] += take[(2 * t + b) * 64];
            epilogue<1, 1, EPI, false>(a, sum, mine, m0 + xrow + 32 * grp, n0 + wrow, lane);
            return;
        }
        else
        {
            if (EPI == kGemmSwiGLU && a.rounded)
                epilogue<MH, NH, EPI, true>(a, acc, mine, m0 + xrow, n0 + wrow, lane);
            else
                epilogue<MH, NH, EPI, false>(a, acc, mine, m0 + xrow, n0 + wrow, lane);
            clear();
        }
    }
    if (grp == 0)
        bar();
}

template <int MH, int NH, int EPI, bool KS = false>
int launch(const TileArgs& a, hipStream_t stream)
{
    using S = Shape<MH, NH>;
    const void* fn = reinterpret_cast<const void*>(&gemm_tile_kernel<MH, NH, EPI, KS>);
    const int rc = set_dynamic_lds(fn, S::kLds, "gemm_f16: dynamic LDS attribute");
    if (rc != SV2_OK)
        return rc;
    // a multiple of the 8 XCDs; KS: one tile per workgroup
    const int all = (a.total + 7) / 8 * 8;
    const int grid = KS ? all : std::min(kCus, all);
    hipLaunchKernelGGL((gemm_tile_kernel<MH, NH, EPI, KS>), dim3(static_cast<unsigned>(grid)), dim3(kThreads), S::kLds,
                       stream, a);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? SV2_OK : hip_error(err, "gemm_tile_kernel launch");
}

// The tile forms and their measured times (us, MI355X, random operands): a
// stage of 64 k of one tile when few CUs run (bounded by LDS) and when all of
// them do (by power and the L2), and a tile's epilogue.
enum Form
{
    kBig,   // 256 x 256
    kTall,  // 256 rows x 128 columns
    kSmall, // 128 x 128
    kSplit, // 128 x 128, K split between the groups
    kWide,  // SwiGLU: 128 rows x (128 gate + 128 value)
    kForms
};
struct FormCost
{
    int rows, cols; // of W rows: SwiGLU outputs are half as many
    double stage_min, stage_full, tile;
};
constexpr FormCost kCost[kForms] = {
    {256, 256, 0.97, 1.42, 3.0}, {256, 128, 0.58, 0.78, 2.0}, {128, 128, 0.39, 0.50, 1.5},
    {128, 128, 0.33, 0.48, 2.0}, {128, 256, 0.60, 0.80, 2.0},
};
constexpr double kLaunch = 7.0; // launch, first fetches, drain

long long tiles_of(Form f, int rows, long long wrows)
{
    return (static_cast<long long>(rows) + kCost[f].rows - 1) / kCost[f].rows * (wrows / kCost[f].cols);
}

double form_us(Form f, int rows, int in, long long wrows)
{
    const long long tiles = tiles_of(f, rows, wrows);
    const double nk = in / kBK;
    const FormCost& c = kCost[f];
    double us = kLaunch + static_cast<double>(tiles / kCus) * (nk * c.stage_full + c.tile);
    const long long left = tiles % kCus;
    if (left > 0)
        us += nk * std::max(c.stage_min, c.stage_full * static_cast<double>(left) / kCus) + c.tile;
    return us;
}

// How the rows of a product are tiled: all of them in one form, or, where the
// last round of 256 x 256 tiles would leave most CUs idle, the row bands that
// fill whole rounds in 256 x 256 tiles and the rest in another form (out
// 6912 -> 2560 at 21658 rows is 3.3 rounds).  The choice depends on the sizes
// alone.
struct Plan
{
    int first_rows; // in 256 x 256 tiles; 0: all rows in `rest`
    Form rest;
    double us;
};

Plan make_plan(int rows, int in, int out, int epi, bool rounded)
{
    const long long wrows = epi == kGemmSwiGLU ? 2LL * out : out;
    Form forms[4];
    int nf = 0;
    if (epi == kGemmSwiGLU)
    {
        forms[nf++] = kBig;
        forms[nf++] = kWide;
    }
    else
    {
        forms[nf++] = kBig;
        forms[nf++] = kTall;
        forms[nf++] = kSmall;
        // the rounded epilogues keep one order of summation in every form
        if (!rounded)
            forms[nf++] = kSplit;
    }
    Plan best{0, kBig, form_us(kBig, rows, in, wrows)};
    for (int i = 1; i < nf; i++)
    {
        const double us = form_us(forms[i], rows, in, wrows);
        if (us < best.us)
            best = Plan{0, forms[i], us};
    }
    const long long per_band = wrows / 256;
    const long long bands = static_cast<long long>(kCus) * (tiles_of(kBig, rows, wrows) / kCus) / per_band;
    const long long first = bands * 256;
    if (first > 0 && first < rows)
        for (int i = 1; i < nf; i++)
        {
            const double us = form_us(kBig, static_cast<int>(first), in, wrows) +
                              form_us(forms[i], rows - static_cast<int>(first), in, wrows);
            if (us < best.us)
                best = Plan{static_cast<int>(first), forms[i], us};
        }
    return best;
}

template <int EPI>
int launch_form(Form f, const TileArgs& a, hipStream_t stream)
{
    if constexpr (EPI == kGemmSwiGLU)
    {
        return f == kBig ? launch<2, 2, EPI>(a, stream) : launch<1, 2, EPI>(a, stream);
    }
    else
    {
        switch (f)
        {
        case kBig: return launch<2, 2, EPI>(a, stream);
        case kTall: return launch<2, 1, EPI>(a, stream);
        case kSmall: return launch<1, 1, EPI>(a, stream);
        default: return launch<1, 1, EPI, true>(a, stream);
        }
    }
}

// Rows r0 .. r0 + rows of the product in form f.
int run_rows(Form f, TileArgs a, int epi, int r0, int rows, hipStream_t stream)
{
    const long long wrows = epi == kGemmSwiGLU ? 2LL * a.n : a.n;
    a.x += static_cast<long long>(r0) * a.k;
    a.y += static_cast<long long>(r0) * a.n;
    if (a.r)
        a.r += static_cast<long long>(r0) * a.n;
    a.m = rows;
    a.tiles_m = (rows + kCost[f].rows - 1) / kCost[f].rows;
    a.tiles_n = static_cast<int>(wrows / kCost[f].cols);
    const long long total = tiles_of(f, rows, wrows);
    if (total > INT_MAX - kCus)
        return set_error(SV2_EUNSUPPORTED, "inner product: too many tiles");
    a.total = static_cast<int>(total);
    // eight row bands a group: an XCD's 32 tiles are then 8 bands x 4 columns
    a.group_m = 8;
    switch (epi)
    {
    case kGemmStore: return launch_form<kGemmStore>(f, a, stream);
    case kGemmResidual: return launch_form<kGemmResidual>(f, a, stream);
    default: return launch_form<kGemmSwiGLU>(f, a, stream);
    }
}

bool operands_fit(int rows, int in, int out)
{
    return static_cast<long long>(rows) * in * 2 <= INT_MAX && static_cast<long long>(out) * in * 2 <= INT_MAX;
}

// Which products of the fp16 blocks take this kernel and which the library,
// from both measured at 256 to 21658 rows with weights out of cache, against
// the two hipBLASLt builds a process may map (torch's and ROCm's).  Figures:
// library time / kernel time, torch's build and ROCm's.  SwiGLU, where the
// library takes three launches, is 1.03 to 1.66 and 0.97 to 1.54 times as fast
// on the kernel and always takes it.
//
// The kernel's tiles are 256 x 256 down to 128 x 128; the library has those
// and others between, so it divides a product of few tiles better wherever
// these leave CUs idle, and about as well where both run whole rounds.

// qkv 2560 -> 7680 and its like.
bool store_pays(int rows, int in, int out)
{
    // few stages: launch and epilogue are most of it, and shorter here
    // (256 -> 768 1.1 to 1.8, 512 -> 1536 1.05 to 1.7, torch's build)
    if (in <= 512)
        return true;
    // two whole rounds of 256 x 256 tiles or more: 0.97 to 1.28, 0.97 to 1.23
    if (tiles_of(kBig, rows, out) >= 2 * kCus)
        return true;
    const Plan p = make_plan(rows, in, out, kGemmStore, false);
    const long long tiles = tiles_of(p.rest, rows - p.first_rows, out);
    // one round and a rest in smaller tiles: a rest of 60 tiles costs a launch
    // and a round all the same (0.94 to 1.00, 0.98 to 1.06), 120 and more pay
    // (0.95 to 1.23, 0.99 to 1.22)
    if (p.first_rows > 0)
        return 5 * tiles >= 2 * kCus;
    // one round: up to 180 tiles 0.84 to 1.07, 0.76 to 1.12 (0.95, 0.91 on
    // average); from 210 on 0.94 to 1.21, 0.95 to 1.23 (1.07, 1.09)
    if (tiles <= kCus)
        return 4 * tiles >= 3 * kCus;
    // up to two rounds of 256 x 256 tiles: 390 tiles 0.92 to 1.02, 0.91 to
    // 1.15; 420 and more 0.96 to 1.03, 0.98 to 1.23 (0.98, 1.10).  More than
    // one round of a smaller tile runs below the large one's rate (720 tiles
    // of 256 x 128 0.94 to 1.01; 3072 -> 9216 in 504 of 128 x 128 0.83)
    return p.rest == kBig && 5 * tiles >= 8 * kCus;
}

// The products with a residual: proj 2560 -> 2560 and out 6912 -> 2560.  Their
// few columns make a third of qkv's tiles, and the residual, read before a
// tile's sums can leave, costs it 2 to 4 us.
bool residual_pays(int rows, int in, int out)
{
    const Plan p = make_plan(rows, in, out, kGemmResidual, false);
    // one launch of the K-split form that fills the CUs, K long enough to hide
    // the epilogue and short enough that 0.33 us a stage do not add up: proj in
    // 200 to 240 tiles 1.00 to 1.08, 0.96 to 1.09, in 160 to 180 0.91 to 1.01,
    // 0.89 to 0.98; 4096 -> 4096 0.99 to 1.10; but 1024 -> 1024 0.8, 1536 ->
    // 1536 0.90 to 1.11 and 6912 -> 2560 0.97 to 1.19 (torch's build; ROCm's
    // takes twice as long there)
    if (p.first_rows == 0 && p.rest == kSplit && in >= 2048 && in <= 4096)
    {
        const long long split = tiles_of(kSplit, rows, out);
        return split <= kCus && 4 * split >= 3 * kCus;
    }
    // K long against the epilogue, from nearly three rounds of 256 x 256 tiles
    // on: out 0.94 to 1.19, 0.95 to 1.12 (1.06, 1.03 on average).  From two
    // rounds to there it is 0.89 to 1.13, 0.94 to 1.06, by the luck of the
    // library's choice, and before 0.55 to 1.09 with torch's build; proj 0.87 to
    // 1.29, 0.88 to 1.02 from two rounds on and 0.57 to 1.02 before.
    return in >= 6144 && 20 * tiles_of(kBig, rows, out) >= 57 * kCus;
}

} // namespace

bool gemm_mfma_supported(int in, int out, int epi)
{
    if (in <= 0 || in % kBK != 0 || out <= 0)
        return false;
    return epi == kGemmSwiGLU ? out % 128 == 0 : out % 256 == 0;
}

bool gemm_mfma_fits(int rows, int in, int out, int epi, const void* x, const void* w, const void* w2, const void* y,
                    const void* residual)
{
    return rows > 0 && gemm_mfma_supported(in, out, epi) && operands_fit(rows, in, out) && !misaligned(x, 16) &&
           !misaligned(w, 16) && !misaligned(w2, 16) && !misaligned(y, 16) && !misaligned(residual, 16);
}

bool gemm_mfma_preferred(int rows, int in, int out, int epi, const void* x, const void* w, const void* w2,
                         const void* y, const void* residual)
{
    // fewer rows leave most CUs without a tile; there the library's smaller
    // tiles are as fast (96 rows, 6912 -> 2560: 22 us against 48)
    if (rows < kPreferRows || !gemm_mfma_fits(rows, in, out, epi, x, w, w2, y, residual))
        return false;
    switch (epi)
    {
    case kGemmStore: return store_pays(rows, in, out);
    case kGemmResidual: return residual_pays(rows, in, out);
    default: return true;
    }
}

int gemm_mfma(hipStream_t stream, int rows, int in, int out, const void* x, const void* w, const void* w2, void* y,
              int epi, bool rounded, const float* bias, const float* gate, const void* residual)
{
    if (rows == 0)
        return SV2_OK;
    if (epi != kGemmStore && epi != kGemmResidual && epi != kGemmSwiGLU)
        return set_error(SV2_EINVAL, "inner product: unknown epilogue");
    if (rows < 0 || !gemm_mfma_supported(in, out, epi))
        return set_error(SV2_EUNSUPPORTED,
                         "inner product: needs in a multiple of 64 and out a multiple of 256 (SwiGLU: 128)");
    if (!x || !w || !y || (epi == kGemmResidual && !residual) || (epi == kGemmSwiGLU && !w2))
        return set_error(SV2_EINVAL, "inner product: null pointer");
    if (misaligned(x, 16) || misaligned(w, 16) || misaligned(w2, 16) || misaligned(y, 16) || misaligned(residual, 16))
        return set_error(SV2_EINVAL, "inner product: x, W, y and residual must be 16-byte aligned");
    if (!operands_fit(rows, in, out))
        return set_error(SV2_EUNSUPPORTED, "inner product: an operand exceeds 2 GiB");
    TileArgs a{};
    a.x = static_cast<const _Float16*>(x);
    a.w = static_cast<const _Float16*>(w);
    a.w2 = static_cast<const _Float16*>(w2);
    a.y = static_cast<_Float16*>(y);
    a.r = static_cast<const _Float16*>(epi == kGemmResidual ? residual : nullptr);
    a.bias = bias;
    a.gate = gate;
    a.n = out;
    a.k = in;
    a.rounded = rounded ? 1 : 0;
    const Plan plan = make_plan(rows, in, out, epi, rounded);
    if (plan.first_rows > 0)
    {
        const int rc = run_rows(kBig, a, epi, 0, plan.first_rows, stream);
        if (rc != SV2_OK)
            return rc;
    }
    return run_rows(plan.rest, a, epi, plan.first_rows, rows - plan.first_rows, stream);
}

} // namespace sv2

extern "C" int sv2_inner_product_f16(const void* x, const void* w, const void* w_value, void* y, int rows, int in,
                                     int out, int epilogue, const float* bias, const float* gate,
                                     const void* residual, void* stream)
try
{
    static_assert(SV2_EPI_STORE == sv2::kGemmStore && SV2_EPI_RESIDUAL == sv2::kGemmResidual &&
                      SV2_EPI_SWIGLU == sv2::kGemmSwiGLU,
                  "epilogue codes of the C ABI and the kernel agree");
    if (epilogue != SV2_EPI_SWIGLU && w_value)
        return sv2::set_error(SV2_EINVAL, "sv2_inner_product_f16: w_value is only read by SV2_EPI_SWIGLU");
    return sv2::gemm_mfma(static_cast<hipStream_t>(stream), rows, in, out, x, w, w_value, y, epilogue, true, bias, gate,
                          residual);
}
catch (...)
{
    return sv2::caught_exception("sv2_inner_product_f16");
}

extern "C" int sv2_inner_product_f16_plan(int rows, int in, int out, int epilogue, int block, sv2_product_plan* plan)
try
{
    static_assert(SV2_FORM_256X256 == sv2::kBig && SV2_FORM_256X128 == sv2::kTall && SV2_FORM_128X128 == sv2::kSmall &&
                      SV2_FORM_128X128_KSPLIT == sv2::kSplit && SV2_FORM_128X256 == sv2::kWide,
                  "form codes of the C ABI and the kernel agree");
    if (!plan || rows <= 0 || in <= 0 || out <= 0 ||
        (epilogue != SV2_EPI_STORE && epilogue != SV2_EPI_RESIDUAL && epilogue != SV2_EPI_SWIGLU))
        return sv2::set_error(SV2_EINVAL, "sv2_inner_product_f16_plan: bad sizes, epilogue or null pointer");
    *plan = sv2_product_plan{0, 0, -1};
    // a null operand is an aligned one: the sizes alone decide
    if (!sv2::gemm_mfma_fits(rows, in, out, epilogue, nullptr, nullptr, nullptr, nullptr, nullptr))
        return block ? SV2_OK
                     : sv2::set_error(SV2_EUNSUPPORTED, "sv2_inner_product_f16_plan: sizes the kernel does not take");
    const sv2::Plan p = sv2::make_plan(rows, in, out, epilogue, !block);
    plan->kernel = !block || sv2::gemm_mfma_preferred(rows, in, out, epilogue, nullptr, nullptr, nullptr, nullptr, nullptr);
    plan->first_rows = p.first_rows;
    plan->form = p.rest;
    return SV2_OK;
}
catch (...)
{
    return sv2::caught_exception("sv2_inner_product_f16_plan");
}
