// GEMMs of the DiT block on the matrix cores (gfx950): out = epilogue(A W^T)
// with A the activations [M][K] and W a weight [N][K], both K-contiguous; the
// video and the text branch's GEMM of one step run in one launch.
//
// fp32 operands are split. A row x (of A or of W) is stored as x 2^s = hi + lo
// with s the row's exponent shift (its largest finite value lies in
// [2^14, 2^15)), hi the value rounded to fp16 and lo the rest rounded to fp16:
// 22 bits and the signs, or 2^-40 of the row's largest value where that is
// coarser. The product is hi hi + hi lo + lo hi on v_mfma_f32_32x32x16_f16
// with fp32 accumulation (the dropped lo lo weighs 2^-24 of a product), three
// fp16 MFMAs in place of one fp32 product at 1/16 of their rate. Off the
// 64-bit product by 5.7e-7 (relative 2-norm, N(0, 1) by N(0, 0.02), K = 2560)
// where fp32 MFMAs are off by 9.0e-7.
//
// What bounds the stage loop is the matrix core and, next, what feeds it: LDS
// (a 256 x 256 bf16 stage is 2048 MFMA cycles a SIMD and as many of LDS reads
// and writes) and the loads' issue. So the next unit's operand reads and the
// next stage's loads go between the MFMAs one by one (8192^3 bf16 1102 -> 1309
// TFLOP/s, split 430 -> 466), and the wave tile is as large as registers allow.
// At block sizes it is the last round of tiles: hence several tile shapes and a
// small one for the text rows, whose tiles fill that round's gaps.
// Measured, 2304 video rows and 64 text rows in one launch, weights from HBM,
// K x N of the block (the library's video GEMM alone took 772 us in fp32 and 99
// in bf16 at 2560 x 7680):
//   2560 x 7680             bf16 107 us, split 238 us
//   2560 x 2560, epilogue   bf16  43 us, split  96 us
//   2560 x 13824, SwiGLU    bf16 175 us, split 430 us
//   6912 x 2560, epilogue   bf16  94 us, split 234 us
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "dit_kernels.h"
#include "dit_split.h"

namespace awa
{
namespace
{

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef __attribute__((address_space(3))) char lds_char;

// 16 bytes a lane from base + offset to the 1 KB of LDS at `lds` (lane order).
// Written out so that the compiler does not wait for it before every LDS read;
// the stage loop waits with vmcnt itself. It has no output register.
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t offset, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base)
                 : "memory");
}

// Waits for all but the N latest loads of the wave and for its LDS reads, then
// for the workgroup.
template <int N>
__device__ __forceinline__ void arrive()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The weight row behind column j of the tile at col0 (the last one beyond the
// end), within its own weight for SwiGLU: those tiles take 16 gate columns,
// then the same 16 input columns.
template <int EPI>
__device__ __forceinline__ int weight_row(const GemmProblem& g, int col0, int j)
{
    if (EPI != kGemmSwiGlu)
        return min(col0 + j, g.n - 1);
    return min((col0 >> 1) + (j >> 5) * 16 + (j & 15), (g.n >> 1) - 1);
}

// silu(a) * b; to be rounded to bf16 (fast) on the hardware's exp2 and
// reciprocal, which are good to 2^-20 here.
template <bool FAST>
__device__ __forceinline__ float silu_mul(float a, float b)
{
    if (FAST)
        return a * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(a * -1.44269504f)) * b;
    return a / (1.f + expf(-a)) * b;
}

template <bool BF16>
__device__ __forceinline__ void load8(const void* p, size_t i, float (&v)[8])
{
    if (BF16)
    {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(static_cast<const __bf16*>(p) + i);
#pragma unroll
        for (int e = 0; e < 8; e++)
            v[e] = static_cast<float>(x[e]);
    }
    else
    {
        const float4 a = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
        const float4 b = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    }
}

template <bool BF16>
__device__ __forceinline__ void store8(void* p, size_t i, const float (&v)[8])
{
    if (BF16)
    {
        bf16x8 x;
#pragma unroll
        for (int e = 0; e < 8; e++)
            x[e] = static_cast<__bf16>(v[e]);
        *reinterpret_cast<bf16x8*>(static_cast<__bf16*>(p) + i) = x;
    }
    else
    {
        *reinterpret_cast<float4*>(static_cast<float*>(p) + i) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(static_cast<float*>(p) + i + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// One product of split rows of which one is not finite, from the planes in
// fp32: an infinity stays one where the split products would give NaN.
__device__ float dot_planes(const GemmProblem& g, const void* weight, int row, int wrow, int ma, int mw)
{
    if ((ma | mw) & kRowNan)
        return __uint_as_float(0x7fc00000u);
    const char* a = static_cast<const char*>(g.a) + static_cast<size_t>(row) * g.lda;
    const char* w = static_cast<const char*>(weight) + static_cast<size_t>(wrow) * g.ldw;
    float sum = 0.f;
    for (int t = 0; t < g.stages; t++)
    {
        const _Float16* pa = reinterpret_cast<const _Float16*>(a + static_cast<size_t>(t) * kStageBytes);
        const _Float16* pw = reinterpret_cast<const _Float16*>(w + static_cast<size_t>(t) * kStageBytes);
        for (int k = 0; k < kGroup; k++)
            sum = fmaf(static_cast<float>(pa[k]) + static_cast<float>(pa[k + kGroup]),
                       static_cast<float>(pw[k]) + static_cast<float>(pw[k + kGroup]), sum);
    }
    return ldexpf(sum, -row_shift(ma) - row_shift(mw));
}

// The outputs of a wave's tile whose row or column holds a NaN or an infinity.
template <int EPI>
__device__ void finish_non_finite(const GemmProblem& g, int row0, int rows, int col0, int cols)
{
    const int width = EPI == kGemmSwiGlu ? g.n >> 1 : g.n;
    for (int i = threadIdx.x & 63; i < rows * cols; i += 64)
    {
        const int row = row0 + i / cols, c = col0 + i % cols;
        if (row >= g.m || c >= width)
            continue;
        const int ma = g.meta_a[row], mw = g.meta_w[c], mi = EPI == kGemmSwiGlu ? g.meta_w[width + c] : 0;
        if (!((ma | mw | mi) & (kRowNan | kRowInf)))
            continue;
        float r = dot_planes(g, g.w, row, c, ma, mw);
        if (EPI == kGemmSwiGlu)
            r = silu_mul<false>(r, dot_planes(g, g.w2, row, c, ma, mi));
        if (EPI == kGemmGate)
        {
            r = (r + (g.bias ? g.bias[c] : 0.f)) * (g.gate ? g.gate[c] : 1.f) +
                static_cast<const float*>(g.residual)[static_cast<size_t>(row) * g.ldr + c];
            r = g.twice ? r + r : r;
        }
        static_cast<float*>(g.out)[static_cast<size_t>(row) * g.ldo + c] = r;
    }
}

// One tile of a problem: rows [row0, row0 + BM) by columns [col0, col0 + BN) on
// WGM x WGN waves with STAGES buffers. A stage is 128 bytes of every row of the
// tile: 64 bf16 values in four units of 16, or (SPLIT) 32 values as two planes
// in two units of 16.
template <bool SPLIT, int BM, int BN, int WGM, int WGN, int STAGES, int EPI>
__device__ __forceinline__ void run_tile(const GemmProblem& g, const int row0, const int col0)
{
    constexpr int kWaves = WGM * WGN;
    constexpr int MB = BM / WGM / 32, NB = BN / WGN / 32;
    constexpr int kLoadsA = BM / 8 / kWaves, kLoadsB = BN / 8 / kWaves, kLoads = kLoadsA + kLoadsB;
    constexpr int kStageA = BM * kStageBytes, kStageB = BN * kStageBytes;
    constexpr int kUnits = SPLIT ? 2 : 4, kPlanes = SPLIT ? 2 : 1;
    static_assert(MB * WGM * 32 == BM && NB * WGN * 32 == BN && kLoadsA * kWaves * 8 == BM &&
                      kLoadsB * kWaves * 8 == BN,
                  "tile split");
    extern __shared__ char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WGN, wn = wave % WGN;

    // Staging: a load moves 8 rows of 128 bytes; lane l takes row l / 8 and
    // the 16-byte piece (l % 8) ^ (row % 8), so that the operand reads below
    // (one piece of 8 consecutive rows) touch all banks.
    const uint32_t piece = ((lane & 7) ^ (lane >> 3)) * 16;
    uint32_t off_a[kLoadsA], off_b[kLoadsB];
#pragma unroll
    for (int i = 0; i < kLoadsA; i++)
        off_a[i] = static_cast<uint32_t>(min(row0 + (wave * kLoadsA + i) * 8 + (lane >> 3), g.m - 1)) * g.lda + piece;
#pragma unroll
    for (int i = 0; i < kLoadsB; i++)
        off_b[i] = static_cast<uint32_t>(weight_row<EPI>(g, col0, (wave * kLoadsB + i) * 8 + (lane >> 3))) * g.ldw +
                   piece;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char*)smem));
    const char* pa = static_cast<const char*>(g.a);
    const char* pb = static_cast<const char*>(g.w);
    const char* pb2 = EPI == kGemmSwiGlu ? static_cast<const char*>(g.w2) : nullptr;
    const int stages = g.stages;
    // Load i of a stage: A's, then W's.
    auto stage_load = [&](int i, uint32_t at_a, uint32_t at_b) {
        if (i < kLoadsA)
            load_to_lds(pa, off_a[i], lds0 + at_a + i * 1024);
        else
        {
            i -= kLoadsA;
            load_to_lds(EPI == kGemmSwiGlu && ((wave * kLoadsB + i) & 2) ? pb2 : pb, off_b[i], lds0 + at_b + i * 1024);
        }
    };
    auto at_a = [&](int buf) { return static_cast<uint32_t>(buf * kStageA + wave * kLoadsA * 1024); };
    auto at_b = [&](int buf) {
        return static_cast<uint32_t>(STAGES * kStageA + buf * kStageB + wave * kLoadsB * 1024);
    };
    auto next_stage = [&]() {
        pa += kStageBytes;
        pb += kStageBytes;
        pb2 += kStageBytes;
    };
    // The last stage of bf16 rows that end inside it: pieces past the row's end
    // are zeros (no load).
    const bool ragged = !SPLIT && g.last_bytes != kStageBytes;
    auto stage = [&](int t, int buf) {
        if (SPLIT || !ragged || t + 1 < stages || piece < g.last_bytes)
        {
#pragma unroll
            for (int i = 0; i < kLoads; i++)
                stage_load(i, at_a(buf), at_b(buf));
        }
        else
        {
#pragma unroll
            for (int i = 0; i < kLoads; i++)
                *reinterpret_cast<uint4*>(smem + (i < kLoadsA ? at_a(buf) + i * 1024 : at_b(buf) + (i - kLoadsA) * 1024) +
                                          lane * 16) = make_uint4(0, 0, 0, 0);
        }
        next_stage();
    };

    f32x16 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                acc[m][n][e] = 0.f;

    // Operands of a unit, in two register sets: the next unit's are read
    // while the matrix core works on this one's.
    const char* ra = smem + (wm * MB * 32 + (lane & 31)) * kStageBytes;
    const char* rb = smem + STAGES * kStageA + (wn * NB * 32 + (lane & 31)) * kStageBytes;
    uint32_t pc[4];
#pragma unroll
    for (int s = 0; s < 4; s++)
        pc[s] = ((2 * s + (lane >> 5)) ^ (lane & 7)) * 16;
    uint4 fa[2][kPlanes][MB], fb[2][kPlanes][NB];
    constexpr int kReads = kPlanes * (MB + NB), kMfma = (SPLIT ? 3 : 1) * MB * NB;
    // Read i of unit u's operands: hi of A and W, then lo.
    auto read = [&](int buf, int u, int i) {
        const int h = i / (MB + NB), j = i % (MB + NB);
        if (j < MB)
            fa[u & 1][h][j] = *reinterpret_cast<const uint4*>(ra + buf * kStageA + j * 32 * kStageBytes + pc[2 * h + u]);
        else
            fb[u & 1][h][j - MB] =
                *reinterpret_cast<const uint4*>(rb + buf * kStageB + (j - MB) * 32 * kStageBytes + pc[2 * h + u]);
    };
    // Unit u's MFMAs, with the reads of the next unit (buffer buf, unit next;
    // next < 0: none) and a stage's loads (into load_buf) spread between them
    // in this order: issued in one go they would hold up the MFMAs behind them.
    auto multiply = [&](int u, int buf, int next, auto loads, int load_buf) {
        constexpr bool kLoad = decltype(loads)::value;
        constexpr int kEvents = kReads + (kLoad ? kLoads : 0);
        const uint32_t la = at_a(load_buf), lb = at_b(load_buf);
        int event = 0;
#pragma unroll
        for (int i = 0; i < kMfma; i++)
        {
            const int x = i / (MB * NB), m = i / NB % MB, n = i % NB;
            const uint4 a = fa[u & 1][x == 1][m], b = fb[u & 1][x == 2][n];
            if constexpr (SPLIT)
                acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a),
                                                                  __builtin_bit_cast(half8, b), acc[m][n], 0, 0, 0);
            else
                acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                                   __builtin_bit_cast(bf16x8, b), acc[m][n], 0, 0, 0);
            // Reads and loads alternate until either runs out.
            const int upto = (i + 1) * kEvents / kMfma;
#pragma unroll
            for (; event < upto; event++)
            {
                constexpr int kBoth = kLoad ? 2 * (kReads < kLoads ? kReads : kLoads) : 0;
                const bool is_read = event < kBoth ? event % 2 == 0 : kReads >= kLoads || !kLoad;
                const int at = event < kBoth ? event / 2 : event - kBoth / 2;
                if (is_read)
                {
                    if (next >= 0)
                        read(buf, next, at);
                }
                else
                    stage_load(at, la, lb);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Stage t + STAGES is loaded into stage t's buffer once every wave has read
    // all of that (the barrier before the last unit), with STAGES - 1 stages in
    // flight. The last stages wait for everything: their loads are fewer.
#pragma unroll
    for (int s = 0; s < STAGES; s++)
        if (s < stages)
            stage(s, s);
    if (STAGES < stages)
        arrive<(STAGES - 1) * kLoads>();
    else
        arrive<0>();
#pragma unroll
    for (int i = 0; i < kReads; i++)
        read(0, 0, i);
    using Loads = std::integral_constant<bool, true>;
    using NoLoads = std::integral_constant<bool, false>;
    int buf = 0, t = 0;
    auto step = [&](auto loads) {
        constexpr bool kLoad = decltype(loads)::value;
#pragma unroll
        for (int u = 0; u + 1 < kUnits; u++)
            multiply(u, buf, u + 1, NoLoads(), 0);
        if (kLoad)
            arrive<(STAGES - 2) * kLoads>();
        else
            arrive<0>();
        const int used = buf;
        buf = buf + 1 == STAGES ? 0 : buf + 1;
        multiply(kUnits - 1, buf, 0, loads, used);
        if (kLoad)
            next_stage();
    };
    for (const int end = stages - STAGES - (ragged ? 1 : 0); t < end; t++)
        step(Loads());
    for (; t + 1 < stages; t++)
    {
        const int used = buf;
        step(NoLoads());
        if (ragged && t + STAGES == stages - 1)
            stage(t + STAGES, used);
    }
#pragma unroll
    for (int u = 0; u < kUnits; u++)
        multiply(u, buf, u + 1 < kUnits ? u + 1 : -1, NoLoads(), 0);

    // Epilogue: 32 rows of a wave's tile at a time through its own part of LDS
    // (accumulator e: column lane % 32, row 8 (e / 4) + 4 (lane / 32) + e % 4),
    // then 8 columns a lane, so that rows are read and written in 16-byte
    // pieces. Rows and columns with a NaN or an infinity are left to
    // finish_non_finite.
    constexpr int kPitch = NB * 32 + 4;
    float* part = reinterpret_cast<float*>(smem) + wave * 32 * kPitch;
    int* meta_row = reinterpret_cast<int*>(smem + kWaves * 32 * kPitch * 4);
    int* meta_col = meta_row + BM;
    const int width = EPI == kGemmSwiGlu ? g.n >> 1 : g.n;
    arrive<0>();
    if (SPLIT)
    {
        for (int i = threadIdx.x; i < BM; i += kWaves * 64)
            meta_row[i] = g.meta_a[min(row0 + i, g.m - 1)];
        for (int i = threadIdx.x; i < BN; i += kWaves * 64)
            meta_col[i] = g.meta_w[weight_row<EPI>(g, col0, i) + (EPI == kGemmSwiGlu && (i & 16) ? width : 0)];
        __syncthreads();
    }
    int flags = 0;
    constexpr int kOutCols = EPI == kGemmSwiGlu ? NB * 16 : NB * 32; // of a wave's tile
    constexpr int kChunks = kOutCols / 8;
    const int out_col0 = (EPI == kGemmSwiGlu ? col0 >> 1 : col0) + wn * kOutCols;
#pragma unroll
    for (int m = 0; m < MB; m++)
    {
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                part[(8 * (e >> 2) + 4 * (lane >> 5) + (e & 3)) * kPitch + n * 32 + (lane & 31)] = acc[m][n][e];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int i = lane; i < 32 * kChunks; i += 64)
        {
            const int r = i / kChunks, ch = i % kChunks;
            const int rl = (wm * MB + m) * 32 + r;
            const int row = row0 + rl, c = out_col0 + 8 * ch;
            if (row >= g.m || c >= width)
                continue;
            // SwiGLU: 16 gate columns, then 16 input columns.
            const int jl = EPI == kGemmSwiGlu ? (ch >> 1) * 32 + (ch & 1) * 8 : 8 * ch;
            float y[8], z[8];
            load8<false>(part, r * kPitch + jl, y);
            if (EPI == kGemmSwiGlu)
                load8<false>(part, r * kPitch + jl + 16, z);
            int bad = 0;
            if (SPLIT)
            {
                const int ma = meta_row[rl];
                const int* mc = meta_col + wn * NB * 32 + jl;
#pragma unroll
                for (int e = 0; e < 8; e++)
                {
                    int f = ma | mc[e];
                    y[e] = ldexpf(y[e], -row_shift(ma) - row_shift(mc[e]));
                    if (EPI == kGemmSwiGlu)
                    {
                        f |= mc[e + 16];
                        z[e] = ldexpf(z[e], -row_shift(ma) - row_shift(mc[e + 16]));
                    }
                    bad |= f & (kRowNan | kRowInf) ? 1 << e : 0;
                }
                flags |= bad;
            }
            if (EPI == kGemmSwiGlu)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    y[e] = silu_mul<!SPLIT>(y[e], z[e]);
            if (EPI == kGemmGate)
            {
                float x[8], bias[8], gate[8];
                load8<!SPLIT>(g.residual, static_cast<size_t>(row) * g.ldr + c, x);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    bias[e] = 0.f, gate[e] = 1.f;
                if (g.bias)
                    load8<false>(g.bias, c, bias);
                if (g.gate)
                    load8<false>(g.gate, c, gate);
#pragma unroll
                for (int e = 0; e < 8; e++)
                {
                    y[e] = (y[e] + bias[e]) * gate[e] + x[e];
                    y[e] = g.twice ? y[e] + y[e] : y[e];
                }
            }
            const size_t at = static_cast<size_t>(row) * g.ldo + c;
            if (!SPLIT || !bad)
                store8<!SPLIT>(g.out, at, y);
            else
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (!(bad >> e & 1))
                        static_cast<float*>(g.out)[at + e] = y[e];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (SPLIT && __builtin_expect(__any(flags), 0))
        finish_non_finite<EPI>(g, row0 + wm * MB * 32, MB * 32, out_col0, kOutCols);
}

// Both problems' tiles: BM x BN for the video rows, TM x TN for the text rows,
// whose 64 or so rows would leave most of a large tile to padding.
template <class T, int EPI>
__global__ __launch_bounds__(T::kWaves * 64, T::kWaves* T::kPerCu / 4) void gemm_kernel(const GemmLaunch p)
{
    // Workgroup b runs on XCD b % 8. Each XCD takes a contiguous run of video
    // tiles (its L2 then holds few A and W panels), then a run of text tiles:
    // those are short and fill the gaps that the last round leaves.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    auto before = [&](int tiles, int x) { return x * (tiles >> 3) + min(x, tiles & 7); };
    const int total = p.tiles[0] + p.tiles[1];
    const int mine = before(p.tiles[0], xcd + 1) - before(p.tiles[0], xcd);
    if (slot < mine)
    {
        // Groups of kGroupM row tiles, columns outer.
        constexpr int kGroupM = 8;
        const GemmProblem& g = p.problem[0];
        const int v = before(p.tiles[0], xcd) + slot;
        const int tm = (g.m + T::kBm - 1) / T::kBm, tn = (g.n + T::kBn - 1) / T::kBn;
        const int band = v / (kGroupM * tn);
        const int bm = min(kGroupM, tm - band * kGroupM);
        const int in_band = v - band * kGroupM * tn;
        run_tile<T::kSplit, T::kBm, T::kBn, T::kWgm, T::kWgn, T::kStages, EPI>(
            g, (band * kGroupM + in_band % bm) * T::kBm, in_band / bm * T::kBn);
    }
    else
    {
        const GemmProblem& g = p.problem[1];
        const int v = before(total, xcd) - before(p.tiles[0], xcd) + slot - mine;
        const int tm = (g.m + T::kTm - 1) / T::kTm;
        run_tile<T::kSplit, T::kTm, T::kTn, T::kTwgm, T::kTwgn, T::kTstages, EPI>(g, v % tm * T::kTm,
                                                                                              v / tm * T::kTn);
    }
}


constexpr long long kCus = 256;

// ---- splitting fp32 rows ----

constexpr int kSplitThreads = 256; // four rows at a time, one wave each

template <bool ALIGNED>
__device__ __forceinline__ void load_row8(const float* p, float (&v)[8])
{
    if (ALIGNED)
    {
        const float4 a = *reinterpret_cast<const float4*>(p);
        const float4 b = *reinterpret_cast<const float4*>(p + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    }
    else
    {
#pragma unroll
        for (int e = 0; e < 8; e++)
            v[e] = p[e];
    }
}

// One wave a row: bound by HBM, 4 bytes read and 4 written a value, 5.4 TB/s at
// [7680][2560]. CHUNKS > 0: a row of up to 512 CHUNKS values stays in registers between the
// scan and the split; 0: rows of any width, read twice.
template <int CHUNKS, bool ALIGNED>
__global__ __launch_bounds__(kSplitThreads) void split_rows_kernel(const SplitLaunch p)
{
    const int lane = threadIdx.x & 63;
    int row = __builtin_amdgcn_readfirstlane(blockIdx.x * (kSplitThreads / 64) + (threadIdx.x >> 6));
    int part = 0;
#pragma unroll
    for (; part < kSplitParts - 1; part++)
    {
        if (row < p.part[part].rows)
            break;
        row -= p.part[part].rows;
    }
    const SplitRows& s = p.part[part];
    if (row >= s.rows)
        return;
    const float* in = s.in + static_cast<size_t>(row) * p.width;
    char* out = static_cast<char*>(s.out) + static_cast<size_t>(row) * p.groups * kStageBytes;
    const int padded = p.groups * kGroup;
    uint32_t max = 0;
    int flags = 0;
    constexpr int kRegs = CHUNKS > 0 ? CHUNKS : 1;
    float v[kRegs][8];
    if (CHUNKS > 0)
    {
#pragma unroll
        for (int j = 0; j < kRegs; j++)
        {
            const int k = (lane + 64 * j) * 8;
            if (k < p.width)
                load_row8<ALIGNED>(in + k, v[j]);
            else
#pragma unroll
                for (int e = 0; e < 8; e++)
                    v[j][e] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < kRegs; j++)
            scan8(v[j], max, flags);
    }
    else
        for (int k = lane * 8; k < p.width; k += 512)
        {
            load_row8<ALIGNED>(in + k, v[0]);
            scan8(v[0], max, flags);
        }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
    {
        const uint32_t m = __shfl_xor(max, off, 64);
        max = m > max ? m : max;
        flags |= __shfl_xor(flags, off, 64);
    }
    const int shift = shift_of(max);
    if (lane == 0)
        s.meta[row] = (shift + kShiftBias) | flags;
    if (CHUNKS > 0)
    {
#pragma unroll
        for (int j = 0; j < kRegs; j++)
        {
            const int k = (lane + 64 * j) * 8;
            if (k < padded)
                store_planes(out, k, v[j], shift);
        }
    }
    else
        for (int k = lane * 8; k < padded; k += 512)
        {
            if (k < p.width)
                load_row8<ALIGNED>(in + k, v[0]);
            else
#pragma unroll
                for (int e = 0; e < 8; e++)
                    v[0][e] = 0.f;
            store_planes(out, k, v[0], shift);
        }
}

// A tile shape: video tile, waves, stages, workgroups a CU, and the text tile.
template <bool SPLIT, int BM, int BN, int WGM, int WGN, int STAGES, int PER_CU, int TN, int TSTAGES>
struct Shape
{
    static constexpr bool kSplit = SPLIT;
    static constexpr int kBm = BM, kBn = BN, kWgm = WGM, kWgn = WGN, kStages = STAGES, kPerCu = PER_CU;
    static constexpr int kWaves = WGM * WGN;
    static constexpr int kTm = 64, kTn = TN, kTwgm = 2, kTwgn = kWaves / 2, kTstages = TSTAGES;
    static constexpr int kLds = STAGES * (BM + BN) * kStageBytes;
    static_assert(kLds * PER_CU <= 160 * 1024 && TSTAGES * (kTm + TN) * kStageBytes <= kLds, "LDS of a CU");
    static_assert(kWaves * 32 * (BN / WGN + 4) * 4 + (BM + BN) * 4 <= kLds &&
                      kWaves * 32 * (TN / kTwgn + 4) * 4 + (kTm + TN) * 4 <= kLds,
                  "the epilogue's LDS");
};

template <class T, int EPI>
hipError_t launch_tile(GemmLaunch p, hipStream_t stream)
{
    const GemmProblem &v = p.problem[0], &t = p.problem[1];
    p.tiles[0] = ((v.m + T::kBm - 1) / T::kBm) * ((v.n + T::kBn - 1) / T::kBn);
    p.tiles[1] = t.m > 0 ? ((t.m + T::kTm - 1) / T::kTm) * ((t.n + T::kTn - 1) / T::kTn) : 0;
    hipLaunchKernelGGL((gemm_kernel<T, EPI>), dim3(p.tiles[0] + p.tiles[1]), dim3(T::kWaves * 64), T::kLds, stream, p);
    return hipGetLastError();
}

template <class T>
hipError_t launch_epilogue(const GemmLaunch& p, hipStream_t stream)
{
    switch (p.epilogue)
    {
    case kGemmStore:
        return launch_tile<T, kGemmStore>(p, stream);
    case kGemmGate:
        return launch_tile<T, kGemmGate>(p, stream);
    default:
        return launch_tile<T, kGemmSwiGlu>(p, stream);
    }
}

// The video tiles and what they cost: a launch takes about
// start + K / 2560 x (stage + share x tiles / CUs + round x (tiles of the
// fullest CU)) us. Small tiles fill the chip and leave the last round full,
// large ones read less LDS and L2 per MFMA; which wins lies at other rows for
// every width, so the estimate decides. It was fitted to all eight tiles at 96
// launches (81 .. 9200 rows, K 1024 .. 6912, N 1024 .. 13824, 64 text rows, weights
// from HBM): its choice is the best tile at 77 of them, 2 % behind it on average.
struct Tile
{
    int bm, bn;
    struct
    {
        float start, stage, share, round;
    } cost[2]; // bf16, split
};

constexpr Tile kTiles[] = {
    {256, 256, {{4.9f, 3.3f, 0.f, 52.6f}, {6.8f, 0.6f, 64.f, 77.1f}}},
    {256, 192, {{0.4f, 0.f, 23.5f, 40.2f}, {6.4f, 28.7f, 81.5f, 68.2f}}},
    {128, 256, {{3.6f, 2.5f, 0.f, 32.6f}, {6.1f, 12.5f, 18.7f, 53.9f}}},
    {128, 192, {{3.2f, 28.5f, 1.1f, 18.5f}, {6.7f, 89.5f, 19.1f, 10.f}}}, // two workgroups a CU
    {128, 192, {{4.9f, 1.2f, 20.5f, 18.2f}, {8.1f, 0.f, 57.5f, 32.3f}}},  // one, deeper
    {128, 128, {{0.3f, 27.4f, 14.8f, 4.9f}, {3.4f, 46.2f, 48.2f, 3.2f}}},
    {64, 128, {{0.3f, 11.9f, 12.4f, 2.9f}, {1.1f, 12.8f, 25.f, 14.1f}}},
    {64, 64, {{0.f, 7.2f, 15.5f, 0.f}, {0.f, 11.2f, 31.5f, 0.f}}},
};

template <bool SPLIT>
hipError_t launch_kind(const GemmLaunch& p, hipStream_t stream)
{
    const GemmProblem& v = p.problem[0];
    int best = 0;
    float least = 0.f;
    for (int i = 0; i < static_cast<int>(sizeof(kTiles) / sizeof(kTiles[0])); i++)
    {
        const Tile& t = kTiles[i];
        const long long tiles = ((v.m + t.bm - 1LL) / t.bm) * ((v.n + t.bn - 1LL) / t.bn);
        const float k = static_cast<float>(v.stages) * (SPLIT ? 32 : 64) / 2560;
        const auto& c = t.cost[SPLIT];
        const float cost = c.start + k * (c.stage + c.share * static_cast<float>(tiles) / kCus +
                                          c.round * static_cast<float>((tiles + kCus - 1) / kCus));
        if (i == 0 || cost < least)
        {
            best = i;
            least = cost;
        }
    }
    switch (best)
    {
    case 0:
        return launch_epilogue<Shape<SPLIT, 256, 256, 2, 4, 2, 1, 256, 3>>(p, stream);
    case 1:
        return launch_epilogue<Shape<SPLIT, 256, 192, 4, 2, 2, 1, 128, 4>>(p, stream);
    case 2:
        return launch_epilogue<Shape<SPLIT, 128, 256, 2, 4, 3, 1, 256, 3>>(p, stream);
    case 3:
        return launch_epilogue<Shape<SPLIT, 128, 192, 2, 2, 2, 2, 192, 2>>(p, stream);
    case 4:
        return launch_epilogue<Shape<SPLIT, 128, 192, 2, 2, 3, 1, 192, 3>>(p, stream);
    case 5:
        return launch_epilogue<Shape<SPLIT, 128, 128, 2, 2, 2, 2, 128, 2>>(p, stream);
    case 6:
        return launch_epilogue<Shape<SPLIT, 64, 128, 2, 2, 3, 2, 128, 3>>(p, stream);
    default:
        return launch_epilogue<Shape<SPLIT, 64, 64, 2, 2, 5, 2, 64, 5>>(p, stream);
    }
}

} // namespace

hipError_t launch_gemm(const GemmLaunch& p, bool split, hipStream_t stream)
{
    const GemmProblem& v = p.problem[0];
    if (v.m <= 0 || v.n <= 0 || v.n % 8 || v.stages <= 0 || (p.epilogue == kGemmSwiGlu && v.n % 16))
        return hipErrorInvalidValue;
    return split ? launch_kind<true>(p, stream) : launch_kind<false>(p, stream);
}

hipError_t launch_split_rows(const SplitLaunch& p, hipStream_t stream)
{
    long long rows = 0;
    bool aligned = p.width % 4 == 0;
    for (const SplitRows& s : p.part)
    {
        rows += s.rows;
        aligned = aligned && (reinterpret_cast<uintptr_t>(s.in) & 15u) == 0;
    }
    if (rows <= 0)
        return hipSuccess;
    if (p.width % 8)
        return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>((rows + 3) / 4)), block(kSplitThreads);
    if (!aligned)
        hipLaunchKernelGGL((split_rows_kernel<0, false>), grid, block, 0, stream, p);
    else if (p.width <= 512 * 6)
        hipLaunchKernelGGL((split_rows_kernel<6, true>), grid, block, 0, stream, p);
    else if (p.width <= 512 * 14)
        hipLaunchKernelGGL((split_rows_kernel<14, true>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((split_rows_kernel<0, true>), grid, block, 0, stream, p);
    return hipGetLastError();
}

} // namespace awa
