// GEMMs of the DiT block on the matrix cores (gfx950): out = epilogue(A W^T)
// with A the activations [M][K] and W a weight [N][K], both K-contiguous; the
// video and the text branch's GEMM of one step run in one launch.
//
// fp32 operands are split. A row x (of A or of W) is stored as x 2^s = hi + lo
// with s the row's exponent shift (its largest finite value lies in
// [2^14, 2^15)), hi the value rounded to fp16 and lo the rest rounded to fp16:
// 2^-22 of a value down to 2^-18 of the row's largest. The product is hi hi +
// hi lo + lo hi on v_mfma_f32_32x32x16_f16 with fp32 accumulation (the dropped
// lo lo weighs at most 2^-22 of a product), three fp16 MFMAs in place of one
// fp32 product at 1/16 of their rate. Off the 64-bit product by 5.7e-7 (relative
// 2-norm, N(0, 1) by N(0, 0.02), K = 2560) where fp32 MFMAs are off by 9.0e-7.
// Smaller values lose bits, down to all of them: each row's meta holds what its
// planes dropped, and an output of which that could be more than 2^-22 is
// computed from the fp32 rows instead (finish_marked), as is every output of a
// row with a NaN or an infinity. A few in 1e6 outputs of a SwiGLU's second GEMM,
// none of N(0, 1) rows: the 33-frame fp32 block takes 1380 us with the check and
// 1357 without. What the marked ones cost there, beside 2890 us of the library's
// fp32 GEMMs: an infinite weight 2060 us, four hidden features 2^20 larger than the
// rest 2970, every output of two GEMMs marked 5220.
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
                 : "memory", "m0");
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

// silu(a) * b; to be rounded to bf16 (2^-9) on the hardware's exp2 and
// reciprocal, in which a log2(e) is rounded: silu is off by at most 2^-20.8 for
// a >= -10, 2^-19 to -40 and 2^-18 to -87.3, below which it is zero (expf and a
// division: 2^-22.5 to -88.7). The 33-frame bf16 block is 3.69e-3 off its 64-bit
// result with either, and 1.9 % slower with expf and the division.
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

// A row of a split GEMM's operand: its planes where they keep every value's 22
// bits, else the fp32 row.
struct OperandRow
{
    const char* at;
    int shift;
    bool full;
};

__device__ __forceinline__ OperandRow operand_row(const float* full, const void* planes, uint32_t pitch, int width,
                                                  int row, const RowMeta& meta)
{
    if (meta.loss == 0.f)
        return {static_cast<const char*>(planes) + static_cast<size_t>(row) * pitch, meta.shift, false};
    return {reinterpret_cast<const char*>(full + static_cast<size_t>(row) * width), 0, true};
}

__device__ __forceinline__ OperandRow operand_a(const GemmProblem& g, int row)
{
    return operand_row(g.full_a, g.a, g.lda, g.width, row, g.meta_a[row]);
}

// Row c of w, or of w2 (SwiGLU).
__device__ __forceinline__ OperandRow operand_w(const GemmProblem& g, int c, bool second)
{
    return operand_row(second ? g.full_w2 : g.full_w, second ? g.w2 : g.w, g.ldw, g.width, c,
                       g.meta_w[second ? (g.n >> 1) + c : c]);
}

// Eight values of a row as they lie in memory (fp32, or hi and lo), so that a
// load is not waited for before they are used.
struct Raw8
{
    uint4 x, y;
};

__device__ __forceinline__ Raw8 load_operand(const OperandRow& r, int k)
{
    typedef uint32_t uint4u __attribute__((ext_vector_type(4), aligned(4)));
    const char* at = r.at + (r.full ? 4 * k : k / kGroup * kStageBytes + k % kGroup * 2);
    const uint4u x = *reinterpret_cast<const uint4u*>(at);
    const uint4u y = *reinterpret_cast<const uint4u*>(at + (r.full ? 16 : 2 * kGroup));
    return {__builtin_bit_cast(uint4, x), __builtin_bit_cast(uint4, y)};
}

__device__ __forceinline__ void operand_values(const OperandRow& r, const Raw8& raw, float (&v)[8])
{
    const half8 hi = __builtin_bit_cast(half8, raw.x), lo = __builtin_bit_cast(half8, raw.y);
    const float full[8] = {__uint_as_float(raw.x.x), __uint_as_float(raw.x.y), __uint_as_float(raw.x.z),
                           __uint_as_float(raw.x.w), __uint_as_float(raw.y.x), __uint_as_float(raw.y.y),
                           __uint_as_float(raw.y.z), __uint_as_float(raw.y.w)};
#pragma unroll
    for (int e = 0; e < 8; e++)
        v[e] = r.full ? full[e] : ldexpf(static_cast<float>(hi[e]) + static_cast<float>(lo[e]), -r.shift);
}

// One product of two rows, the lanes of a wave along K. Bound by latency: the
// loads of kAhead steps are in flight together.
__device__ __forceinline__ float row_product(const OperandRow& a, const OperandRow& w, int width)
{
    constexpr int kAhead = 4;
    float sum = 0.f;
#pragma unroll 1
    for (int k = (threadIdx.x & 63) * 8; k < width; k += 512 * kAhead)
    {
        Raw8 x[kAhead], y[kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; s++)
        {
            // Past the end: the last eight again, not summed.
            x[s] = load_operand(a, min(k + 512 * s, width - 8));
            y[s] = load_operand(w, min(k + 512 * s, width - 8));
        }
#pragma unroll
        for (int s = 0; s < kAhead; s++)
        {
            float u[8], v[8];
            operand_values(a, x[s], u);
            operand_values(w, y[s], v);
            if (k + 512 * s < width)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    sum = fmaf(u[e], v[e], sum);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
        sum += __shfl_xor(sum, off, 64);
    return sum;
}

// The products of 32 by 32 rows on the fp32 matrix core (lane l holds row
// l % 32 of both and, of every 32 values, the 16 at 16 (l / 32)); laid out as
// the accumulators of run_tile. A step takes whole 128-byte lines of every row
// (the rows of a CU's waves do not fit its L1, so a line read by halves comes
// from L2 twice), and the next step's are loaded while the matrix core works.
__device__ __forceinline__ f32x16 block_product(const OperandRow& a, const OperandRow& w, int width)
{
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; e++)
        acc[e] = 0.f;
    const int first = ((threadIdx.x >> 5) & 1) * 16;
    Raw8 x[2], y[2];
    // Past the rows' end: the last eight values, which a step then takes as zeros.
    auto load = [&](int k) {
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            x[h] = load_operand(a, min(k + first + 8 * h, width - 8));
            y[h] = load_operand(w, min(k + first + 8 * h, width - 8));
        }
    };
    auto step = [&](int k, bool tail) {
        const Raw8 p[2] = {x[0], x[1]}, q[2] = {y[0], y[1]};
        if (!tail)
            load(k + 32);
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            float u[8], v[8];
            operand_values(a, p[h], u);
            operand_values(w, q[h], v);
            if (tail && k + first + 8 * h >= width)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    u[e] = v[e] = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(u[e], v[e], acc, 0, 0, 0);
        }
    };
    load(0);
    int k = 0;
    for (; k + 32 < width; k += 32)
        step(k, false);
    step(k, true);
    return acc;
}

// One output of a split GEMM from its product(s).
template <int EPI>
__device__ __forceinline__ void store_output(const GemmProblem& g, int row, int c, float y, float z)
{
    if (EPI == kGemmSwiGlu)
        y = silu_mul<false>(y, z);
    if (EPI == kGemmGate)
    {
        y = (y + (g.bias ? g.bias[c] : 0.f)) * (g.gate ? g.gate[c] : 1.f) +
            static_cast<const float*>(g.residual)[static_cast<size_t>(row) * g.ldr + c];
        y = g.twice ? y + y : y;
    }
    static_cast<float*>(g.out)[static_cast<size_t>(row) * g.ldo + c] = y;
}

// Up to this many marked outputs of 32 rows of a wave's tile are computed one
// by one (about 6 us each at K = 6912), more of them by blocks of 32 x 32. One
// marked column of all rows (an infinite weight) takes the 33-frame fp32 block
// 2150 us one by one and 2540 by blocks.
constexpr int kFewMarked = 32;

// The marked outputs of a wave's tile (rows from row0, output columns from
// col0), from the fp32 operands. Lane l's marks of 32 rows m: bit 8 s + e is
// column 8 (i % kChunks) + e of row i / kChunks, i = l + 64 s (the epilogue's
// order). Rare: values of one row that differ by more than 2^18 and carry the
// output, infinities and NaN.
template <int EPI, int MB, int NB>
__device__ void finish_marked(const GemmProblem& g, const uint64_t* marks, int row0, int col0)
{
    constexpr bool kPair = EPI == kGemmSwiGlu;
    constexpr int kBlockCols = kPair ? 16 : 32; // output columns of a 32-column block
    constexpr int kChunks = NB * kBlockCols / 8, kSteps = kChunks / 2;
    static_assert(kChunks % 2 == 0 && kSteps <= 8, "marks of a lane in 64 bits");
    const int lane = threadIdx.x & 63;
    const int width = kPair ? g.n >> 1 : g.n;
#pragma unroll 1
    for (int m = 0; m < MB; m++)
    {
        uint64_t mine = marks[m * 64 + lane];
        int count = __popcll(mine);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1)
            count += __shfl_xor(count, off, 64);
        if (count == 0)
            continue;
        if (count <= kFewMarked)
        {
            for (uint64_t lanes; (lanes = __ballot(mine != 0)) != 0;)
            {
                const int from = __ffsll(static_cast<unsigned long long>(lanes)) - 1;
                const int bit = __shfl(__ffsll(static_cast<unsigned long long>(mine)) - 1, from, 64);
                const int i = from + 64 * (bit >> 3);
                const int row = row0 + m * 32 + i / kChunks, c = col0 + 8 * (i % kChunks) + (bit & 7);
                const OperandRow a = operand_a(g, row);
                const float y = row_product(a, operand_w(g, c, false), g.width);
                const float z = kPair ? row_product(a, operand_w(g, c, true), g.width) : 0.f;
                if (lane == from)
                {
                    store_output<EPI>(g, row, c, y, z);
                    mine &= mine - 1;
                }
            }
            continue;
        }
        const int j = kPair ? lane & 15 : lane & 31;
        const bool second = kPair && (lane & 16);
        const OperandRow a = operand_a(g, min(row0 + m * 32 + (lane & 31), g.m - 1));
#pragma unroll 1
        for (int n = 0; n < NB; n++)
        {
            // A block without marks is left out.
            bool any = false;
            for (int i = lane; i < 32 * kChunks; i += 64)
                any |= i % kChunks / (kBlockCols / 8) == n && (mine >> (i >> 6 << 3) & 0xff) != 0;
            if (!__any(any))
                continue;
            const int c = col0 + n * kBlockCols + j;
            const f32x16 acc = block_product(a, operand_w(g, min(c, width - 1), second), g.width);
#pragma unroll
            for (int e = 0; e < 16; e++)
            {
                const float z = kPair ? __shfl_xor(acc[e], 16, 64) : 0.f;
                const int r = 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                const int i = r * kChunks + (n * kBlockCols + j) / 8;
                if (!second && (marks[m * 64 + (i & 63)] >> (8 * (i >> 6) + (j & 7)) & 1))
                    store_output<EPI>(g, row0 + m * 32 + r, c, acc[e], z);
            }
        }
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
    // pieces. SPLIT: an output of which the planes may have lost more than
    // 2^-22 (its rows' losses) is left to finish_marked.
    constexpr int kPitch = NB * 32 + 4;
    float* part = reinterpret_cast<float*>(smem) + wave * 32 * kPitch;
    RowMeta* meta_row = reinterpret_cast<RowMeta*>(smem + kWaves * 32 * kPitch * 4);
    RowMeta* meta_col = meta_row + BM;
    uint64_t* marks = reinterpret_cast<uint64_t*>(meta_col + BN) + wave * MB * 64;
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
    bool marked = false;
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
        uint64_t mine = 0;
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
                const RowMeta ma = meta_row[rl];
                const RowMeta* mc = meta_col + wn * NB * 32 + jl;
#pragma unroll
                for (int e = 0; e < 8; e++)
                {
                    bool keep = fabsf(y[e]) >= ma.loss + mc[e].loss; // false for NaN
                    y[e] = ldexpf(y[e], -ma.shift - mc[e].shift);
                    if (EPI == kGemmSwiGlu)
                    {
                        keep = keep && fabsf(z[e]) >= ma.loss + mc[e + 16].loss;
                        z[e] = ldexpf(z[e], -ma.shift - mc[e + 16].shift);
                    }
                    bad |= keep ? 0 : 1 << e;
                }
                mine |= static_cast<uint64_t>(bad) << (i >> 6 << 3);
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
        if (SPLIT)
        {
            marks[m * 64 + lane] = mine;
            marked |= mine != 0;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if constexpr (SPLIT)
        if (__builtin_expect(__any(marked), 0))
            finish_marked<EPI, MB, NB>(g, marks, row0 + wm * MB * 32, out_col0);
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
            scan8(v[j], max);
    }
    else
        for (int k = lane * 8; k < p.width; k += 512)
        {
            load_row8<ALIGNED>(in + k, v[0]);
            scan8(v[0], max);
        }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
    {
        const uint32_t m = __shfl_xor(max, off, 64);
        max = m > max ? m : max;
    }
    const int shift = shift_of(max);
    float dropped = 0.f;
    if (CHUNKS > 0)
    {
#pragma unroll
        for (int j = 0; j < kRegs; j++)
        {
            const int k = (lane + 64 * j) * 8;
            if (k < padded)
                dropped += store_planes(out, k, v[j], shift);
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
            dropped += store_planes(out, k, v[0], shift);
        }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
        dropped += __shfl_xor(dropped, off, 64);
    if (lane == 0)
        s.meta[row] = {shift, row_loss(dropped)};
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
    static_assert(kWaves * 32 * (BN / WGN + 4) * 4 + (BM + BN) * 8 + kWaves * (BM / WGM / 32) * 512 <= kLds &&
                      kWaves * 32 * (TN / kTwgn + 4) * 4 + (kTm + TN) * 8 + kWaves * 512 <= kLds,
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

// The tile shapes and what they cost: a launch takes about
// start + K / 2560 x (stage + share x video tiles / CUs + round x rounds) us,
// a round being one tile of either branch on every CU: text tiles that open a
// round of their own cost nearly a whole one (3078 rows of 2560 columns, K 6912,
// are 250 + 10 tiles of 128 x 256: 185 us, 136 with 128 x 192). Small tiles fill the
// chip and leave the last round full, large ones read less LDS and L2 per MFMA;
// which wins lies at other rows for every width, so the estimate decides. It was
// fitted at 240 launches (81 .. 9200 video rows, 64 text rows, the four GEMMs of
// hidden 1024, 2048 and 2560; 132 bf16, 108 split; weights from HBM): it takes the
// best shape, or one within 0.5 % of it, at 202, is 0.5 % behind the best on
// average, and at worst 20 % in bf16 (420 x 6144, K 2048: 31 us) and 6 % split. At 280
// launches that were not fitted (other rows of the same widths) it is 0.9 %
// behind on average, at worst 15 % in bf16 and 11 % split.
struct Tile
{
    int bm, bn, tn;
    struct
    {
        float start, stage, share, round;
    } cost[2]; // bf16, split
};

constexpr Tile kTiles[kGemmTiles] = {
    {256, 256, 256, {{3.3f, 14.1f, 24.5f, 37.9f}, {5.2f, 17.7f, 141.2f, 54.2f}}},
    {256, 192, 128, {{4.5f, 4.1f, 23.8f, 32.3f}, {13.5f, 0.f, 103.7f, 46.7f}}},
    {128, 256, 256, {{2.7f, 5.4f, 6.2f, 31.9f}, {10.f, 3.f, 47.7f, 51.2f}}},
    {128, 192, 192, {{7.3f, 13.6f, 7.1f, 17.4f}, {5.1f, 24.9f, 24.3f, 41.7f}}}, // two workgroups a CU
    {128, 192, 192, {{6.4f, 0.3f, 5.7f, 27.7f}, {8.2f, 0.f, 40.5f, 41.f}}},     // one, deeper
    {64, 128, 128, {{1.5f, 8.5f, 4.3f, 11.4f}, {1.7f, 11.3f, 13.1f, 24.f}}},
    {64, 64, 64, {{2.5f, 4.8f, 1.4f, 9.5f}, {0.f, 14.4f, 6.1f, 15.2f}}},
};

template <bool SPLIT>
hipError_t launch_kind(const GemmLaunch& p, int tile, hipStream_t stream)
{
    switch (tile)
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
        return launch_epilogue<Shape<SPLIT, 64, 128, 2, 2, 3, 2, 128, 3>>(p, stream);
    default:
        return launch_epilogue<Shape<SPLIT, 64, 64, 2, 2, 5, 2, 64, 5>>(p, stream);
    }
}

} // namespace

int gemm_tile(const GemmLaunch& p, bool split)
{
    const GemmProblem &v = p.problem[0], &text = p.problem[1];
    int best = 0;
    float least = 0.f;
    for (int i = 0; i < kGemmTiles; i++)
    {
        const Tile& t = kTiles[i];
        const long long tiles = ((v.m + t.bm - 1LL) / t.bm) * ((v.n + t.bn - 1LL) / t.bn);
        const long long text_tiles = ((text.m + 63LL) / 64) * ((text.n + t.tn - 1LL) / t.tn);
        const float k = static_cast<float>(v.stages) * (split ? 32 : 64) / 2560;
        const auto& c = t.cost[split];
        const float cost = c.start + k * (c.stage + c.share * static_cast<float>(tiles) / kCus +
                                          c.round * static_cast<float>((tiles + text_tiles + kCus - 1) / kCus));
        if (i == 0 || cost < least)
        {
            best = i;
            least = cost;
        }
    }
    return best;
}

hipError_t launch_gemm(const GemmLaunch& p, bool split, hipStream_t stream, int tile)
{
    const GemmProblem& v = p.problem[0];
    if (v.m <= 0 || v.n <= 0 || v.n % 8 || v.stages <= 0 || (p.epilogue == kGemmSwiGlu && v.n % 16) ||
        tile >= kGemmTiles)
        return hipErrorInvalidValue;
    if (tile < 0)
        tile = gemm_tile(p, split);
    return split ? launch_kind<true>(p, tile, stream) : launch_kind<false>(p, tile, stream);
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
