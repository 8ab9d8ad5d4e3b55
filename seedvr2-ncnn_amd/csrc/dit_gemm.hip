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
// What bounds the stage loop is the matrix core and, next, LDS: per stage a
// 128 x 192 tile reads 80 KB of operands and writes 40 KB for 36 MFMAs a wave
// (1152 cycles), with two workgroups on a CU so that one's barrier and
// epilogue overlap the other's MFMAs. Measured with the text GEMM of 64 rows
// in the same launch, [2304][2560] by [7680][2560]: 258 us, 361 TFLOP/s of the
// fp32 product (772 us as an fp32 library GEMM alone); SwiGLU pair 13824 wide
// 476 us; [2304][2560] by [2560][2560] 121 us; K = 6912 283 us.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "dit_kernels.h"
#include "dit_split.h"

namespace awa
{
namespace
{

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

typedef __attribute__((address_space(3))) char lds_char;

// 16 bytes a lane from base + offset to the 1 KB of LDS at `lds` (lane order).
// Written out so that the compiler does not wait for it before every LDS read;
// the stage loop waits with vmcnt itself. It has no output register.
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t offset, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base)
                 : "memory");
}

// The weight row behind column j of the tile at col0 (the last one beyond the
// end). SwiGLU tiles take 16 gate columns, then the same 16 input columns.
template <int EPI>
__device__ __forceinline__ int weight_row(const GemmProblem& g, int col0, int j)
{
    if (EPI != kGemmSwiGlu)
        return min(col0 + j, g.n - 1);
    const int cols = g.n >> 1;
    return min((col0 >> 1) + (j >> 5) * 16 + (j & 15), cols - 1) + (j & 16 ? cols : 0);
}

__device__ __forceinline__ float silu_mul(float a, float b)
{
    return a / (1.f + expf(-a)) * b;
}

__device__ __forceinline__ float gate_residual(const GemmProblem& g, float h, float bias, float gate, int row, int c)
{
    const float x = static_cast<const float*>(g.residual)[static_cast<size_t>(row) * g.ldr + c];
    const float r = (h + bias) * gate + x;
    return g.twice ? r + r : r;
}

// One product of rows of which one is not finite, from the planes in fp32:
// an infinity stays one where the split products would give NaN.
__device__ float dot_planes(const GemmProblem& g, int row, int wrow)
{
    const int ma = g.meta_a[row], mw = g.meta_w[wrow];
    if ((ma | mw) & kRowNan)
        return __uint_as_float(0x7fc00000u);
    const char* a = static_cast<const char*>(g.a) + static_cast<size_t>(row) * g.lda;
    const char* w = static_cast<const char*>(g.w) + static_cast<size_t>(wrow) * g.ldw;
    float sum = 0.f;
    for (int t = 0; t < g.groups; t++)
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
        const int f = g.meta_a[row] | g.meta_w[c] | (EPI == kGemmSwiGlu ? g.meta_w[width + c] : 0);
        if (!(f & (kRowNan | kRowInf)))
            continue;
        float r = dot_planes(g, row, c);
        if (EPI == kGemmSwiGlu)
            r = silu_mul(r, dot_planes(g, row, width + c));
        if (EPI == kGemmGate)
            r = gate_residual(g, r, g.bias ? g.bias[c] : 0.f, g.gate ? g.gate[c] : 1.f, row, c);
        static_cast<float*>(g.out)[static_cast<size_t>(row) * g.ldo + c] = r;
    }
}

template <int BM, int BN, int WGM, int WGN, int EPI>
__global__ __launch_bounds__(WGM* WGN * 64, 2) void gemm_kernel(const GemmLaunch p)
{
    constexpr int kWaves = WGM * WGN;
    constexpr int MB = BM / WGM / 32, NB = BN / WGN / 32;
    constexpr int kLoadsA = BM / 8 / kWaves, kLoadsB = BN / 8 / kWaves;
    constexpr int kStageA = BM * kStageBytes, kStageB = BN * kStageBytes;
    extern __shared__ char smem[];

    // Each XCD takes a contiguous run of tiles (its L2 then holds few A and W
    // panels): workgroup b runs on XCD b % 8.
    const int total = p.tiles[0] + p.tiles[1];
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int q = total >> 3, rem = total & 7;
    int v = xcd * q + min(xcd, rem) + slot;
    const int which = v < p.tiles[1] ? 1 : 0;
    v -= which ? 0 : p.tiles[1];
    const GemmProblem& g = p.problem[which];

    // Within a problem: groups of kGroupM row tiles, columns outer.
    constexpr int kGroupM = 8;
    const int tm = (g.m + BM - 1) / BM, tn = (g.n + BN - 1) / BN;
    const int band = v / (kGroupM * tn);
    const int bm = min(kGroupM, tm - band * kGroupM);
    const int in_band = v - band * kGroupM * tn;
    const int row0 = (band * kGroupM + in_band % bm) * BM;
    const int col0 = (in_band / bm) * BN;

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
    {
        const int r = min(row0 + (wave * kLoadsA + i) * 8 + (lane >> 3), g.m - 1);
        off_a[i] = static_cast<uint32_t>(r) * g.lda + piece;
    }
#pragma unroll
    for (int i = 0; i < kLoadsB; i++)
    {
        const int j = (wave * kLoadsB + i) * 8 + (lane >> 3);
        const int r = weight_row<EPI>(g, col0, j);
        off_b[i] = static_cast<uint32_t>(r) * g.ldw + piece;
    }
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char*)smem));
    const char* pa = static_cast<const char*>(g.a);
    const char* pb = static_cast<const char*>(g.w);
    auto stage = [&](int buf) {
        const uint32_t la = lds0 + buf * kStageA + wave * kLoadsA * 1024;
        const uint32_t lb = lds0 + 2 * kStageA + buf * kStageB + wave * kLoadsB * 1024;
#pragma unroll
        for (int i = 0; i < kLoadsA; i++)
            load_to_lds(pa, off_a[i], la + i * 1024);
#pragma unroll
        for (int i = 0; i < kLoadsB; i++)
            load_to_lds(pb, off_b[i], lb + i * 1024);
        pa += kStageBytes;
        pb += kStageBytes;
    };

    f32x16 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                acc[m][n][e] = 0.f;

    const char* ra = smem + (wm * MB * 32 + (lane & 31)) * kStageBytes;
    const char* rb = smem + 2 * kStageA + (wn * NB * 32 + (lane & 31)) * kStageBytes;
    uint32_t pc[4];
#pragma unroll
    for (int s = 0; s < 4; s++)
        pc[s] = ((2 * s + (lane >> 5)) ^ (lane & 7)) * 16;
    auto compute = [&](int buf) {
        const char* ta = ra + buf * kStageA;
        const char* tb = rb + buf * kStageB;
#pragma unroll
        for (int j = 0; j < 2; j++)
        {
            half8 ah[MB], al[MB], bh[NB], bl[NB];
#pragma unroll
            for (int m = 0; m < MB; m++)
                ah[m] = *reinterpret_cast<const half8*>(ta + m * 32 * kStageBytes + pc[j]);
#pragma unroll
            for (int n = 0; n < NB; n++)
                bh[n] = *reinterpret_cast<const half8*>(tb + n * 32 * kStageBytes + pc[j]);
#pragma unroll
            for (int m = 0; m < MB; m++)
                al[m] = *reinterpret_cast<const half8*>(ta + m * 32 * kStageBytes + pc[2 + j]);
#pragma unroll
            for (int n = 0; n < NB; n++)
                bl[n] = *reinterpret_cast<const half8*>(tb + n * 32 * kStageBytes + pc[2 + j]);
#pragma unroll
            for (int m = 0; m < MB; m++)
#pragma unroll
                for (int n = 0; n < NB; n++)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[m], bh[n], acc[m][n], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < MB; m++)
#pragma unroll
                for (int n = 0; n < NB; n++)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[m], bh[n], acc[m][n], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < MB; m++)
#pragma unroll
                for (int n = 0; n < NB; n++)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[m], bl[n], acc[m][n], 0, 0, 0);
        }
    };
    // A stage's loads are complete when every wave's own are (vmcnt) and all
    // have passed the barrier; by then every wave has read the other buffer.
    auto arrive = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    const int groups = g.groups;
    stage(0);
    int t = 0;
    for (; t + 2 <= groups; t += 2)
    {
        arrive();
        stage(1);
        compute(0);
        arrive();
        if (t + 2 < groups)
            stage(0);
        compute(1);
    }
    if (t < groups)
    {
        arrive();
        compute(0);
    }

    // Epilogue. Accumulator e of block (m, n): column lane % 32, row
    // 8 (e / 4) + 4 (lane / 32) + e % 4. Rows and columns with a NaN or an
    // infinity are left to finish_non_finite.
    // The shifts wait in LDS, where the stages were.
    int* meta_row = reinterpret_cast<int*>(smem);
    int* meta_col = meta_row + BM;
    arrive();
    for (int i = threadIdx.x; i < BM; i += kWaves * 64)
        meta_row[i] = g.meta_a[min(row0 + i, g.m - 1)];
    for (int i = threadIdx.x; i < BN; i += kWaves * 64)
        meta_col[i] = g.meta_w[weight_row<EPI>(g, col0, i)];
    __syncthreads();
    const int half = lane >> 5;
    int flags = 0;
    int col[NB], mw[NB], mi[NB];
    float bias[NB], gate[NB];
#pragma unroll
    for (int n = 0; n < NB; n++)
    {
        const int jb = (wn * NB + n) * 32;
        if (EPI == kGemmSwiGlu)
        {
            col[n] = (col0 >> 1) + (jb >> 1) + (lane & 15);
            mw[n] = meta_col[jb + (lane & 15)];
            mi[n] = meta_col[jb + 16 + (lane & 15)];
        }
        else
        {
            col[n] = col0 + jb + (lane & 31);
            mw[n] = meta_col[jb + (lane & 31)];
            if (EPI == kGemmGate)
            {
                const int c = min(col[n], g.n - 1);
                bias[n] = g.bias ? g.bias[c] : 0.f;
                gate[n] = g.gate ? g.gate[c] : 1.f;
            }
        }
    }
    const int width = EPI == kGemmSwiGlu ? g.n >> 1 : g.n;
#pragma unroll
    for (int m = 0; m < MB; m++)
    {
        const int rb = (wm * MB + m) * 32 + 4 * half + (EPI == kGemmSwiGlu ? lane & 16 : 0);
#pragma unroll
        for (int e = 0; e < (EPI == kGemmSwiGlu ? 8 : 16); e++)
        {
            const int rl = rb + 8 * (e >> 2) + (e & 3);
            const int row = row0 + rl;
            const int ma = meta_row[rl];
            float* out = static_cast<float*>(g.out) + static_cast<size_t>(row) * g.ldo;
#pragma unroll
            for (int n = 0; n < NB; n++)
            {
                float a = acc[m][n][e], b = 0.f;
                int f = ma | mw[n];
                if (EPI == kGemmSwiGlu)
                {
                    // Lanes 0..15 of a half hold gate columns, 16..31 input
                    // columns: after the swap the first 16 have both of row
                    // e, the other 16 both of row e + 8.
                    const u32x2 s = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[m][n][e]),
                                                                     __float_as_uint(acc[m][n][e + 8]), false, false);
                    a = __uint_as_float(s[0]);
                    b = ldexpf(__uint_as_float(s[1]), -row_shift(ma) - row_shift(mi[n]));
                    f |= mi[n];
                }
                a = ldexpf(a, -row_shift(ma) - row_shift(mw[n]));
                f &= kRowNan | kRowInf;
                flags |= f;
                if (row < g.m && col[n] < width && !f)
                {
                    if (EPI == kGemmSwiGlu)
                        a = silu_mul(a, b);
                    if (EPI == kGemmGate)
                        a = gate_residual(g, a, bias[n], gate[n], row, col[n]);
                    out[col[n]] = a;
                }
            }
            if (e % 4 == 3)
                __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (__builtin_expect(__any(flags), 0))
        finish_non_finite<EPI>(g, row0 + wm * MB * 32, MB * 32,
                               EPI == kGemmSwiGlu ? (col0 + wn * NB * 32) >> 1 : col0 + wn * NB * 32,
                               EPI == kGemmSwiGlu ? NB * 16 : NB * 32);
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

template <int BM, int BN, int WGM, int WGN, int EPI>
hipError_t launch_tile(GemmLaunch p, hipStream_t stream)
{
    for (int i = 0; i < 2; i++)
        p.tiles[i] = p.problem[i].m > 0
                         ? ((p.problem[i].m + BM - 1) / BM) * ((p.problem[i].n + BN - 1) / BN)
                         : 0;
    constexpr int lds = 2 * (BM + BN) * kStageBytes;
    hipLaunchKernelGGL((gemm_kernel<BM, BN, WGM, WGN, EPI>), dim3(p.tiles[0] + p.tiles[1]), dim3(WGM * WGN * 64), lds,
                       stream, p);
    return hipGetLastError();
}

template <int BM, int BN, int WGM, int WGN>
hipError_t launch_epilogue(const GemmLaunch& p, hipStream_t stream)
{
    switch (p.epilogue)
    {
    case kGemmStore:
        return launch_tile<BM, BN, WGM, WGN, kGemmStore>(p, stream);
    case kGemmGate:
        return launch_tile<BM, BN, WGM, WGN, kGemmGate>(p, stream);
    default:
        return launch_tile<BM, BN, WGM, WGN, kGemmSwiGlu>(p, stream);
    }
}

} // namespace

hipError_t launch_split_gemm(const GemmLaunch& p, hipStream_t stream)
{
    const GemmProblem& v = p.problem[0];
    auto rounds = [&](long long bm, long long bn) {
        long long tiles = 0;
        for (const GemmProblem& q : p.problem)
            if (q.m > 0)
                tiles += ((q.m + bm - 1) / bm) * ((q.n + bn - 1) / bn);
        return (tiles + kCus - 1) / kCus;
    };
    if (v.m <= 0 || v.n <= 0 || v.groups <= 0 || (p.epilogue == kGemmSwiGlu && v.n % 2))
        return hipErrorInvalidValue;
    // Time is about (tiles a CU gets) x (a tile's time): 87 us for a 128 x 192
    // tile of K = 2560 and 62 us for a 128 x 128 one (measured with two
    // workgroups on a CU), so the tile with the lower product is taken: it
    // differs where the last round is nearly empty.
    if (rounds(128, 192) * 87 < rounds(128, 128) * 62)
        return launch_epilogue<128, 192, 2, 2>(p, stream);
    return launch_epilogue<128, 128, 2, 2>(p, stream);
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
