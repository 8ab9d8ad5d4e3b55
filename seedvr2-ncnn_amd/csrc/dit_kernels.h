// Launch interface of the DiT block's row-wise kernels (gfx950). Pointers
// are device pointers; strides are in elements; activations are fp32
// (elemsize 4) or bf16 (elemsize 2), parameter vectors fp32.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace awa
{

struct RowMeta; // csrc/dit_split.h

// ada[r][c] = emb[c][r / 3][r % 3] + learned[r][c] for the 6 rows (attn
// shift, scale, gate, mlp shift, scale, gate) of each branch (learned = null:
// none): the Ada vectors the row kernels below read.
struct AdaPrepare
{
    const void* emb;
    int emb_elemsize;
    const float* learned[2];
    float* ada[2];
    int width;
};

hipError_t launch_ada_prepare(const AdaPrepare& p, hipStream_t stream);

// out = rmsnorm(in) * scale + shift, per row of `width`; scale = shift = null
// skips the modulation.
struct RowNormModulate
{
    const void* in;
    int in_elemsize;
    long long in_stride;
    void* out;
    int out_elemsize;
    long long out_stride;
    int rows, width;
    float eps;
    const float* shift;
    const float* scale;
    // Set: out takes the rows' fp16 planes (csrc/dit_split.h, `groups` groups
    // a row) and meta what belongs to them; full takes the rows themselves
    // (stride width) where the planes lose bits.
    RowMeta* meta = nullptr;
    float* full = nullptr;
    int groups = 0;
};

// Both branches' rows (rows = 0: none), both with meta or both without.
struct RowNormPair
{
    RowNormModulate branch[2];
};

// out = (h + bias) * gate + residual (bias may be null; gate = null takes it as 1).
struct GateResidual
{
    const void* h;
    int h_elemsize;
    long long h_stride;
    const float* bias;
    const void* residual;
    int residual_elemsize;
    long long residual_stride;
    void* out;
    int out_elemsize;
    long long out_stride;
    int rows, width;
    const float* gate;
};

// out[:, c] = silu(in[:, c]) * in[:, width + c].
struct SwiGlu
{
    const void* in;
    int in_elemsize;
    long long in_stride;
    void* out;
    int out_elemsize;
    long long out_stride;
    int rows, width;
};

// fp32 rows split into fp16 planes (csrc/dit_gemm.hip): per 32 values of a
// row 64 bytes of hi and 64 bytes of lo, rows padded with zeros to a whole
// number of such groups, and each row's meta (csrc/dit_split.h).
struct SplitRows
{
    const float* in; // [rows][width], contiguous
    void* out;       // [rows][groups][128 bytes]
    RowMeta* meta;   // [rows]
    int rows;
};

constexpr int kSplitParts = 4;

struct SplitLaunch
{
    SplitRows part[kSplitParts];
    int width, groups;
};

// One GEMM: out = epilogue(A W^T); rows of 128-byte stages (bf16, or split
// planes). out, residual: bf16 or (split) fp32, rows 16-byte aligned.
struct GemmProblem
{
    const void* a;
    const void* w;
    const void* w2;    // SwiGLU: the weight of the second half of the columns
    // split: the meta of A's rows and the weights' (w, then w2), and the fp32
    // operands, rows of `width` values at any 4-byte address: the weights', and
    // A's at least for the rows that lose bits as planes.
    const RowMeta* meta_a;
    const RowMeta* meta_w;
    const float* full_a;
    const float* full_w;
    const float* full_w2;
    int width;
    uint32_t lda, ldw; // row strides in bytes, multiples of 16
    int m, n, stages;
    uint32_t last_bytes; // bf16: bytes of a row in its last stage
    void* out;
    long long ldo; // in elements
    const float* bias;
    const float* gate;
    const void* residual;
    long long ldr;
    int twice;
};

enum GemmEpilogue
{
    kGemmStore = 0, // out = y
    kGemmGate,      // out = (y + bias) * gate + residual, doubled if twice
    kGemmSwiGlu     // out[:, c] = silu(y[:, c]) * y[:, n / 2 + c]
};

struct GemmLaunch
{
    GemmProblem problem[2]; // video, text (m = 0: none)
    int tiles[2];           // set by the launch
    int epilogue;
};

hipError_t launch_split_rows(const SplitLaunch& p, hipStream_t stream);
// The tile shape (0 .. kGemmTiles - 1) that launch_gemm estimates to be the
// fastest; tile >= 0 asks for that one instead.
constexpr int kGemmTiles = 7;
int gemm_tile(const GemmLaunch& p, bool split);
hipError_t launch_gemm(const GemmLaunch& p, bool split, hipStream_t stream, int tile = -1);

hipError_t launch_rmsnorm_modulate(const RowNormPair& pair, hipStream_t stream);
hipError_t launch_gate_residual(const GateResidual& p, hipStream_t stream);
hipError_t launch_swiglu(const SwiGlu& p, hipStream_t stream);
hipError_t launch_double(const void* in, int in_elemsize, long long in_stride, void* out, int out_elemsize,
                         long long out_stride, int rows, int width, hipStream_t stream);

} // namespace awa
