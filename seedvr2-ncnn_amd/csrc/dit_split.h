// fp32 rows as two fp16 planes (gfx950 device code): a row x is stored as
// x 2^s = hi + lo with s the row's shift (its largest finite value lies in
// [2^14, 2^15)), hi the value rounded to fp16 and lo the rest rounded to fp16.
// A value keeps 22 bits and the sign down to 2^-18 of the row's largest, fewer
// below that, and none below 2^-40; RowMeta says what the row lost that way.
// Per 32 values: 64 bytes of hi, then 64 bytes of lo, so that one stage of a
// GEMM is 128 contiguous bytes of a row. Rows are padded with zeros to a whole
// number of such groups.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace awa
{

constexpr int kStageBytes = 128; // a group: 32 fp16 hi and 32 fp16 lo
constexpr int kGroup = 32;       // values of a group

// What a GEMM needs to know of a split row beside its planes. loss bounds what
// the planes' missing bits add to an output, as a multiple of the other row:
// an output whose scaled product is not at least the sum of both rows' losses
// is computed from the fp32 rows instead (csrc/dit_gemm.hip). 0: every value
// kept its 22 bits; NaN: the row holds a NaN or an infinity.
struct RowMeta
{
    int shift;
    float loss;
};

// The shift for a row whose largest finite magnitude has these bits: that value
// goes to [2^14, 2^15); subnormal rows as 2^-126, zero rows unshifted.
__device__ __forceinline__ int shift_of(uint32_t max)
{
    return max ? 14 - (static_cast<int>(max >> 23) - (max >> 23 ? 127 : 126)) : 0;
}

// The largest finite magnitude's bits.
__device__ __forceinline__ void scan8(const float (&v)[8], uint32_t& max)
{
#pragma unroll
    for (int e = 0; e < 8; e++)
    {
        const uint32_t b = __float_as_uint(v[e]) & 0x7fffffffu;
        if (b < 0x7f800000u)
            max = b > max ? b : max;
    }
}

__device__ __forceinline__ uint32_t pack_half(_Float16 a, _Float16 b)
{
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, a)) |
           static_cast<uint32_t>(__builtin_bit_cast(uint16_t, b)) << 16;
}

// The two planes of 8 values: hi, then lo, 16 bytes each, 64 bytes apart.
// Returns what they drop of values that keep fewer than 22 bits (those below
// about 2^-18 of the row's largest, and nothing of them below 2^-40), as a sum
// of scaled magnitudes; NaN if a value is not finite.
__device__ __forceinline__ float store_planes(char* row, int k, const float (&v)[8], int shift)
{
    uint32_t h[4], l[4];
    float dropped = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++)
    {
        _Float16 hi[2], lo[2];
#pragma unroll
        for (int i = 0; i < 2; i++)
        {
            const float x = ldexpf(v[2 * e + i], shift);
            hi[i] = static_cast<_Float16>(x);
            const float rest = x - static_cast<float>(hi[i]);
            lo[i] = static_cast<_Float16>(rest);
            const float drop = fabsf(rest - static_cast<float>(lo[i]));
            dropped += drop <= 0x1p-22f * fabsf(x) ? 0.f : drop;
        }
        h[e] = pack_half(hi[0], hi[1]);
        l[e] = pack_half(lo[0], lo[1]);
    }
    // A value that the scaling itself made zero counts as 2^-100.
    if (shift < 0)
#pragma unroll
        for (int e = 0; e < 8; e++)
            dropped += v[e] != 0.f && ldexpf(v[e], shift) == 0.f ? 0x1p-100f : 0.f;
    char* at = row + static_cast<size_t>(k / kGroup) * kStageBytes + (k % kGroup) * 2;
    *reinterpret_cast<uint4*>(at) = make_uint4(h[0], h[1], h[2], h[3]);
    *reinterpret_cast<uint4*>(at + 2 * kGroup) = make_uint4(l[0], l[1], l[2], l[3]);
    return dropped;
}

// The loss of a row whose planes drop that much: times the other row's largest
// scaled value (below 2^15), and at most 2^-22 of the product.
__device__ __forceinline__ float row_loss(float dropped)
{
    return dropped * 0x1p37f;
}

} // namespace awa
