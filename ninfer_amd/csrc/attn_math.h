// Device arithmetic shared by the attention kernels (verify_attention.hip, prompt_attention.hip):
// the INT8-G64 decode into FP16 MFMA operands and the lazy online softmax's constants and maxima.
#pragma once

#include "device_utils.h"

namespace nmi {
namespace {

// Probabilities are FP16 exp2(score - m + 8); the reference maximum m moves only when a score
// exceeds it by more than 2^7, so P <= 2^15 stays inside FP16 and most chunks skip the rescale.
constexpr float kPOffset = 8.0f;
constexpr float kLazyTau = 7.0f;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// 8 INT8 codes (two dwords) -> 8 FP16 values, exactly.
__device__ __forceinline__ h8 cvt_codes8(int lo, int hi) {
    const uint32_t w[4] = {
        i8_bytes_to_f16x2<0, 1>(static_cast<uint32_t>(lo)),
        i8_bytes_to_f16x2<2, 3>(static_cast<uint32_t>(lo)),
        i8_bytes_to_f16x2<0, 1>(static_cast<uint32_t>(hi)),
        i8_bytes_to_f16x2<2, 3>(static_cast<uint32_t>(hi)),
    };
    return __builtin_bit_cast(h8, w);
}

__device__ __forceinline__ h8 scale_h8(h8 x, h2 s) {
    h2 p[4];
    __builtin_memcpy(p, &x, sizeof(p));
#pragma unroll
    for (int i = 0; i < 4; ++i) { p[i] *= s; }
    return __builtin_bit_cast(h8, p);
}

// Byte (T & 3) of word (T >> 2) from key slots 2w and 2w+1 -> packed FP16 pair (V transpose).
template <int T, typename V>
__device__ __forceinline__ uint32_t v_pair(const V& a, const V& b) {
    return i8x2_to_f16x2<T & 3>(static_cast<uint32_t>(a[T >> 2]), static_cast<uint32_t>(b[T >> 2]));
}

// Maximum of a lane's 8 scores over the 4 lanes that share its row (lanes c, c+16, c+32, c+48).
// IEEE maximum (NaN-propagating) runs as v_maximum3_f32 on gfx950, without the canonicalizing
// moves fmaxf needs for operands read back from MFMA accumulators; a NaN score makes the row's
// output NaN under either maximum.
__device__ __forceinline__ float fmax_ieee(float a, float b) { return __builtin_elementwise_maximum(a, b); }

__device__ __forceinline__ float score_max(const float (&sv)[8]) {
    float v = fmax_ieee(fmax_ieee(fmax_ieee(sv[0], sv[1]), fmax_ieee(sv[2], sv[3])),
                        fmax_ieee(fmax_ieee(sv[4], sv[5]), fmax_ieee(sv[6], sv[7])));
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmax_ieee(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmax_ieee(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// The FP16 V scales of the lane's group for its 8 keys (4g + j and 16 + 4g + j), as 4 key pairs.
// D = 128: the lane's dims 8c..8c+7 lie in group c >> 3, and a key's scales are one word.
// D = 256: dims 16c..16c+15 lie in group c >> 2, and a key's scales are two words.
template <int D>
__device__ __forceinline__ void v_scale_pairs(const i4 (&vsw)[2][D / 128], int c, h2 (&vsp)[4]) {
    if constexpr (D == 128) {
        const uint32_t vsel = (c >> 3) ? 0x07060302u : 0x05040100u; // FP16 half of this lane's group
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            vsp[2 * half] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(static_cast<uint32_t>(vsw[half][0][1]), static_cast<uint32_t>(vsw[half][0][0]), vsel));
            vsp[2 * half + 1] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(static_cast<uint32_t>(vsw[half][0][3]), static_cast<uint32_t>(vsw[half][0][2]), vsel));
        }
    } else {
        const int grp = c >> 2;                               // FP16 index of the group in a key's 4
        const uint32_t vsel = (grp & 1) ? 0x07060302u : 0x05040100u;
        const int w = grp >> 1;                               // word of the key holding it
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            // keys j and j + 1 of this half: words [2j + w] of the 32 bytes (two i4)
#pragma unroll
            for (int p2 = 0; p2 < 2; ++p2) {
                const uint32_t a = static_cast<uint32_t>(vsw[half][p2][w]);      // key 2 p2
                const uint32_t b = static_cast<uint32_t>(vsw[half][p2][2 + w]);  // key 2 p2 + 1
                vsp[2 * half + p2] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(b, a, vsel));
            }
        }
    }
}

} // namespace
} // namespace nmi
