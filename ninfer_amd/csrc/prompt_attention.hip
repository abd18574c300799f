// Prompt attention (A1/A3 above the verify extents: one sequence, causal) on gfx950.
//
// Semantics (reference include/ninfer/ops/gqa_attention.h:52-73): the new rows are in the cache
// already; query token t attends over every cache row [0, positions[t]] below the envelope, reading
// INT8-G64 codes with FP16 scales or BF16 rows.
//
// What bounds it: with T x G query rows per KV head the products dominate (a 2,048-token prompt at
// 40/8/128 over 2,048 history rows is 129 GFLOP against 59 MB), so each key is decoded once for as many
// rows as a workgroup can hold and everything else is kept off the matrix cores' way:
//  * One workgroup of 8 waves = one tile of query rows (row = token * G + head of the group, so the
//    heads of a token share the keys) of one KV head. The workgroup walks the keys in tiles of
//    16,384 values per plane (128 keys at head_dim 128, 64 at 256): the codes of tile j + 2 are in
//    flight to registers while tile j + 1 is decoded into the spare half of a double LDS buffer (K
//    rows and V^T rows in MFMA operand order, FP16, 16-byte pieces XOR-swizzled so that neither the
//    writes nor the operand reads conflict) and tile j is multiplied. One barrier per tile.
//  * S^T = K' Q^T and O^T = V'^T P^T on 16x16x32 MFMAs, as in verify_attention.hip: the S^T
//    accumulator layout is the P^T operand layout (the V^T key order inside 32 keys follows it), so
//    probabilities stay in registers. Same operand roundings and lazy softmax as the verify kernels; a
//    tile's rows see all keys in one workgroup, so no FP16 partials are written unless the keys are split.
//  * WK waves share a row tile and take different 32-key chunks of each key tile (merged through
//    LDS at the end), so that short prompts still give every CU rows of its own.
//  * A prompt with too few row tiles for the chip also splits the keys over workgroups (FP16 O / l
//    partials in the verify launches' workspace, as theirs are) and merges them in a second launch.
//  * Tiles are dispatched last-first (the last tokens see the most keys), KV head fastest, so an XCD
//    keeps few heads' keys in its L2.
//
// Measured on MI355X (A1, append included) against the verify launches of 32 tokens: 2,048 tokens over
// 2,048 rows at 40/8/128 1,403 -> 187 us (689 TFLOP/s of the causal products; 8,192 tokens 916, where a
// large library product reaches 1,180), BF16 cache 1,804 -> 243 us; 1,000 tokens at 24/4/256 758 -> 46
// us; 65 tokens over 2,048 rows 51 -> 23 us. What is left at 2,048 tokens: MFMA is busy 42% and the VALU
// (decode, exponentials) 57% of the SIMD time (profiles/prompts_and_column_acceptance.txt) and the two hardly
// overlap; issuing the next chunk's S^T under the exponentials (833), alternating the wave halves by
// barriers (842) and raised issue priority (911) were no better than the plain order (919 TFLOP/s at 8,192
// tokens, all four in one build).
#include "attn_math.h"
#include "common.h"
#include "device_utils.h"
#include "ops_internal.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "lds_dma.h"

namespace nmi {
namespace {

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
using u16x2 = unsigned short __attribute__((ext_vector_type(2)));

struct PromptArgs {
    const uint16_t* q;
    const int32_t* positions;
    const int8_t* kc;
    const int8_t* vc;
    const uint16_t* ks;
    const uint16_t* vs;
    const uint16_t* kb;
    const uint16_t* vb;
    void* out;
    int32_t out_f32;
    int32_t P;
    int32_t T;
    int32_t Hq;
    int32_t Hkv;
    int32_t G;
    int32_t tiles;
    int32_t nsplit;   // key splits of a row tile; above 1 the partials go to part_o / part_ml and a merge launch
    uint16_t* part_o; // FP16 O / l [row tile][KV head][split][BM][D]
    float* part_ml;   // FP32 (log2-domain max, row sum), same order
    int32_t max_keys;
    float scale_log2;
};

constexpr int kPromptThreads = 512;

// D: head dimension; BF: BF16 cache; WK: waves that share a row tile over the keys.
template <int D, bool BF, int WK>
struct PromptGeo {
    static constexpr int NT = D == 128 ? 2 : 1;  // 16-row MFMA tiles per wave
    static constexpr int WR = 8 / WK;            // row waves
    static constexpr int BM = 16 * NT * WR;      // query rows per workgroup
    static constexpr int KT = 16384 / D;         // keys per tile
    static constexpr int NCH = KT / 32;          // 32-key chunks per tile
    static constexpr int kRowK = 2 * D;          // LDS bytes of one K row
    static constexpr int kRowV = 2 * KT;         // LDS bytes of one V^T row
    static constexpr int kPlane = 32768;         // one K or V^T plane of a tile
    static constexpr int kBuf = 2 * kPlane;
    // the flag of a second walk, and its bit per key tile: a cache plane of 2^31 bytes has 131,072 tiles
    static constexpr int kSmem = 2 * kBuf + 131072 / 8;
    static_assert(NCH % WK == 0, "every wave takes whole chunks");
};

// 16-byte slot of piece p of V^T row d. ds_read_b128 serves 16 lanes at a time, {0-3, 12-15} of one
// 16-lane group with {4-11} of the next (whose piece differs in bit 0), over 256 B; ds_write_b128
// serves 8 consecutive lanes over 128 B. The operand reads take one piece of rows 16t + c and the
// decode writes one piece of rows 4i + const: both sets fall on distinct slots (counted conflict-free
// on MI355X; the plain bit swap read at half rate).
template <int D>
__device__ __forceinline__ int v_slot(int piece, int d) {
    const int hi = (d >> 2) & 3;
    const int base = hi ^ ((hi & 1) << 1);
    if constexpr (D == 128) {
        return piece ^ (base | (((d ^ (d >> 4)) & 1) << 2) | ((d & 2) << 2));
    } else { // 128-byte rows: d & 1 picks the half of the banks
        return piece ^ (base | ((((d >> 1) ^ (d >> 4)) & 1) << 2));
    }
}

// The K operand's dims run in the order the decode's units leave them: a unit of 16 codes fills the
// 8-dim pieces p and p + D/16 (8 lanes writing pieces 2p would share half of the banks). Piece -> dim.
template <int D, bool BF>
__device__ __forceinline__ int k_dim(int piece) {
    return BF ? 8 * piece : 16 * (piece & (D / 16 - 1)) + 8 * (piece / (D / 16));
}

// One thread's part of a key tile in flight.
template <int D, bool BF>
struct TileRegs;

template <int D>
struct TileRegs<D, false> {
    u4 k[2];             // 16 codes of two (key, 16-dim piece) units
    uint32_t ksc[2];     // their FP16 scales
    uint32_t v[8];       // 4 codes (dims 4 dq ..) of the unit's 8 keys
    i4 vsw[2][D / 128];  // the scales of keys 4g.. and 16 + 4g..
};

template <int D>
struct TileRegs<D, true> {
    u4 k[4];       // 8 values of four (key, 8-dim piece) units
    u2 v[8];       // 4 values of the unit's 8 keys
};

template <int D, bool BF>
struct HeadPlanes {
    __amdgpu_buffer_rsrc_t k, v, ks, vs;
};

template <int D, bool BF>
__device__ __forceinline__ void load_tile(const HeadPlanes<D, BF>& hp, int key0, int tid, TileRegs<D, BF>& r) {
    const int dq = tid % (D / 4);
    const int oct = tid / (D / 4);
    const int kv0 = key0 + 32 * (oct >> 2) + 4 * (oct & 3); // the octet's keys: kv0 + 0..3 and kv0 + 16 + 0..3
    if constexpr (!BF) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int u = tid + kPromptThreads * i;
            const int key = key0 + u / (D / 16);
            const int piece = u % (D / 16);
            r.k[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(hp.k, key * D + 16 * piece, 0, 0));
            r.ksc[i] = __builtin_amdgcn_raw_buffer_load_b16(hp.ks, 2 * (key * (D / 64) + (piece >> 2)), 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            r.v[j] = __builtin_amdgcn_raw_buffer_load_b32(hp.v, (kv0 + (j & 3) + 16 * (j >> 2)) * D + 4 * dq, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int w = 0; w < D / 128; ++w) {
                r.vsw[h][w] = __builtin_bit_cast(i4, __builtin_amdgcn_raw_buffer_load_b128(hp.vs, (kv0 + 16 * h) * (D / 32) + 16 * w, 0, 0));
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = tid + kPromptThreads * i;
            r.k[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(hp.k, (key0 + u / (D / 8)) * 2 * D + 16 * (u % (D / 8)), 0, 0));
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            r.v[j] = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(hp.v, (kv0 + (j & 3) + 16 * (j >> 2)) * 2 * D + 8 * dq, 0, 0));
        }
    }
}

// Decode a thread's part into an LDS buffer. Keys at or past `window` get zero V values (those rows
// may hold anything; their scores are masked). `top` collects the largest bits of the live INT8 scales.
template <int D, bool BF>
__device__ __forceinline__ void store_tile(const TileRegs<D, BF>& r, char* buf, int key0, int window, int tid, u16x2& top) {
    using PG = PromptGeo<D, BF, 1>;
    const int dq = tid % (D / 4);
    const int oct = tid / (D / 4);
    const int kv0 = key0 + 32 * (oct >> 2) + 4 * (oct & 3);
    char* vp = buf + PG::kPlane;
    if constexpr (!BF) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int u = tid + kPromptThreads * i;
            const int key = u / (D / 16);
            const int piece = u % (D / 16);
            const uint32_t sc = r.ksc[i] & 0xffffu;
            top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, key0 + key < window ? sc : 0u));
            const h2 s2 = __builtin_bit_cast(h2, sc | (sc << 16));
            char* row = buf + key * PG::kRowK;
            *reinterpret_cast<h8*>(row + 16 * (piece ^ (key & 15))) =
                scale_h8(cvt_codes8(static_cast<int>(r.k[i][0]), static_cast<int>(r.k[i][1])), s2);
            *reinterpret_cast<h8*>(row + 16 * ((piece + D / 16) ^ (key & 15))) =
                scale_h8(cvt_codes8(static_cast<int>(r.k[i][2]), static_cast<int>(r.k[i][3])), s2);
        }
        h2 vsp[4];
        v_scale_pairs<D>(r.vsw, dq / (D == 128 ? 2 : 4), vsp);
        if (key0 + PG::KT > window) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (kv0 + (j & 3) + 16 * (j >> 2) >= window) { vsp[j >> 1][j & 1] = static_cast<_Float16>(0.0f); }
            }
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) { top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, vsp[w])); }
        const auto put = [&](auto byte) {
            constexpr int B = decltype(byte)::value;
            h2 pr[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) { pr[w] = __builtin_bit_cast(h2, i8x2_to_f16x2<B>(r.v[2 * w], r.v[2 * w + 1])) * vsp[w]; }
            const int d = 4 * dq + B;
            *reinterpret_cast<h8*>(vp + d * PG::kRowV + 16 * v_slot<D>(oct, d)) = __builtin_bit_cast(h8, pr);
        };
        put(std::integral_constant<int, 0>{});
        put(std::integral_constant<int, 1>{});
        put(std::integral_constant<int, 2>{});
        put(std::integral_constant<int, 3>{});
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = tid + kPromptThreads * i;
            const int key = u / (D / 8);
            *reinterpret_cast<u4*>(buf + key * PG::kRowK + 16 * ((u % (D / 8)) ^ (key & 15))) = r.k[i];
        }
        u2 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) { v[j] = r.v[j]; }
        if (key0 + PG::KT > window) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (kv0 + (j & 3) + 16 * (j >> 2) >= window) { v[j] = u2{0u, 0u}; }
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
            u4 pr;
#pragma unroll
            for (int w = 0; w < 4; ++w) { pr[w] = __builtin_amdgcn_perm(v[2 * w + 1][i >> 1], v[2 * w][i >> 1], sel); }
            const int d = 4 * dq + i;
            *reinterpret_cast<u4*>(vp + d * PG::kRowV + 16 * v_slot<D>(oct, d)) = pr;
        }
    }
}

// A scale of 512 or more (an FP16 exponent of 24), NaN included.
__device__ __forceinline__ bool wide_scale(u16x2 top) { return max(top.x, top.y) >= 0x6000; }

// Zeros a thread's infinite and NaN BF16 V values of keys below `window`; returns whether there were any.
template <int D>
__device__ __forceinline__ bool drop_nonfinite(TileRegs<D, true>& r, int key0, int window, int tid) {
    const int oct = tid / (D / 4);
    const int kv0 = key0 + 32 * (oct >> 2) + 4 * (oct & 3);
    bool any = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t x = r.v[j][w];
            const uint32_t bad = ((x & 0x7f807f80u) + 0x00800080u) & 0x80008000u; // an exponent of ones carries out
            any |= bad != 0u && kv0 + (j & 3) + 16 * (j >> 2) < window;
            r.v[j][w] = x & ~((bad >> 15) * 0xffffu);
        }
    }
    return any;
}

// Online-softmax state of one wave.
template <int D, bool BF, int NT>
struct PromptRows {
    u4 q[NT][D / 32];  // B operand of Q^T: rows 16nt + c, dims 32ks + 8g ..
    float rowmul[NT];
    float rowthr[NT];
    int pos[NT];       // the row's last visible key (-1: no row)
    float m[NT];
    f4 l[NT];
    f4 O[NT][D / 16];  // O^T: tile t entry e of lane (c, g) is dim 16t + 4g + e of row 16nt + c
};

// S^T = K' Q^T of chunk ci of the tile in `buf`.
template <int D, bool BF, int NT>
__device__ __forceinline__ void chunk_scores(const char* buf, int ci, int c, int g, const PromptRows<D, BF, NT>& s, f4 (&sacc)[2][NT]) {
    using PG = PromptGeo<D, BF, 1>;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
        const char* krow = buf + (32 * ci + 16 * kt + c) * PG::kRowK;
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            const u4 ka = *reinterpret_cast<const u4*>(krow + 16 * ((4 * ks + g) ^ c));
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const f4 acc = ks == 0 ? f4{0.f, 0.f, 0.f, 0.f} : sacc[kt][nt];
                if constexpr (BF) {
                    sacc[kt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, ka), __builtin_bit_cast(bf8, s.q[nt][ks]), acc, 0, 0, 0);
                } else {
                    sacc[kt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, ka), __builtin_bit_cast(h8, s.q[nt][ks]), acc, 0, 0, 0);
                }
            }
        }
    }
}

// The chunk's scores (-inf where the key is past the row's last one), and the lazy rescale of the state to its
// running maximum (constants and rounding as in verify_attention.hip).
template <int D, bool BF, int NT>
__device__ __forceinline__ void chunk_rescale(const f4 (&sacc)[2][NT], int c0, bool masked, int g, PromptRows<D, BF, NT>& s, float (&sv)[NT][8]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int i = 0; i < 8; ++i) { sv[nt][i] = sacc[i >> 2][nt][i & 3]; }
    }
    if (masked) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int key = c0 + 16 * (i >> 2) + 4 * g + (i & 3);
                sv[nt][i] = key <= s.pos[nt] ? sv[nt][i] : -INFINITY;
            }
        }
    }
    float cmax[NT];
    bool need_any = false;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        cmax[nt] = score_max(sv[nt]);
        need_any |= cmax[nt] > s.m[nt] + s.rowthr[nt];
    }
    if (__any(need_any)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const bool need = cmax[nt] > s.m[nt] + s.rowthr[nt];
            const float mn = need ? cmax[nt] : s.m[nt];
            const float alpha = need ? __builtin_amdgcn_exp2f((s.m[nt] - mn) * s.rowmul[nt]) : 1.0f;
#pragma unroll
            for (int t = 0; t < D / 16; ++t) { s.O[nt][t] *= alpha; }
            s.l[nt] *= alpha;
            s.m[nt] = mn;
        }
    }
}

// O^T += V'^T P^T, l += ones x P^T.
template <int D, bool BF, int NT>
__device__ __forceinline__ void chunk_values(const char* buf, int ci, int c, int g, const float (&sv)[NT][8], PromptRows<D, BF, NT>& s) {
    using PG = PromptGeo<D, BF, 1>;
    u4 ph[NT], pl[NT]; // P^T operand: FP16, or two BF16 terms
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const float bias = s.m[nt] == -INFINITY ? 0.0f : fmaf(-s.m[nt], s.rowmul[nt], kPOffset);
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) { p[i] = __builtin_amdgcn_exp2f(fmaf(sv[nt][i], s.rowmul[nt], bias)); }
        if constexpr (BF) {
            bf8 hi, lo;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                hi[i] = static_cast<__bf16>(p[i]);
                lo[i] = static_cast<__bf16>(p[i] - static_cast<float>(hi[i]));
            }
            ph[nt] = __builtin_bit_cast(u4, hi);
            pl[nt] = __builtin_bit_cast(u4, lo);
        } else {
            h8 x;
#pragma unroll
            for (int i = 0; i < 8; ++i) { x[i] = static_cast<_Float16>(p[i]); }
            ph[nt] = __builtin_bit_cast(u4, x);
        }
    }
    const char* vp = buf + PG::kPlane + c * PG::kRowV;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
        const u4 va = *reinterpret_cast<const u4*>(vp + 16 * t * PG::kRowV + 16 * v_slot<D>(4 * ci + g, 16 * t + c));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if constexpr (BF) {
                s.O[nt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, va), __builtin_bit_cast(bf8, ph[nt]), s.O[nt][t], 0, 0, 0);
                s.O[nt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, va), __builtin_bit_cast(bf8, pl[nt]), s.O[nt][t], 0, 0, 0);
            } else {
                s.O[nt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, va), __builtin_bit_cast(h8, ph[nt]), s.O[nt][t], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        if constexpr (BF) {
            bf8 ones;
#pragma unroll
            for (int i = 0; i < 8; ++i) { ones[i] = static_cast<__bf16>(1.0f); }
            s.l[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, __builtin_bit_cast(bf8, ph[nt]), s.l[nt], 0, 0, 0);
            s.l[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, __builtin_bit_cast(bf8, pl[nt]), s.l[nt], 0, 0, 0);
        } else {
            const h8 ones = {1, 1, 1, 1, 1, 1, 1, 1};
            s.l[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, __builtin_bit_cast(h8, ph[nt]), s.l[nt], 0, 0, 0);
        }
    }
}

// ---- tiles that need care ------------------------------------------------------------------------
//
// The FP16 operands K' and V' cannot hold a code times a scale of 512 or more, and a masked key's zero
// probability times an infinite V is NaN on the matrix cores. Both are rare (outliers of a cache), so the loop over
// the tiles only notices them; a workgroup that did walks its keys once more, with the forms below in the
// tiles that have such values.
// One K group of scale 600 in the history, 512 tokens at 40/8/128 on MI355X: over 2,000 rows 191 us (64 without it;
// verify launches 1,040, whose merge computes the group's split again), over 8,000 rows 439 (180; 2,975).

// S^T of one 32-key chunk with FP32 operands: FP32(code) * scale (reference decode
// include/ninfer/ops/gqa_attention.h:30), q in FP32 in the units of the wave's FP16 operand.
template <int D, int NT>
__device__ __forceinline__ void scores_f32(const PromptArgs& a, const HeadPlanes<D, false>& hp, int h, int c0, int row0, int rows, int c, int g,
                                           const float (&rowmul)[NT], f4 (&sacc)[2][NT]) {
    const uint16_t* src[NT];
    float factor[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int r = min(row0 + 16 * nt + c, rows - 1); // rows past the end are masked
        const int t = r / a.G;
        src[nt] = a.q + static_cast<int64_t>(D) * (h * a.G + (r - t * a.G) + static_cast<int64_t>(a.Hq) * t);
        factor[nt] = a.scale_log2 / rowmul[nt]; // an exact power of two
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) { sacc[kt][nt] = f4{0.f, 0.f, 0.f, 0.f}; }
    }
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
        const int key = c0 + 16 * kt + c;
#pragma unroll 1
        for (int ks = 0; ks < D / 32; ++ks) {
            const int d0 = 8 * (4 * ks + g);
            const u2 code = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(hp.k, key * D + d0, 0, 0));
            const float sc = f16_bits_to_f32(__builtin_amdgcn_raw_buffer_load_b16(hp.ks, 2 * (key * (D / 64) + d0 / 64), 0, 0));
            u4 q[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) { q[nt] = *reinterpret_cast<const u4*>(src[nt] + d0); }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float k = static_cast<float>(static_cast<int8_t>(code[e >> 2] >> (8 * (e & 3)))) * sc;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float x = __uint_as_float((e & 1) ? q[nt][e >> 1] & 0xffff0000u : q[nt][e >> 1] << 16) * factor[nt];
                    sacc[kt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, x, sacc[kt][nt], 0, 0, 0);
                }
            }
        }
    }
}

// Four V values (dims d0 .. d0 + 3) of a key, in FP32.
template <int D, bool BF>
__device__ __forceinline__ f4 v_values(const HeadPlanes<D, BF>& hp, int key, int d0) {
    if constexpr (BF) {
        const u2 w = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(hp.v, 2 * (key * D + d0), 0, 0));
        return f4{__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16),
                  __uint_as_float(w[1] & 0xffff0000u)};
    } else {
        const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(hp.v, key * D + d0, 0, 0);
        const float sc = f16_bits_to_f32(__builtin_amdgcn_raw_buffer_load_b16(hp.vs, 2 * (key * (D / 64) + d0 / 64), 0, 0));
        return f4{static_cast<float>(static_cast<int8_t>(w)), static_cast<float>(static_cast<int8_t>(w >> 8)),
                  static_cast<float>(static_cast<int8_t>(w >> 16)), static_cast<float>(static_cast<int8_t>(w >> 24))} * sc;
    }
}

// O^T += V^T P^T of one chunk with FP32 operands (infinite and NaN values left out), l += sum of P.
// p[nt][i] of lane (c, g): key c0 + 16 (i >> 2) + 4g + (i & 3) of row 16nt + c, which is the B operand of step i.
template <int D, int NT>
__device__ __forceinline__ void values_f32(const HeadPlanes<D, false>& hp, int c0, int c, int g, const float (&p)[NT][8],
                                           f4 (&O)[NT][D / 16], f4 (&l)[NT]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int key = c0 + 16 * (i >> 2) + 4 * g + (i & 3);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) { l[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(1.0f, p[nt][i], l[nt], 0, 0, 0); }
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            if (t % 4 == 0) { __builtin_amdgcn_sched_barrier(0); } // few loads at once: the state fills the registers
            const int d = 16 * t + c;
            const float code = static_cast<float>(static_cast<int8_t>(__builtin_amdgcn_raw_buffer_load_b8(hp.v, key * D + d, 0, 0)));
            const float v = code * f16_bits_to_f32(__builtin_amdgcn_raw_buffer_load_b16(hp.vs, 2 * (key * (D / 64) + d / 64), 0, 0));
            const float x = __builtin_isfinite(v) ? v : 0.0f;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) { O[nt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, p[nt][i], O[nt][t], 0, 0, 0); }
        }
    }
}

// A chunk's probabilities in FP32.
template <int D, bool BF, int NT>
__device__ __forceinline__ void chunk_probabilities(const float (&sv)[NT][8], const PromptRows<D, BF, NT>& s, float (&p)[NT][8]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            p[nt][i] = s.m[nt] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(fmaf(sv[nt][i] - s.m[nt], s.rowmul[nt], kPOffset));
        }
    }
}

// The infinite and NaN V values of a chunk, to the rows that give their key a probability above zero only.
template <int D, bool BF, int NT>
__device__ __forceinline__ void add_nonfinite(const HeadPlanes<D, BF>& hp, int c0, int window, int c, int g, const float (&p)[NT][8],
                                              f4 (&O)[NT][D / 16]) {
#pragma unroll 1
    for (int kk = 0; kk < 32; ++kk) {
        const int key = c0 + kk;
        if (key >= window) { break; }
        bool any = false;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            if (t % 4 == 0) { __builtin_amdgcn_sched_barrier(0); }
            const f4 v = v_values<D, BF>(hp, key, 16 * t + 4 * g);
            any |= !(__builtin_isfinite(v[0]) && __builtin_isfinite(v[1]) && __builtin_isfinite(v[2]) && __builtin_isfinite(v[3]));
        }
        if (!__any(any)) { continue; }
        const int i = 4 * (kk >> 4) + (kk & 3);
        const int from = 16 * ((kk >> 2) & 3) + c;
        float pk[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float x = p[nt][0];
#pragma unroll
            for (int e = 1; e < 8; ++e) { x = i == e ? p[nt][e] : x; }
            pk[nt] = __shfl(x, from, 64);
        }
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            if (t % 4 == 0) { __builtin_amdgcn_sched_barrier(0); }
            const f4 v = v_values<D, BF>(hp, key, 16 * t + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (__builtin_isfinite(v[e])) { continue; }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    if (pk[nt] != 0.0f) { O[nt][t][e] = fmaf(pk[nt], v[e], O[nt][t][e]); }
                }
            }
        }
    }
}

// A workgroup's part: one row tile of one KV head over one key split. CARE: the walk with the forms above.
// Returns whether this thread saw a value that needs it: a live INT8 scale of 512 or more, or a BF16 result that is
// not finite.
template <int D, bool BF, int WK, bool CARE>
__device__ __forceinline__ bool prompt_tile(const PromptArgs& a, char* smem) {
    using PG = PromptGeo<D, BF, WK>;
    constexpr int NT = PG::NT;
    constexpr int KT = PG::KT;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15;
    const int g = lane >> 4;
    const int wr = wave / WK;
    const int wk = wave % WK;
    const int h = static_cast<int>(blockIdx.x) % a.Hkv;
    const int unit = static_cast<int>(blockIdx.x) / a.Hkv;
    const int split = unit % a.nsplit;
    const int tile = a.tiles - 1 - unit / a.nsplit;
    const int rows = a.T * a.G; // of this KV head
    const int r0 = tile * PG::BM;
    HeadPlanes<D, BF> hp;
    {
        const int64_t plane = static_cast<int64_t>(a.P) * D;
        if constexpr (!BF) {
            hp.k = raw_buffer(a.kc + h * plane, plane);
            hp.v = raw_buffer(a.vc + h * plane, plane);
            hp.ks = raw_buffer(a.ks + h * (plane / 64), plane / 32);
            hp.vs = raw_buffer(a.vs + h * (plane / 64), plane / 32);
        } else {
            hp.k = raw_buffer(a.kb + h * plane, plane * 2);
            hp.v = raw_buffer(a.vb + h * plane, plane * 2);
        }
    }
    // The first key tile of an unsplit row tile does not depend on the positions: its loads (inside the
    // padded cache) go out before them.
    TileRegs<D, BF> tr;
    if (!CARE && a.nsplit == 1) { load_tile<D, BF>(hp, 0, tid, tr); }
    const int window = max(0, min(a.positions[a.T - 1] + 1, a.max_keys));
    const int t_last = (min(r0 + PG::BM, rows) - 1) / a.G;
    const int kend = min(window, a.positions[t_last] + 1); // keys any row of the tile sees
    int ntile = (max(kend, 0) + KT - 1) / KT;
    const int per = (ntile + a.nsplit - 1) / a.nsplit;
    const int j0 = split * per;
    ntile = min(ntile, j0 + per); // key tiles [j0, ntile) are this workgroup's
    if (!CARE && a.nsplit > 1 && j0 < ntile) { load_tile<D, BF>(hp, j0 * KT, tid, tr); }

    // ---- the wave's rows: Q operand, positions, softmax state
    PromptRows<D, BF, NT> s;
    int wave_min = 0x7fffffff, wave_max_pos = -1; // first and last visible-key bound of the wave's rows
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int r = r0 + 16 * (NT * wr + nt) + c;
        const bool valid = r < rows;
        const int t = valid ? r / a.G : 0;
        const int gi = valid ? r - t * a.G : 0;
        s.pos[nt] = valid ? min(a.positions[t], window - 1) : -1;
        const uint16_t* src = a.q + static_cast<int64_t>(D) * (h * a.G + gi + static_cast<int64_t>(a.Hq) * t);
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            s.q[nt][ks] = valid ? *reinterpret_cast<const u4*>(src + k_dim<D, BF>(4 * ks + g)) : u4{0u, 0u, 0u, 0u};
        }
        if constexpr (BF) {
            s.rowmul[nt] = a.scale_log2;
            s.rowthr[nt] = kLazyTau / a.scale_log2;
        } else {
            // BF16 -> FP16, exact after a per-row power of two (as in verify_attention.hip)
            float amax = 0.0f;
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(s.q[nt][ks][w] << 16)), fabsf(__uint_as_float(s.q[nt][ks][w] & 0xffff0000u))));
                }
            }
            amax = group4_max(amax);
            int fexp = 0;
            if (amax > 0.0f && amax < INFINITY) {
                fexp = 14 - max(static_cast<int>((__float_as_uint(amax) >> 23) & 0xff) - 127, -100);
            }
            const float factor = ldexpf(1.0f, fexp);
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t x = s.q[nt][ks][w];
                    const h2 p = {static_cast<_Float16>(__uint_as_float(x << 16) * factor),
                                  static_cast<_Float16>(__uint_as_float(x & 0xffff0000u) * factor)};
                    s.q[nt][ks][w] = __builtin_bit_cast(uint32_t, p);
                }
            }
            s.rowmul[nt] = ldexpf(a.scale_log2, -fexp);
            s.rowthr[nt] = ldexpf(kLazyTau / a.scale_log2, fexp);
        }
        s.m[nt] = -INFINITY;
        s.l[nt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t8 = 0; t8 < D / 16; ++t8) { s.O[nt][t8] = f4{0.f, 0.f, 0.f, 0.f}; }
        int lo = s.pos[nt], hi = s.pos[nt];
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
            lo = min(lo, __shfl_xor(lo, off, 64));
            hi = max(hi, __shfl_xor(hi, off, 64));
        }
        wave_min = min(wave_min, lo);
        wave_max_pos = max(wave_max_pos, hi);
    }
    wave_min = __builtin_amdgcn_readfirstlane(wave_min);
    wave_max_pos = __builtin_amdgcn_readfirstlane(wave_max_pos);

    u16x2 top_scale = {0, 0};
    if constexpr (!CARE) {
        if (ntile > j0) { store_tile<D, BF>(tr, smem + (j0 & 1) * PG::kBuf, j0 * KT, window, tid, top_scale); }
        if (ntile > j0 + 1) { load_tile<D, BF>(hp, (j0 + 1) * KT, tid, tr); }
        __syncthreads();
#pragma unroll 1
        for (int j = j0; j < ntile; ++j) {
            const char* buf = smem + (j & 1) * PG::kBuf;
            if (j + 1 < ntile) {
                store_tile<D, BF>(tr, smem + ((j + 1) & 1) * PG::kBuf, (j + 1) * KT, window, tid, top_scale);
                if (j + 2 < ntile) { load_tile<D, BF>(hp, (j + 2) * KT, tid, tr); }
            }
#pragma unroll
            for (int cw = 0; cw < PG::NCH / WK; ++cw) {
                const int ci = cw * WK + wk;
                const int c0 = j * KT + 32 * ci;
                if (c0 > wave_max_pos) { continue; }
                f4 sacc[2][NT];
                float sv[NT][8];
                chunk_scores<D, BF, NT>(buf, ci, c, g, s, sacc);
                chunk_rescale<D, BF, NT>(sacc, c0, c0 + 31 > wave_min, g, s, sv);
                chunk_values<D, BF, NT>(buf, ci, c, g, sv, s);
            }
            __syncthreads(); // buf is free, the next tile is in place
        }
    } else {
        // bit j - j0: tile j needs care
        uint32_t* marks = reinterpret_cast<uint32_t*>(smem + 2 * PG::kBuf);
        for (int i = tid; 32 * i < ntile - j0; i += kPromptThreads) { marks[i] = 0u; }
        __syncthreads();
#pragma unroll 1
        for (int j = j0; j < ntile; ++j) {
            load_tile<D, BF>(hp, j * KT, tid, tr);
            bool mark = false;
            if constexpr (BF) { mark = drop_nonfinite<D>(tr, j * KT, window, tid); }
            top_scale = u16x2{0, 0};
            store_tile<D, BF>(tr, smem, j * KT, window, tid, top_scale);
            mark |= wide_scale(top_scale);
            if (mark) { atomicOr(&marks[(j - j0) >> 5], 1u << ((j - j0) & 31)); }
            __syncthreads();
            const bool care = ((marks[(j - j0) >> 5] >> ((j - j0) & 31)) & 1u) != 0u;
#pragma unroll 1
            for (int cw = 0; cw < PG::NCH / WK; ++cw) {
                const int ci = cw * WK + wk;
                const int c0 = j * KT + 32 * ci;
                if (c0 > wave_max_pos || (!BF && care)) { continue; }
                f4 sacc[2][NT];
                float sv[NT][8];
                chunk_scores<D, BF, NT>(smem, ci, c, g, s, sacc);
                chunk_rescale<D, BF, NT>(sacc, c0, true, g, s, sv);
                chunk_values<D, BF, NT>(smem, ci, c, g, sv, s);
                if constexpr (BF) {
                    if (care) {
                        float p[NT][8];
                        chunk_probabilities<D, BF, NT>(sv, s, p);
                        add_nonfinite<D, BF, NT>(hp, c0, window, c, g, p, s.O);
                    }
                }
            }
            __syncthreads();
        }
        if constexpr (!BF) { // the marked tiles (a softmax takes its keys in any order)
#pragma unroll 1
            for (int base = 0; base < ntile - j0; base += 32) {
                uint32_t bits = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(marks[base >> 5])));
#pragma unroll 1
                for (; bits != 0u; bits &= bits - 1u) {
                    const int j = j0 + base + __builtin_ctz(bits);
#pragma unroll 1
                    for (int cw = 0; cw < PG::NCH / WK; ++cw) {
                        const int c0 = j * KT + 32 * (cw * WK + wk);
                        if (c0 > wave_max_pos) { continue; }
                        f4 sacc[2][NT];
                        float sv[NT][8], p[NT][8];
                        scores_f32<D, NT>(a, hp, h, c0, r0 + 16 * NT * wr, rows, c, g, s.rowmul, sacc);
                        chunk_rescale<D, BF, NT>(sacc, c0, true, g, s, sv);
                        chunk_probabilities<D, BF, NT>(sv, s, p);
                        values_f32<D, NT>(hp, c0, c, g, p, s.O, s.l);
                        add_nonfinite<D, BF, NT>(hp, c0, window, c, g, p, s.O);
                    }
                }
            }
        }
    }

    // ---- merge the WK key waves of each row tile through LDS, or take the one wave's rows as they are
    float M[NT], L[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        M[nt] = s.m[nt] == -INFINITY ? -INFINITY : s.m[nt] * s.rowmul[nt];
        L[nt] = s.l[nt][0];
    }
    if constexpr (WK > 1) {
        // [WK - 1][WR][NT][D/16][64] f4 of O, then (m, l): the waves wk > 0 hand theirs to wave wk = 0
        f4* xo = reinterpret_cast<f4*>(smem);
        constexpr int kPer = NT * (D / 16) * 64;
        static_assert((WK - 1) * PG::WR * kPer * 16 + (WK - 1) * PG::WR * NT * 64 * 8 <= 2 * PG::kBuf, "merge exceeds the buffers");
        float2* xm = reinterpret_cast<float2*>(smem + (WK - 1) * PG::WR * kPer * 16);
        if (wk > 0) {
            const int slot = (wk - 1) * PG::WR + wr;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
                for (int t = 0; t < D / 16; ++t) { xo[slot * kPer + (nt * (D / 16) + t) * 64 + lane] = s.O[nt][t]; }
                xm[(slot * NT + nt) * 64 + lane] = float2{M[nt], L[nt]};
            }
        }
        __syncthreads();
        if (wk == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                float mw[WK], wgt[WK], Mx = M[nt], Lx = 0.0f;
                float lw[WK];
                mw[0] = M[nt];
                lw[0] = L[nt];
#pragma unroll
                for (int w = 1; w < WK; ++w) {
                    const float2 x = xm[(((w - 1) * PG::WR + wr) * NT + nt) * 64 + lane];
                    mw[w] = x.x;
                    lw[w] = x.y;
                    Mx = fmax_ieee(Mx, x.x);
                }
#pragma unroll
                for (int w = 0; w < WK; ++w) {
                    wgt[w] = mw[w] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mw[w] - Mx);
                    Lx = fmaf(lw[w], wgt[w], Lx);
                }
#pragma unroll
                for (int t = 0; t < D / 16; ++t) {
                    __builtin_amdgcn_sched_barrier(0); // the tiles' loads one after another: the registers are full
                    f4 o = s.O[nt][t] * wgt[0];
#pragma unroll
                    for (int w = 1; w < WK; ++w) { o += xo[((w - 1) * PG::WR + wr) * kPer + (nt * (D / 16) + t) * 64 + lane] * wgt[w]; }
                    s.O[nt][t] = o;
                }
                L[nt] = Lx;
                M[nt] = Mx;
            }
        }
    }
    bool again = !CARE && wide_scale(top_scale);
    const int64_t part = ((static_cast<int64_t>(tile) * a.Hkv + h) * a.nsplit + split) * PG::BM; // first partial row
    if (wk == 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int rr = 16 * (NT * wr + nt) + c; // row within the tile
            const int r = r0 + rr;
            const float inv = L[nt] > 0.0f ? 1.0f / L[nt] : 0.0f;
            uint32_t top = 0u; // the largest magnitude's bits, doubled
#pragma unroll
            for (int t8 = 0; t8 < D / 16; ++t8) {
                s.O[nt][t8] = L[nt] > 0.0f ? s.O[nt][t8] * inv : f4{0.f, 0.f, 0.f, 0.f};
                if constexpr (BF && !CARE) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) { top = max(top, __float_as_uint(s.O[nt][t8][e]) << 1); }
                }
            }
            again |= top >= 0xff000000u;
            if (a.nsplit > 1) {
                uint16_t* dst = a.part_o + (part + rr) * D + 4 * g;
#pragma unroll
                for (int t8 = 0; t8 < D / 16; ++t8) {
                    const f4 o = s.O[nt][t8];
                    *reinterpret_cast<u2*>(dst + 16 * t8) =
                        u2{static_cast<uint32_t>(f32_to_f16_bits(o[0])) | (static_cast<uint32_t>(f32_to_f16_bits(o[1])) << 16),
                           static_cast<uint32_t>(f32_to_f16_bits(o[2])) | (static_cast<uint32_t>(f32_to_f16_bits(o[3])) << 16)};
                }
            } else if (r < rows) {
                const int t = r / a.G;
                const int64_t first = static_cast<int64_t>(D) * (h * a.G + (r - t * a.G) + static_cast<int64_t>(a.Hq) * t) + 4 * g;
                if (a.out_f32) {
#pragma unroll
                    for (int t8 = 0; t8 < D / 16; ++t8) { *reinterpret_cast<f4*>(static_cast<float*>(a.out) + first + 16 * t8) = s.O[nt][t8]; }
                } else {
#pragma unroll
                    for (int t8 = 0; t8 < D / 16; ++t8) {
                        const f4 o = s.O[nt][t8];
                        *reinterpret_cast<u2*>(static_cast<uint16_t*>(a.out) + first + 16 * t8) =
                            u2{static_cast<uint32_t>(f32_to_bf16_bits(o[0])) | (static_cast<uint32_t>(f32_to_bf16_bits(o[1])) << 16),
                               static_cast<uint32_t>(f32_to_bf16_bits(o[2])) | (static_cast<uint32_t>(f32_to_bf16_bits(o[3])) << 16)};
                    }
                }
            }
        }
    }
    if (a.nsplit > 1 && wk == 0 && g == 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int64_t i = part + 16 * (NT * wr + nt) + c;
            *reinterpret_cast<float2*>(a.part_ml + 2 * i) = float2{M[nt], L[nt]};
        }
    }
    return again;
}

template <int D, bool BF, int WK>
__global__ __launch_bounds__(kPromptThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void prompt_attn_kernel(PromptArgs a) {
    using PG = PromptGeo<D, BF, WK>;
    __shared__ __attribute__((aligned(16))) char smem[PG::kSmem];
    int* flag = reinterpret_cast<int*>(smem + 2 * PG::kBuf);
    if (threadIdx.x == 0) { *flag = 0; } // barriers below
    if (prompt_tile<D, BF, WK, false>(a, smem)) { *flag = 1; }
    __syncthreads();
    if (__builtin_expect(*flag != 0, 0)) {
        __syncthreads(); // the flag is read, the first walk's buffers are free
        (void)prompt_tile<D, BF, WK, true>(a, smem);
    }
}

// One row over the keys [k0, k1) in FP32 (the tiles' FP32 form), for a split whose O / l the FP16 partial
// could not hold: the log2-domain maximum and the sum (with the partials' 2^kPOffset) to every thread, O to
// xo[D]. Whole workgroup.
constexpr int kExactFloats(int D) { return D + kPromptThreads + 16 + 4 * kPromptThreads; }

template <int D>
__device__ void exact_split_row(const PromptArgs& a, int h, int t, int qh, int k0, int k1, float* xs, float& M, float& L, const float*& xo) {
    constexpr int GQ = D / 64;
    constexpr int TPR = D / 4;                  // threads per V row
    constexpr int PARTS = kPromptThreads / TPR; // key parts of a block
    float* xq = xs;                    // [D] q * scale * log2(e)
    float* xp = xs + D;                // probabilities of a block of keys
    float* xr = xp + kPromptThreads;   // reductions
    float* xv = xr + 16;               // [PARTS][D]
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int d4 = 4 * (tid % TPR);
    const int part = tid / TPR;
    const int64_t orow = static_cast<int64_t>(D) * (qh + static_cast<int64_t>(a.Hq) * t);
    const int8_t* kbase = a.kc + static_cast<int64_t>(h) * a.P * D;
    const int8_t* vbase = a.vc + static_cast<int64_t>(h) * a.P * D;
    const uint16_t* ksb = a.ks + static_cast<int64_t>(h) * a.P * GQ;
    const uint16_t* vsb = a.vs + static_cast<int64_t>(h) * a.P * GQ;
    __syncthreads(); // the caller's use of xs is over
    if (tid < D) { xq[tid] = bf16_to_f32(a.q[orow + tid]) * a.scale_log2; }
    __syncthreads();
    M = -INFINITY;
    L = 0.0f;
    f4 O = {0.f, 0.f, 0.f, 0.f};
    for (int base = k0; base < k1; base += kPromptThreads) {
        const int key = base + tid;
        float sc = -INFINITY;
        if (key < k1) {
            sc = 0.0f;
#pragma unroll
            for (int gq = 0; gq < GQ; ++gq) {
                const float ksc = f16_bits_to_f32(ksb[static_cast<int64_t>(key) * GQ + gq]);
                u4 code[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) { code[i] = *reinterpret_cast<const u4*>(kbase + static_cast<int64_t>(key) * D + 64 * gq + 16 * i); }
                float p = 0.0f;
#pragma unroll
                for (int d = 0; d < 64; ++d) {
                    p = fmaf(xq[64 * gq + d], static_cast<float>(static_cast<int8_t>(code[d >> 4][(d >> 2) & 3] >> (8 * (d & 3)))) * ksc, p);
                }
                sc += p;
            }
        }
        const float wm = wave_max(sc);
        if (lane == 0) { xr[wave] = wm; }
        __syncthreads();
        float Mn = M;
        for (int w = 0; w < kPromptThreads / 64; ++w) { Mn = fmaxf(Mn, xr[w]); }
        const float alpha = (M == -INFINITY || Mn == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(M - Mn);
        const float p = (sc == -INFINITY || Mn == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(sc - Mn + kPOffset);
        xp[tid] = p;
        const float wsum = wave_sum(p);
        if (lane == 0) { xr[8 + wave] = wsum; }
        __syncthreads();
        float bs = 0.0f;
        for (int w = 0; w < kPromptThreads / 64; ++w) { bs += xr[8 + w]; }
        L = fmaf(L, alpha, bs);
        f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int j = 0; j < kPromptThreads / PARTS; ++j) {
            const int i = part * (kPromptThreads / PARTS) + j;
            const int k = min(base + i, k1 - 1); // past the end: probability zero
            const uint32_t w = *reinterpret_cast<const uint32_t*>(vbase + static_cast<int64_t>(k) * D + d4);
            const float vs = f16_bits_to_f32(vsb[static_cast<int64_t>(k) * GQ + d4 / 64]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = static_cast<float>(static_cast<int8_t>(w >> (8 * e))) * vs;
                acc[e] = xp[i] != 0.0f ? fmaf(xp[i], x, acc[e]) : acc[e];
            }
        }
        O = O * alpha + acc;
        M = Mn;
        __syncthreads(); // xp and xr are reused
    }
    *reinterpret_cast<f4*>(xv + part * D + d4) = O;
    __syncthreads();
    if (tid < D) {
        float o = 0.0f;
        for (int w = 0; w < PARTS; ++w) { o += xv[w * D + tid]; }
        xp[tid] = o;
    }
    __syncthreads();
    xo = xp;
}

// Log-sum-exp merge of a row's key splits: D / 4 threads per row, four dims each.
template <int D, bool BF>
__global__ __launch_bounds__(kPromptThreads) void prompt_merge_kernel(PromptArgs a, int bm) {
    constexpr int TPR = D / 4;
    constexpr int RPB = kPromptThreads / TPR;
    constexpr int KT = 16384 / D;
    __shared__ __attribute__((aligned(16))) float xs[kExactFloats(D)];
    __shared__ uint32_t redo[RPB]; // per row: the splits to compute again
    const int tid = threadIdx.x;
    if (tid < RPB) { redo[tid] = 0u; }
    __syncthreads();
    const int h = static_cast<int>(blockIdx.x) % a.Hkv;
    const int rb = static_cast<int>(blockIdx.x) / a.Hkv * RPB;
    const int rows = a.T * a.G;
    const int r = rb + tid / TPR;
    const int d = 4 * (tid % TPR);
    float M = -INFINITY, L = 0.0f;
    f4 O = {0.f, 0.f, 0.f, 0.f};
    const auto add = [&](float m, float l, f4 o) { // o: O / l
        const float Mn = fmaxf(M, m);
        const float al = M == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(M - Mn);
        const float be = l * __builtin_amdgcn_exp2f(m - Mn);
        O = O * al + o * be;
        L = fmaf(L, al, be);
        M = Mn;
    };
    if (r < rows) {
        const int64_t first = ((static_cast<int64_t>(r / bm) * a.Hkv + h) * a.nsplit) * bm + r % bm;
        for (int k = 0; k < a.nsplit; ++k) {
            const int64_t i = first + static_cast<int64_t>(k) * bm;
            const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + 2 * i);
            const u2 w = *reinterpret_cast<const u2*>(a.part_o + i * D + d);
            if (ml.y == 0.0f) { continue; } // no visible key (a NaN sum stays: the row's output is 0, as without splits)
            const f4 o = {f16_bits_to_f32(static_cast<uint16_t>(w[0])), f16_bits_to_f32(static_cast<uint16_t>(w[0] >> 16)),
                          f16_bits_to_f32(static_cast<uint16_t>(w[1])), f16_bits_to_f32(static_cast<uint16_t>(w[1] >> 16))};
            if constexpr (!BF) {
                // O / l beyond FP16 (a V scale of 512 or more)
                if (!(__builtin_isfinite(o[0]) && __builtin_isfinite(o[1]) && __builtin_isfinite(o[2]) && __builtin_isfinite(o[3]))) {
                    atomicOr(&redo[tid / TPR], 1u << k);
                }
            }
            add(ml.x, ml.y, o);
        }
    }
    if constexpr (!BF) {
        __syncthreads();
        uint32_t any = 0u;
        for (int i = 0; i < RPB; ++i) { any |= redo[i]; }
        if (any != 0u) {
            // a row with such a split is merged again in the same order, those splits in FP32
            const int window = max(0, min(a.positions[a.T - 1] + 1, a.max_keys));
#pragma unroll 1
            for (int i = 0; i < RPB; ++i) {
                const uint32_t again = redo[i];
                if (again == 0u) { continue; }
                const int rr = rb + i;
                const int t = rr / a.G;
                const int last = (min(rr / bm * bm + bm, rows) - 1) / a.G; // the row tile's last token bounds its key tiles
                const int ntile = (max(min(window, a.positions[last] + 1), 0) + KT - 1) / KT;
                const int per = (ntile + a.nsplit - 1) / a.nsplit;
                const int seen = min(a.positions[t] + 1, window);
                const bool mine = tid / TPR == i;
                if (mine) {
                    M = -INFINITY;
                    L = 0.0f;
                    O = f4{0.f, 0.f, 0.f, 0.f};
                }
                const int64_t first = ((static_cast<int64_t>(rr / bm) * a.Hkv + h) * a.nsplit) * bm + rr % bm;
#pragma unroll 1
                for (int k = 0; k < a.nsplit; ++k) {
                    if ((again >> k) & 1u) {
                        float m, l;
                        const float* xo;
                        exact_split_row<D>(a, h, t, h * a.G + (rr - t * a.G), k * per * KT, min((k + 1) * per * KT, seen), xs, m, l, xo);
                        if (mine && l != 0.0f) { add(m, l, *reinterpret_cast<const f4*>(xo + d) * (1.0f / l)); }
                    } else if (mine) {
                        const int64_t at = first + static_cast<int64_t>(k) * bm;
                        const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + 2 * at);
                        const u2 w = *reinterpret_cast<const u2*>(a.part_o + at * D + d);
                        if (ml.y != 0.0f) {
                            add(ml.x, ml.y, f4{f16_bits_to_f32(static_cast<uint16_t>(w[0])), f16_bits_to_f32(static_cast<uint16_t>(w[0] >> 16)),
                                               f16_bits_to_f32(static_cast<uint16_t>(w[1])), f16_bits_to_f32(static_cast<uint16_t>(w[1] >> 16))});
                        }
                    }
                }
            }
        }
    }
    if (r >= rows) { return; }
    const f4 o = L > 0.0f ? O * (1.0f / L) : f4{0.f, 0.f, 0.f, 0.f};
    const int t = r / a.G;
    const int64_t orow = static_cast<int64_t>(D) * (h * a.G + (r - t * a.G) + static_cast<int64_t>(a.Hq) * t);
    if (a.out_f32) {
        *reinterpret_cast<f4*>(static_cast<float*>(a.out) + orow + d) = o;
    } else {
        *reinterpret_cast<u2*>(static_cast<uint16_t*>(a.out) + orow + d) =
            u2{static_cast<uint32_t>(f32_to_bf16_bits(o[0])) | (static_cast<uint32_t>(f32_to_bf16_bits(o[1])) << 16),
               static_cast<uint32_t>(f32_to_bf16_bits(o[2])) | (static_cast<uint32_t>(f32_to_bf16_bits(o[3])) << 16)};
    }
}

// How a prompt is cut: waves per row tile over the keys and key splits. Measured on MI355X, a key tile
// costs a CU 4.7 us with 256 rows at head_dim 128 (WK = 1), 2.8 us with 128 (2) and 1.95 us with 64 (4);
// 2.75 us with 128 rows at head_dim 256 (1) and 1.95 us with 64 (2); a workgroup about 5 us besides, and
// a merge launch about 5 us. So large tiles win as soon as they fill the chip, small ones and then key
// splits below that. The splits' partials fit the workspace of the verify launches (`bytes`).
struct PromptPlan {
    int wk = 1;
    int nsplit = 1;
};

PromptPlan plan_prompt(int32_t D, int64_t rows, int32_t Hkv, int32_t T, int64_t max_keys, size_t bytes) {
    constexpr double kCus = kAttnTargetWorkgroups / 2;
    const double kt = 16384.0 / D;
    const double longest = static_cast<double>(max_keys) / kt;
    const double mean = (static_cast<double>(max_keys) - 0.5 * T) / kt;
    PromptPlan best;
    double best_us = 1.0e30;
    for (int wk = 1; wk <= (D == 128 ? 4 : 2); wk *= 2) {
        const int64_t bm = (D == 128 ? 256 : 128) / wk;
        const double tile_us = D == 128 ? (wk == 1 ? 4.7 : wk == 2 ? 2.8 : 1.95) : (wk == 1 ? 2.75 : 1.95);
        const int64_t units = (rows + bm - 1) / bm * Hkv;
        const int64_t fit = static_cast<int64_t>(bytes / (static_cast<size_t>(units * bm) * (2 * D + 8)));
        for (int ns = 1; ns == 1 || (ns <= fit && ns <= 16 && 2.0 * ns <= longest); ++ns) {
            const double per_cu = static_cast<double>(units) * ns / kCus;
            double us = ns > 1 ? 5.0 : 0.0;
            if (per_cu <= 1.0) {
                us += 5.0 + tile_us * longest / ns;
            } else {
                us += 5.0 * per_cu + tile_us * (per_cu * mean + 0.5 * longest) / ns;
            }
            if (us < best_us) {
                best_us = us;
                best.wk = wk;
                best.nsplit = ns;
            }
        }
    }
    return best;
}

// The time of plan_prompt's choice by the same model, for the choice between this kernel and verify launches:
// constants fitted to 612 calls on MI355X (nine geometries, 65 to 1,024 tokens over 4,096 to 131,072 rows; 90% within
// 14%).
double plan_us(const PromptPlan& plan, int32_t D, bool bf16, int64_t rows, int32_t Hkv, int32_t T, int64_t max_keys) {
    struct Fit {
        double call, merge, tile[3]; // per key tile, by rows per workgroup: WK = 1, 2, 4
        double far;                  // a tile's cost grows by this share up to a history of 131,072 rows
    };
    constexpr Fit fits[2][2] = {{{8.4, 3.4, {4.0, 2.35, 1.57}, 0.0}, {4.3, 5.3, {5.48, 3.36, 2.09}, 0.1}},
                                {{9.3, 4.0, {2.42, 1.74, 0.0}, 0.02}, {8.9, 2.25, {3.04, 2.16, 0.0}, 0.08}}};
    const Fit& f = fits[D == 128 ? 0 : 1][bf16 ? 1 : 0];
    const double kt = 16384.0 / D;
    const int64_t bm = (D == 128 ? 256 : 128) / plan.wk;
    const double per_cu = static_cast<double>((rows + bm - 1) / bm * Hkv) * plan.nsplit / (kAttnTargetWorkgroups / 2);
    const double longest = static_cast<double>(max_keys) / kt;
    const double tiles = per_cu <= 1.0 ? longest : per_cu * (longest - 0.5 * T / kt) + 0.5 * longest;
    return f.call + (plan.nsplit > 1 ? f.merge : 0.0) + 5.0 * std::max(per_cu, 1.0) +
           f.tile[plan.wk == 1 ? 0 : plan.wk == 2 ? 1 : 2] * (1.0 + f.far * std::min(1.0, static_cast<double>(max_keys) / 131072.0)) * tiles /
               plan.nsplit;
}

template <int D, bool BF>
void launch_prompt(const PromptArgs& args, const PromptPlan& plan, void* workspace, hipStream_t stream) {
    PromptArgs a = args;
    a.nsplit = plan.nsplit;
    const auto go = [&](auto wkc) {
        constexpr int WK = decltype(wkc)::value;
        constexpr int BM = PromptGeo<D, BF, WK>::BM;
        const int64_t rows = static_cast<int64_t>(a.T) * a.G;
        a.tiles = static_cast<int32_t>((rows + BM - 1) / BM);
        a.part_o = static_cast<uint16_t*>(workspace);
        a.part_ml = reinterpret_cast<float*>(a.part_o + static_cast<int64_t>(a.tiles) * a.Hkv * a.nsplit * BM * D);
        hipLaunchKernelGGL((prompt_attn_kernel<D, BF, WK>), dim3(a.tiles * a.Hkv * a.nsplit), dim3(kPromptThreads), 0, stream, a);
        check_launch("prompt_attn_kernel");
        if (a.nsplit > 1) {
            constexpr int RPB = kPromptThreads / (D / 4);
            hipLaunchKernelGGL((prompt_merge_kernel<D, BF>), dim3(static_cast<int>((rows + RPB - 1) / RPB) * a.Hkv), dim3(kPromptThreads), 0, stream, a, BM);
            check_launch("prompt_merge_kernel");
        }
    };
    if (plan.wk == 1) {
        go(std::integral_constant<int, 1>{});
    } else if (plan.wk == 2) {
        go(std::integral_constant<int, 2>{});
    } else if constexpr (D == 128) {
        go(std::integral_constant<int, 4>{});
    }
}

} // namespace

double prompt_attention_us(int32_t T, int32_t Hq, int32_t Hkv, int32_t D, bool bf16, uint32_t max_keys, size_t workspace_bytes) {
    const int64_t rows = static_cast<int64_t>(T) * (Hq / Hkv);
    return plan_us(plan_prompt(D, rows, Hkv, T, max_keys, workspace_bytes), D, bf16, rows, Hkv, T, max_keys);
}

void launch_prompt_attention(const uint16_t* q, const int32_t* positions, int32_t T, int32_t Hq, const CacheRef& c,
                             float scale, uint32_t max_keys, void* workspace, size_t workspace_bytes, void* out, bool out_f32,
                             hipStream_t stream) {
    PromptArgs a{};
    a.q = q;
    a.positions = positions;
    a.kc = c.kc;
    a.vc = c.vc;
    a.ks = c.ks;
    a.vs = c.vs;
    a.kb = c.kb;
    a.vb = c.vb;
    a.out = out;
    a.out_f32 = out_f32 ? 1 : 0;
    a.P = c.P;
    a.T = T;
    a.Hq = Hq;
    a.Hkv = c.Hkv;
    a.G = Hq / c.Hkv;
    a.max_keys = static_cast<int32_t>(max_keys);
    a.scale_log2 = scale * 1.4426950408889634f;
    const PromptPlan plan = plan_prompt(c.D, static_cast<int64_t>(T) * a.G, c.Hkv, T, max_keys, workspace_bytes);
    if (c.D == 128 && c.kb == nullptr) {
        launch_prompt<128, false>(a, plan, workspace, stream);
    } else if (c.D == 128) {
        launch_prompt<128, true>(a, plan, workspace, stream);
    } else if (c.D == 256 && c.kb == nullptr) {
        launch_prompt<256, false>(a, plan, workspace, stream);
    } else if (c.D == 256) {
        launch_prompt<256, true>(a, plan, workspace, stream);
    } else {
        throw Unsupported("prompt attention: head_dim 128 and 256 are built");
    }
}

} // namespace nmi
