// Gated delta rule over a prompt (gfx950): the recurrence of gdn_snapshot.hip for many tokens, 32 at a
// time on the matrix cores.
//
// Contract as include/ninfer/ops/gated_delta_rule.h:26-55 (state in, state out, one output per token). For a
// chunk of tokens t = 0..31 with decays a_t, let G_t = a_0 .. a_t and D_ti = a_(i+1) .. a_t. With S the
// state before the chunk (rows = value index, columns = key index), the sequential rule
//   d_t = b_t (v_t - a_t S_(t-1) k_t),  S_t = a_t S_(t-1) + d_t k_t^T,  o_t = scale S_t q_t
// unrolls into
//   d_t = b_t (v_t - G_t S k_t) - sum_(i<t) A_ti d_i,   A_ti = b_t D_ti (k_t . k_i)
//   o_t = scale (G_t S q_t) + sum_(i<=t) P_ti d_i,      P_ti = scale D_ti (q_t . k_i)
//   S'  = G_31 S + sum_i D_31,i d_i k_i^T
// so the state is read and written once per 32 tokens, and everything but the substitution for d is a
// matrix product. (The chunked form of the delta rule is published: Yang et al., "Parallelizing Linear
// Transformers with the Delta Rule over Sequence Length" and "Gated Delta Networks"; here the
// substitution is done directly, without forming an inverse.)
//
// Precision: k and q enter as the BF16 values they are (their normalization factors are per-token scalars
// outside the products), and the FP32 operands S and d go through the BF16 matrix cores as three
// BF16 terms that hold all 24 bits, so every product is exact and only FP32 sums round. A, P and the
// substitution are FP32 (P d on the FP32 matrix instruction), the decays exp of differences of a running
// sum in 64 bits. The substitution sums A_ti d_i apart from the right-hand side and subtracts once:
// subtracting term by term rounds at the size of d each time and was worse than the token-by-token
// kernel (state 1.5e-7 from 64 bits over 64 tokens). State against 64 bits, measured: 8.4e-8 to 9.0e-8 for
// 20 to 2,000 tokens (token by token 1.1e-7 to 1.25e-7).
//
// What bounds it: the chain S k -> d -> S' of each chunk. A wave owns 16 state rows (S^T tiles in the
// accumulator layout, which is also the operand layout of the next product, so the state and d never
// leave its registers), two such waves share a workgroup with a third that stages the next chunk's k, q
// and computes its A and P meanwhile: one barrier per chunk.
#include "common.h"
#include "device_utils.h"
#include "gdn_internal.h"
#include "lds_dma.h"

#include <type_traits>

namespace nmi {
namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef uint32_t w4 __attribute__((ext_vector_type(4)));
typedef uint32_t w2 __attribute__((ext_vector_type(2)));

constexpr int kS = 128;           // head dimension
constexpr int kC = 32;            // tokens per chunk
constexpr int kSerial = 2;        // waves that own 16 state rows each
constexpr int kChunkThreads = 64 * (kSerial + 1);
constexpr int kRowBlocks = kS / (16 * kSerial); // workgroups per head
constexpr int kMatStride = 36;    // floats per row of A and P

// One chunk in LDS. Rows of k and q hold the 16-byte pieces (s, g) = dims 32s + {4g..4g+3, 16+4g..+3}
// (the order in which the accumulator layout presents the state's columns), k^T rows the pieces
// g = tokens {4g..4g+3, 16+4g..+3}; pieces XOR-swizzled against bank conflicts.
struct Chunk {
    char k[kC * 2 * kS];
    char q[kC * 2 * kS];
    char kt[kS * 2 * kC];
    float A[kC * kMatStride];
    float P[kC * kMatStride];
    float beta[kC]; // b_t
    float gk[kC];   // b_t G_t |k_t|^-1
    float gq[kC];   // scale G_t |q_t|^-1
    float dk[kC];   // D_31,t |k_t|^-1
    double run[kC]; // g_0 + .. + g_t
    float gc;       // G_31
    float pad[3];
};

__device__ __forceinline__ int row_at(int token, int piece) { return token * (2 * kS) + 16 * (piece ^ (token & 15)); }
__device__ __forceinline__ int kt_at(int dim, int piece) { return dim * (2 * kC) + 16 * (piece ^ ((dim >> 2) & 3)); }

// x = hi + mid + lo exactly (three BF16 terms of 8 bits each).
__device__ __forceinline__ void split3(const float (&x)[8], b8& hi, b8& mid, b8& lo) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        hi[i] = static_cast<__bf16>(x[i]);
        const float r = x[i] - static_cast<float>(hi[i]);
        mid[i] = static_cast<__bf16>(r);
        lo[i] = static_cast<__bf16>(r - static_cast<float>(mid[i]));
    }
}

__device__ __forceinline__ f4 mfma_b(b8 a, b8 b, f4 acc) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0); }

// The staging wave's registers: two (token quad, dim octet) units of k and q, and the decays.
struct Stage {
    w4 k[2][4];
    w4 q[2][4];
    float g, beta; // token lane & 31
};

// Tokens past the prompt read as zero (range-checked buffers of the chunk's rows): with b_t = 0 and decay
// 1 they change nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t chunk_rows(const void* base, int64_t row_bytes, int t0, int T) {
    return raw_buffer(static_cast<const char*>(base) + row_bytes * t0, row_bytes * min(kC, T - t0));
}

__device__ __forceinline__ void stage_load(const GdnArgs& a, int t0, int h, int qh, int lane, Stage& r) {
    const int row = a.Hqk * kS * 2;
    const __amdgpu_buffer_rsrc_t kb = chunk_rows(a.k, row, t0, a.T);
    const __amdgpu_buffer_rsrc_t qb = chunk_rows(a.q, row, t0, a.T);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int unit = lane + 64 * u; // (token quad, dim octet)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int off = (4 * (unit >> 4) + e) * row + (qh * kS + 8 * (unit & 15)) * 2;
            r.k[u][e] = __builtin_bit_cast(w4, __builtin_amdgcn_raw_buffer_load_b128(kb, off, 0, 0));
            r.q[u][e] = __builtin_bit_cast(w4, __builtin_amdgcn_raw_buffer_load_b128(qb, off, 0, 0));
        }
    }
    // lanes 32.. read past the chunk: zeros
    const int off = (lane * a.Hv + h) * 4;
    const int past = lane < kC ? off : 0x7fffff00;
    r.g = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(chunk_rows(a.g, 4 * a.Hv, t0, a.T), past, 0, 0));
    r.beta = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(chunk_rows(a.beta, 4 * a.Hv, t0, a.T), past, 0, 0));
}

// Zeros the staged rows of v whose factors are 0: a squared norm beyond FP32. Their normalized row is 0 where every value
// is finite; a row with an infinite value stays as it is (0 x inf is NaN in its products, as it is in the row).
__device__ __forceinline__ void drop_overflowed(w4 (&v)[2][4], const float* factors, int lane) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int quad = (lane + 64 * u) >> 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 4; ++i) { bad |= (((v[u][e][i] & 0x7f807f80u) + 0x00800080u) & 0x80008000u) != 0u; }
            const uint64_t row = (__ballot(bad) >> (lane & 48)) & 0xffffu; // 16 lanes hold a row
            if (factors[4 * quad + e] == 0.0f && row == 0u) { v[u][e] = w4{0u, 0u, 0u, 0u}; }
        }
    }
}

// The rows of k and q and the columns of k^T of chunk x, from the staging wave's registers.
__device__ __forceinline__ void stage_rows(const Stage& r, Chunk& x, int lane) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int unit = lane + 64 * u;
        const int quad = unit >> 4;
        const int oct = unit & 15;
        const int s = oct >> 2;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 4 * quad + e;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int grp = 2 * (oct & 3) + hf; // 4-dim group of the 32-dim block
                const int at = row_at(t, 4 * s + (grp & 3)) + 8 * (grp >> 2);
                *reinterpret_cast<w2*>(x.k + at) = w2{r.k[u][e][2 * hf], r.k[u][e][2 * hf + 1]};
                *reinterpret_cast<w2*>(x.q + at) = w2{r.q[u][e][2 * hf], r.q[u][e][2 * hf + 1]};
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
            const w2 p = {__builtin_amdgcn_perm(r.k[u][1][i >> 1], r.k[u][0][i >> 1], sel),
                          __builtin_amdgcn_perm(r.k[u][3][i >> 1], r.k[u][2][i >> 1], sel)};
            *reinterpret_cast<w2*>(x.kt + kt_at(8 * oct + i, quad & 3) + 8 * (quad >> 2)) = p;
        }
    }
}

// Products of the chunk's tokens: [token tile][i tile], row 4g + e, column c. The wave's own LDS writes are complete
// before these reads (in-order LDS).
__device__ __forceinline__ void stage_products(const Chunk& x, int c, int g, f4 (&kk)[2][2], f4 (&qk)[2][2], f4 (&qq)[2]) {
    b8 kr[2][4], qr[2][4];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            kr[tt][s] = *reinterpret_cast<const b8*>(x.k + row_at(16 * tt + c, 4 * s + g));
            qr[tt][s] = *reinterpret_cast<const b8*>(x.q + row_at(16 * tt + c, 4 * s + g));
        }
    }
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
        for (int ii = 0; ii <= tt; ++ii) {
            kk[tt][ii] = zero;
            qk[tt][ii] = zero;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                kk[tt][ii] = mfma_b(kr[tt][s], kr[ii][s], kk[tt][ii]);
                qk[tt][ii] = mfma_b(qr[tt][s], kr[ii][s], qk[tt][ii]);
            }
        }
        qq[tt] = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) { qq[tt] = mfma_b(qr[tt][s], qr[tt][s], qq[tt]); }
    }
}

// Per-token factors to x.gk and x.gq: the squared norms sit on the diagonals (lane (c, c / 4), entry c % 4). Returns
// whether a factor is 0.
__device__ __forceinline__ bool stage_factors(bool normalize, const f4 (&kk)[2][2], const f4 (&qq)[2], Chunk& x, int c, int g) {
    bool none = false;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        const float nk = (c & 2) ? ((c & 1) ? kk[tt][tt][3] : kk[tt][tt][2]) : ((c & 1) ? kk[tt][tt][1] : kk[tt][tt][0]);
        const float nq = (c & 2) ? ((c & 1) ? qq[tt][3] : qq[tt][2]) : ((c & 1) ? qq[tt][1] : qq[tt][0]);
        if (g == (c >> 2)) {
            // x / sqrt(sum(x^2) + 1e-6) over the row (gated_delta_rule.h:35-36)
            const float fk = normalize ? 1.0f / sqrtf(nk + 1.0e-6f) : 1.0f;
            const float fq = normalize ? 1.0f / sqrtf(nq + 1.0e-6f) : 1.0f;
            x.gk[16 * tt + c] = fk;
            x.gq[16 * tt + c] = fq;
            none |= fk == 0.0f || fq == 0.0f;
        }
    }
    return none;
}

// Fills chunk x (one wave).
__device__ __forceinline__ void stage_store(const GdnArgs& a, Stage& r, Chunk& x, int lane) {
    const int c = lane & 15;
    const int g = lane >> 4;
    f4 kk[2][2], qk[2][2], qq[2];
    stage_rows(r, x, lane);
    stage_products(x, c, g, kk, qk, qq);
    if (__builtin_expect(__any(stage_factors(a.normalize_qk != 0, kk, qq, x, c, g)), 0)) {
        drop_overflowed(r.k, x.gk, lane);
        drop_overflowed(r.q, x.gq, lane);
        stage_rows(r, x, lane);
        stage_products(x, c, g, kk, qk, qq);
        (void)stage_factors(a.normalize_qk != 0, kk, qq, x, c, g);
    }
    // decays as exp of differences of the running sum of g in 64 bits (beyond +-1000 exp(g) is 0 or
    // infinite either way; a NaN stays)
    const float gg = r.g != r.g ? r.g : fminf(fmaxf(r.g, -1000.0f), 1000.0f);
    const double run = wave_inclusive_scan(static_cast<double>(gg)); // lanes 31.. hold the chunk's sum
    if (lane < kC) {
        x.beta[lane] = r.beta;
        x.run[lane] = run;
    }
    asm volatile("" ::: "memory");
    const auto decay = [](double v) { return expf(static_cast<float>(v)); };
    const double gi[2] = {x.run[c], x.run[16 + c]};
    f4 D[2][2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const double gt = x.run[16 * tt + 4 * g + e];
#pragma unroll
            for (int ii = 0; ii <= tt; ++ii) { D[tt][ii][e] = decay(gt - gi[ii]); }
        }
    }
    const float mine = decay(run);                    // G_t of token t = lane
    const float last = decay(x.run[kC - 1] - run);    // D_31,t
    const float ki[2] = {x.gk[c], x.gk[16 + c]};
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        const f4 bt = *reinterpret_cast<const f4*>(x.beta + 16 * tt + 4 * g);
        const f4 kt = *reinterpret_cast<const f4*>(x.gk + 16 * tt + 4 * g);
        const f4 qt = *reinterpret_cast<const f4*>(x.gq + 16 * tt + 4 * g);
#pragma unroll
        for (int ii = 0; ii <= tt; ++ii) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * tt + 4 * g + e;
                const int i = 16 * ii + c;
                x.A[t * kMatStride + i] = i < t ? bt[e] * (D[tt][ii][e] * (kk[tt][ii][e] * (kt[e] * ki[ii]))) : 0.0f;
                x.P[t * kMatStride + i] = i <= t ? a.scale * (D[tt][ii][e] * (qk[tt][ii][e] * (qt[e] * ki[ii]))) : 0.0f;
            }
        }
    }
    const float kn = x.gk[lane & 31];
    const float qn = x.gq[lane & 31];
    asm volatile("" ::: "memory");
    if (lane < 32) {
        x.gk[lane] = r.beta * (mine * kn);
        x.gq[lane] = a.scale * (mine * qn);
        x.dk[lane] = last * kn;
        if (lane == 31) { x.gc = mine; }
    }
}

// The value of lane group FROM (lanes 16 FROM + c) in every group: v_permlane16_swap leaves the even
// groups' values in one register and the odd ones' in the other, v_permlane32_swap the halves'.
template <int FROM>
__device__ __forceinline__ float from_group(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(a[FROM & 1], a[FROM & 1], false, false);
    return __uint_as_float(b[FROM >> 1]);
}

__global__ __launch_bounds__(kChunkThreads) void gdn_chunk_kernel(GdnArgs a) {
    __shared__ __attribute__((aligned(16))) Chunk chunk[2];
    __shared__ float spill[kSerial][kC][16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Blocks are dealt to the 8 XCDs round-robin: the row blocks of a head, and consecutive heads (which
    // share k and q), go to one XCD and its L2.
    const int per = (a.Hv + 7) / 8; // heads per XCD
    const int idx = static_cast<int>(blockIdx.x) >> 3;
    const int h = (static_cast<int>(blockIdx.x) & 7) * per + idx / kRowBlocks;
    const int rblock = idx % kRowBlocks;
    if (h >= a.Hv) { return; }
    const int qh = h / (a.Hv / a.Hqk);
    const int chunks = (a.T + kC - 1) / kC;
    if (wave == kSerial) {
        // chunk j + 2's loads go out before chunk j + 1 is staged: two register sets, taken in turn
        Stage r0, r1;
        stage_load(a, 0, h, qh, lane, r0);
        if (chunks > 1) { stage_load(a, kC, h, qh, lane, r1); }
        stage_store(a, r0, chunk[0], lane);
        __syncthreads();
#pragma unroll 1
        for (int j = 0; j < chunks; j += 2) {
            if (j + 2 < chunks) { stage_load(a, (j + 2) * kC, h, qh, lane, r0); }
            if (j + 1 < chunks) { stage_store(a, r1, chunk[1], lane); }
            __syncthreads();
            if (j + 1 == chunks) { break; }
            if (j + 3 < chunks) { stage_load(a, (j + 3) * kC, h, qh, lane, r1); }
            if (j + 2 < chunks) { stage_store(a, r0, chunk[0], lane); }
            __syncthreads();
        }
        return;
    }
    const int c = lane & 15;
    const int g = lane >> 4;
    const int r = (rblock * kSerial + wave) * 16 + c; // this lane's state row
    const int64_t srow = (static_cast<int64_t>(h) * kS + r) * kS;
    f4 S[8]; // S^T tile dt: entry e is column 16dt + 4g + e of row r
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) { S[dt] = *reinterpret_cast<const f4*>(a.state_in + srow + 16 * dt + 4 * g); }
    uint16_t vn[8]; // v of token 16tt + 4g + e, next chunk's in flight
    const int vrow = a.Hv * kS * 2;
    const int vat = 4 * g * vrow + (h * kS + r) * 2;
    const auto load_v = [&](int t0) {
        const __amdgpu_buffer_rsrc_t vb = chunk_rows(a.v, vrow, t0, a.T);
#pragma unroll
        for (int i = 0; i < 8; ++i) { vn[i] = __builtin_amdgcn_raw_buffer_load_b16(vb, vat + (16 * (i >> 2) + (i & 3)) * vrow, 0, 0); }
    };
    load_v(0);
    __syncthreads();
#pragma unroll 1
    for (int j = 0; j < chunks; ++j) {
        const Chunk& x = chunk[j & 1];
        const int t0 = j * kC;
        // ---- X = S k_t and Y = S q_t of every token: S as three exact BF16 terms
        f4 X[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        f4 Y[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        b8 hi[4], mid[4], lo[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) { v[i] = S[2 * s + (i >> 2)][i & 3]; }
            split3(v, hi[s], mid[s], lo[s]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const b8 kr = *reinterpret_cast<const b8*>(x.k + row_at(16 * tt + c, 4 * s + g));
                X[tt] = mfma_b(kr, lo[s], X[tt]);
                X[tt] = mfma_b(kr, mid[s], X[tt]);
                X[tt] = mfma_b(kr, hi[s], X[tt]);
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const b8 qr = *reinterpret_cast<const b8*>(x.q + row_at(16 * tt + c, 4 * s + g));
                Y[tt] = mfma_b(qr, lo[s], Y[tt]);
                Y[tt] = mfma_b(qr, mid[s], Y[tt]);
                Y[tt] = mfma_b(qr, hi[s], Y[tt]);
            }
        }
        // ---- right-hand side, then substitution in blocks of four tokens: the lane group that owns a
        // block solves it, hands it to the other groups, and every lane subtracts it from its later tokens
        f4 d[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const f4 bt = *reinterpret_cast<const f4*>(x.beta + 16 * tt + 4 * g);
            const f4 gk = *reinterpret_cast<const f4*>(x.gk + 16 * tt + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) { d[tt][e] = bt[e] * bf16_to_f32(vn[4 * tt + e]) - gk[e] * X[tt][e]; }
        }
        if (j + 1 < chunks) { load_v(t0 + kC); }
        f4 sum[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}; // sum_(i<t) A_ti d_i so far
        // A's rows of a block, read a block ahead: its own 4 x 4 triangle, and the lane's 8 tokens
        f4 tri[2][3], rows[2][2][4];
        const auto fetch = [&](auto bc) {
            constexpr int b = decltype(bc)::value;
#pragma unroll
            for (int e = 0; e < 3; ++e) { tri[b & 1][e] = *reinterpret_cast<const f4*>(x.A + (4 * b + 1 + e) * kMatStride + 4 * b); }
#pragma unroll
            for (int tt = b >> 2; tt < 2; ++tt) {
                if (tt == (b >> 2) && (b & 3) == 3) { continue; } // no later token in this tile
#pragma unroll
                for (int e = 0; e < 4; ++e) { rows[b & 1][tt][e] = *reinterpret_cast<const f4*>(x.A + (16 * tt + 4 * g + e) * kMatStride + 4 * b); }
            }
        };
        const auto block = [&](auto bc) {
            constexpr int b = decltype(bc)::value;
            constexpr int tb = b >> 2; // tile and lane group of tokens 4b .. 4b + 3
            constexpr int gb = b & 3;
            if constexpr (b < 7) { fetch(std::integral_constant<int, b + 1>{}); }
            const f4 r1 = tri[b & 1][0], r2 = tri[b & 1][1], r3 = tri[b & 1][2];
            float y[4];
            y[0] = d[tb][0] - sum[tb][0];
            y[1] = d[tb][1] - fmaf(r1[0], y[0], sum[tb][1]);
            y[2] = d[tb][2] - fmaf(r2[1], y[1], fmaf(r2[0], y[0], sum[tb][2]));
            y[3] = d[tb][3] - fmaf(r3[2], y[2], fmaf(r3[1], y[1], fmaf(r3[0], y[0], sum[tb][3])));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                d[tb][e] = g == gb ? y[e] : d[tb][e];
                y[e] = from_group<gb>(y[e]);
            }
#pragma unroll
            for (int tt = tb; tt < 2; ++tt) {
                if (tt == tb && gb == 3) { continue; }
                // rows at or before the block add products with A's zeros or to sums no longer used
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) { sum[tt][e] = fmaf(rows[b & 1][tt][e][q], y[q], sum[tt][e]); }
                }
            }
        };
        fetch(std::integral_constant<int, 0>{});
        block(std::integral_constant<int, 0>{});
        block(std::integral_constant<int, 1>{});
        block(std::integral_constant<int, 2>{});
        block(std::integral_constant<int, 3>{});
        block(std::integral_constant<int, 4>{});
        block(std::integral_constant<int, 5>{});
        block(std::integral_constant<int, 6>{});
        block(std::integral_constant<int, 7>{});
        // ---- S' = G_31 S + (D_31,i d_i) k_i^T, d as three exact BF16 terms
        {
            float v[8];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const f4 dk = *reinterpret_cast<const f4*>(x.dk + 16 * tt + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) { v[4 * tt + e] = d[tt][e] * dk[e]; }
            }
            b8 dh, dm, dl;
            split3(v, dh, dm, dl);
            const float gc = x.gc;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                const b8 kt = *reinterpret_cast<const b8*>(x.kt + kt_at(16 * dt + c, g));
                f4 u = {0.f, 0.f, 0.f, 0.f};
                u = mfma_b(kt, dl, u);
                u = mfma_b(kt, dm, u);
                u = mfma_b(kt, dh, u);
#pragma unroll
                for (int e = 0; e < 4; ++e) { S[dt][e] = fmaf(gc, S[dt][e], u[e]); }
            }
        }
        // ---- o = scale G_t S q_t + P d (FP32 matrix instruction; k = g of step (ii, e) is token 16ii + 4g + e)
        f4 o[2];
        bool finite = true;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const f4 gq = *reinterpret_cast<const f4*>(x.gq + 16 * tt + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[tt][e] = gq[e] * Y[tt][e];
                finite &= __builtin_isfinite(d[tt][e]);
            }
        }
        if (__all(finite)) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
                for (int ii = 0; ii <= tt; ++ii) {
                    const f4 p = *reinterpret_cast<const f4*>(x.P + (16 * tt + c) * kMatStride + 16 * ii + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) { o[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[e], d[ii][e], o[tt], 0, 0, 0); }
                }
            }
        } else {
            // a product with P's zeros would carry an infinite or NaN d back to earlier tokens
#pragma unroll
            for (int i = 0; i < 8; ++i) { spill[wave][16 * (i >> 2) + 4 * g + (i & 3)][c] = d[i >> 2][i & 3]; }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int t = 16 * (i >> 2) + 4 * g + (i & 3);
                float v = o[i >> 2][i & 3];
                for (int k = 0; k <= t; ++k) { v = fmaf(x.P[t * kMatStride + k], spill[wave][k][c], v); }
                o[i >> 2][i & 3] = v;
            }
        }
        const __amdgpu_buffer_rsrc_t ob = chunk_rows(a.out, vrow, t0, a.T); // stores past the prompt are dropped
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16_bits(o[i >> 2][i & 3]), ob, vat + (16 * (i >> 2) + (i & 3)) * vrow, 0, 0);
        }
        __syncthreads(); // this chunk's buffer is free, the next one's is filled
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) { *reinterpret_cast<f4*>(a.state_out + srow + 16 * dt + 4 * g) = S[dt]; }
}

} // namespace

bool gdn_chunk_serves(const GdnArgs& a, int32_t S) {
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    return S == kS && a.initial_slot == nullptr && a.T > 16 && aligned(a.q) && aligned(a.k) && aligned(a.state_in) &&
           aligned(a.state_out);
}

void launch_gdn_chunk(const GdnArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL(gdn_chunk_kernel, dim3(8 * ((a.Hv + 7) / 8) * kRowBlocks), dim3(kChunkThreads), 0, stream, a);
    check_launch("gdn_chunk_kernel");
}

} // namespace nmi
