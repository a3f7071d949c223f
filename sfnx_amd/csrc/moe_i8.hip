// The prompt path's BigJobs in the int8 (q8_1) arithmetic, FNX_PF_MOE_Q8 (src/moe.cuh:360-443): out[job.out[j]][row] =
// row of the expert . activation row job.y[j], bit for bit the sums of the decode's dot lanes (mv.hpp), with the integer
// dots on v_mfma_i32_32x32x32_i8.
//
// A dot there is, per 32-value block, an exact integer sum, scaled into fp32 and added in a fixed order: lane l of a row's
// LPR lanes takes the steps l + LPR i in order (a step: two blocks of a K-quant's 64-value group, or one block), then the
// lanes' sums meet in a xor butterfly.  An i8 MFMA of 32 k-slots is exactly one block's integer sum for 32 rows x 32
// tokens; the fp32 part follows on the accumulators in the same order: steps l, l + LPR, ... of one l in turn (a strip),
// the strips in bit-reversed order of l, so the butterfly is the pairwise merge of consecutive strips (at most 4 partial
// sums a value are live).  Lane (nn, h) of a wavefront holds weight row nn of its 32 and 16 tokens (8 (q / 4) + 4 h + q %
// 4); groups of 8 tokens past the job's rows are left out.
//
// What bounds it is that fp32 part: 14 VALU instructions a (row, token, 64 values) for the K-quants, against 2 MFMAs a
// step and ~40 to unpack a step's weights for 32 tokens.  The K-quants' first product sc (float) dot costs one of them:
// the MFMA starts from the bits of M = 1.5 2^23, so its result read as a float is M + dot, and fmaf(sc, M + dot, -sc M) is
// sc dot, exactly (|dot| < 2^22, every product exact).
//
// Measured at 1000 tokens, 2048 columns, 512 experts x FF 512, top-10 + shared, Q4_K: gate|up 655 -> 312 us, down 620 ->
// 239 us against one v_dot4 lane group a row (whose 16 dots a group and LDS reads this replaces); Q8_0 670 -> 390 and
// 2,360 -> 228 us.  VALU issue takes 95% of the SIMDs' cycles in
// gate|up and 80% in down (counters, 2048 tokens); down adds h, made once a block.
#include <algorithm>

#include "decode.hpp"

namespace sfnx {
namespace {

typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int16v __attribute__((ext_vector_type(16)));

constexpr int I8_THREADS = 256, I8_WAVES = I8_THREADS / WAVE, I8_ROWS = 32 * I8_WAVES;
// Jobs of at most i8_few rows take the decode's dot lanes (mv.hpp), a weight row's pieces all requested at once: the
// matrix-core walk unpacks a step's weights for 32 tokens whatever the job holds.  Measured, the 32-value types, whose 16 strips
// make that walk longest (Q8_0, 2048 columns, 512 experts, gate|up / down): 100 tokens 215 / 115 us with jobs of 1 row on the
// lanes, 178 / 127 up to 4, 166 / 146 up to 8.  K-quants, gate|up from 2048 columns: jobs of 1 and 2 rows, 40 tokens, 512 experts,
// Q4_K 84 -> 65 us, Q5_K 100 -> 82; 64 tokens, 2560 columns, 178 -> 157 and 246 -> 209; up to 4 rows lost 5% again at 100 tokens,
// and at 1024 columns and below the walk is as short (17 tokens 15.4 -> 16.6).
constexpr int i8_few(uint32_t type, int nr, bool down) { return is_kquant(type) ? (!down && nr >= 4 ? 2 : 0) : down ? 4 : 8; }
constexpr float I8_M = 12582912.0f;           // 1.5 2^23
constexpr int I8_MBITS = 0x4B400000;

template <int TYPE> constexpr int i8_lpr() { return is_kquant(TYPE) ? 8 : 16; }   // strips
template <int TYPE> constexpr int i8_sub() { return is_kquant(TYPE) ? 2 : 1; }    // 32-value blocks a step

// ------------------------------------------------------------------------------------------------ weights
// one lane's raw weights of a step: its lane-half's 16 bytes and the row's scales
template <int TYPE> struct I8W {
    uint4 q;
    uint4 hdr;   // K-quants: the super-block header; Q8_0, Q4_0: x = f16 d; Q5_1: x = (f16 d, f16 m), y = qh word
    uint4 qh;    // Q5_K
};
// Where a wavefront's 32 rows lie: the row tile's (uniform) address in each plane, and the lane's byte offsets in them
template <int TYPE> struct I8At {
    const uint8_t *q, *s, *x;   // quants; headers or scales; fifth bits
    uint32_t oq, os, ox, tq, ts, tx;   // lane offsets; bytes from one 32-row tile to the next
    __device__ __forceinline__ I8At(const uint8_t* mat, int R, int C, int row0, int nn, int h) {
        const int tile = min(row0, R - 1) / 32, r = min(nn, R - 1 - 32 * tile);   // rows past R repeat the last
        if constexpr (is_kquant(TYPE)) {
            const KqPlanes P = kq_planes<TYPE == SFNX_Q5_K>(mat, R, C);
            q = P.nib, s = P.hdr, x = P.qh;
            tq = 32 * (C / 2), ts = 32 * (C / 16), tx = 32 * (C / 8);
            oq = 16 * r + 8 * PIECE_STRIDE * h, os = 16 * r, ox = 16 * r + PIECE_STRIDE * h;
        } else if constexpr (TYPE == SFNX_Q8_0) {
            const Q80Planes P = q80_planes(mat, R, C);
            q = P.q, s = P.d, x = nullptr;
            tq = 32 * C, ts = 32 * (C / 16), tx = 0;
            oq = tiled16<Q80_RT>(r, C, 16 * h), os = tiled16<Q80_RT>(r, C / 16, 0), ox = 0;
        } else {
            const NbPlanes P = nb_planes<TYPE>(mat, R, C);
            const int rs = TYPE == SFNX_Q4_0 ? C / 16 : C / 8;
            q = P.q, s = P.s, x = P.qh;
            tq = 32 * (C / 2), ts = 32 * rs, tx = 32 * (C / 8);
            oq = tiled16<Q80_RT>(r, C / 2, 0), os = tiled16<Q80_RT>(r, rs, 0), ox = tiled16<Q80_RT>(r, C / 8, 0);
        }
        q += (size_t) tile * tq, s += (size_t) tile * ts, x += (size_t) tile * tx;
    }
    // step i of strip l, the row tiles `tiles` on
    __device__ __forceinline__ void load(I8W<TYPE>& w, int l, int i, int tiles) const {
        const uint8_t *pq = q + (size_t) tiles * tq, *ps = s + (size_t) tiles * ts;
        [[maybe_unused]] const uint8_t* px = x + (size_t) tiles * tx;
        if constexpr (is_kquant(TYPE)) {
            w.q = *reinterpret_cast<const uint4*>(pq + PIECE_STRIDE * (16 * i + l) + oq);
            w.hdr = *reinterpret_cast<const uint4*>(ps + PIECE_STRIDE * (2 * i + (l >> 2)) + os);
            if constexpr (TYPE == SFNX_Q5_K) w.qh = *reinterpret_cast<const uint4*>(px + PIECE_STRIDE * 2 * (2 * i + (l >> 2)) + ox);
        } else {
            constexpr int PS = Q80_RT * 16;   // bytes from one piece of a row to the next
            w.q = *reinterpret_cast<const uint4*>(pq + PS * ((TYPE == SFNX_Q8_0 ? 32 : 16) * i + l) + oq);
            if constexpr (TYPE == SFNX_Q5_1) {
                w.hdr.x = *reinterpret_cast<const uint32_t*>(ps + PS * (4 * i + (l >> 2)) + 4 * (l & 3) + os);
                w.hdr.y = *reinterpret_cast<const uint32_t*>(px + PS * (4 * i + (l >> 2)) + 4 * (l & 3) + ox);
            } else {
                w.hdr.x = *reinterpret_cast<const uint16_t*>(ps + PS * (2 * i + (l >> 3)) + 2 * (l & 7) + os);
            }
        }
    }
};
// the int8 operands of a step's blocks: values 16 h .. 16 h + 15 of each
template <int TYPE> __device__ __forceinline__ void i8_unpack(const I8W<TYPE>& w, int l, int h, int4v (&b)[2]) {
    const uint32_t q[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
    if constexpr (is_kquant(TYPE)) {
        const uint32_t x[4] = {w.qh.x, w.qh.y, w.qh.z, w.qh.w};
        const int j = 2 * (l & 3);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t lo = q[k] & 0x0F0F0F0Fu, hi = (q[k] >> 4) & 0x0F0F0F0Fu;
            if constexpr (TYPE == SFNX_Q5_K) {
                lo |= ((x[k] >> j) & 0x01010101u) << 4;
                hi |= ((x[k] >> (j + 1)) & 0x01010101u) << 4;
            }
            b[0][k] = (int) lo;
            b[1][k] = (int) hi;
        }
    } else if constexpr (TYPE == SFNX_Q8_0) {
        // (copies made here: the slot's registers take the next request while these are multiplied)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int v;
            asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "v"(q[k]));
            b[0][k] = v;
        }
    } else {
        // a block's 16 bytes: values 0-15 in the low nibbles, 16-31 in the high
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t v = (q[k] >> (4 * h)) & 0x0F0F0F0Fu;
            if constexpr (TYPE == SFNX_Q5_1) v |= spread4(w.hdr.y >> (16 * h + 4 * k));
            b[0][k] = (int) v;
        }
    }
}

// ------------------------------------------------------------------------------------------------ activations
// A strip's activations in LDS for TOK tokens and NB = nr SUB blocks each: int8 values [TOK][32 NB + 16], block scales
// [NB][TOK] and block sums [NB][TOK] as floats
template <int TOK, int NB> struct I8Acts {
    static constexpr int PITCH = 32 * NB + 16, BYTES = TOK * PITCH + 2 * NB * TOK * 4;
    unsigned char* base;
    __device__ __forceinline__ int8_t* q(int t, int b) const { return reinterpret_cast<int8_t*>(base + t * PITCH + 32 * b); }
    __device__ __forceinline__ float* d(int b) const { return reinterpret_cast<float*>(base + TOK * PITCH) + b * TOK; }
    __device__ __forceinline__ float* s(int b) const { return reinterpret_cast<float*>(base + TOK * PITCH) + (NB + b) * TOK; }
};
// tokens a block: 32; down keeps every strip of its tokens in LDS, so 16 where 32 would pass 64 KB
template <int TYPE, int NR, bool DOWN> constexpr int i8_tok() {
    return DOWN && i8_lpr<TYPE>() * I8Acts<32, NR * i8_sub<TYPE>()>::BYTES > 64 * 1024 ? 16 : 32;
}

// the strip taken k-th: lane l of the butterfly, in the order whose pairwise merges are its tree
template <int LPR> __device__ __forceinline__ int strip_of(int k) { return (int) (__brev((unsigned) k) >> (LPR == 8 ? 29 : 28)); }

// q8_1 blocks (36 bytes) of a strip through registers: a thread an item (token, block of the strip), NI items a thread;
// items past the job's tokens repeat the last one
template <int TYPE, int NR> struct I8Stage {
    static constexpr int SUB = i8_sub<TYPE>(), LPR = i8_lpr<TYPE>(), NB = NR * SUB, NI = (32 * NB + I8_THREADS - 1) / I8_THREADS;
    const uint8_t* src[NI];   // the item's block of strip 0
    uint32_t w[NI][9];
    __device__ __forceinline__ void init(const uint8_t* xq, const int* ys, int n) {
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            const int e = threadIdx.x + it * I8_THREADS, t = min(e / NB, n - 1), j = e % NB;
            src[it] = xq + ((size_t) ys[t] * (16 * NR) + SUB * LPR * (j / SUB) + j % SUB) * Q81_BYTES;
        }
    }
    __device__ __forceinline__ void load(int l) {
#pragma unroll
        for (int it = 0; it < NI; ++it)
#pragma unroll
            for (int k = 0; k < 9; ++k) w[it][k] = reinterpret_cast<const uint32_t*>(src[it] + SUB * l * Q81_BYTES)[k];
    }
    template <typename ACTS> __device__ __forceinline__ void store(const ACTS& a, int n) const {
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            const int e = threadIdx.x + it * I8_THREADS, t = e / NB, j = e % NB;
            if (t < n) {
                int s = 0;
#pragma unroll
                for (int k = 0; k < 8; ++k) s = dot4((int) w[it][1 + k], 0x01010101, s);
                uint4* dst = reinterpret_cast<uint4*>(a.q(t, j));
                dst[0] = make_uint4(w[it][1], w[it][2], w[it][3], w[it][4]);
                dst[1] = make_uint4(w[it][5], w[it][6], w[it][7], w[it][8]);
                a.d(j)[t] = h2f((uint16_t) w[it][0]);
                a.s(j)[t] = (float) s;
            }
        }
    }
};
// h = silu(gate) up of gu rows as q8_1 (stage_swiglu's values), every strip at once: 8 threads a block, 4 values each
template <int TYPE, typename ACTS>
__device__ __forceinline__ void stage_h(unsigned char* lds, const float* gu, int C, const int* ys, int n) {
    constexpr int SUB = i8_sub<TYPE>(), LPR = i8_lpr<TYPE>();
    const int nb = C / 32, l8 = threadIdx.x % 8;
    for (int it = threadIdx.x / 8; it < n * nb; it += I8_THREADS / 8) {
        const int t = it / nb, kb = it % nb;
        const float* g = gu + (size_t) ys[t] * 2 * C + 32 * kb + 4 * l8;
        const float4 gv = *reinterpret_cast<const float4*>(g), uv = *reinterpret_cast<const float4*>(g + C);
        const float x[4] = {silu_f(gv.x) * uv.x, silu_f(gv.y) * uv.y, silu_f(gv.z) * uv.z, silu_f(gv.w) * uv.w};
        const float amax = group_max<8>(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))));
        const float d = amax / 127.0f;
        int s = 0;
        uint32_t pk = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int q = amax == 0.0f ? 0 : (int) roundf(x[k] / d);
            s += q;
            pk |= (uint32_t) (uint8_t) (int8_t) q << (8 * k);
        }
        s = group_isum<8>(s);
        const int st = kb / SUB, l = st % LPR, j = st / LPR * SUB + kb % SUB;
        const ACTS a{lds + l * ACTS::BYTES};
        *reinterpret_cast<uint32_t*>(a.q(t, j) + 4 * l8) = pk;
        if (l8 == 0) {
            a.d(j)[t] = h2f(f2h(d));
            a.s(j)[t] = (float) s;
        }
    }
}

// ------------------------------------------------------------------------------------------------ the sums
// the row's scales of a step: K-quants d, dmin, the two sub-blocks' sc and m; else d (and Q5_1's m)
template <int TYPE> struct I8Scale {
    float d, dmin, sc0, m0, sc1, m1;
    __device__ __forceinline__ I8Scale(const I8W<TYPE>& w, int l) {
        d = h2f((uint16_t) (w.hdr.x & 0xffff));
        if constexpr (is_kquant(TYPE) || TYPE == SFNX_Q5_1) dmin = h2f((uint16_t) (w.hdr.x >> 16));
        if constexpr (is_kquant(TYPE)) {
            // q4k_scale_min of sub-blocks 2 (l & 3) and the next, as byte pairs and without a branch on l (the compiler
            // would thread it through the unrolled steps)
            const int sh = 16 * (l & 1);
            const uint32_t y = w.hdr.y >> sh, z = w.hdr.z >> sh, x = w.hdr.w >> sh;
            const uint32_t lo = l & 2 ? 0u : 0x3F3Fu, hi = l & 2 ? 0x0F0Fu : 0u, top = l & 2 ? 0x3030u : 0u;
            const uint32_t sc = (y & lo) | (x & hi) | ((y >> 2) & top), m = (z & lo) | ((x >> 4) & hi) | ((z >> 2) & top);
            sc0 = (float) (sc & 0xFF), sc1 = (float) ((sc >> 8) & 0xFF);
            m0 = (float) (m & 0xFF), m1 = (float) ((m >> 8) & 0xFF);
        }
    }
    __device__ __forceinline__ void pin() {
        asm volatile("" : "+v"(d));
        if constexpr (is_kquant(TYPE) || TYPE == SFNX_Q5_1) asm volatile("" : "+v"(dmin));
        if constexpr (is_kquant(TYPE)) asm volatile("" : "+v"(sc0), "+v"(m0), "+v"(sc1), "+v"(m1));
    }
};
// a uniform value the compiler cannot reason about, so that it does not make a copy of the loop for each of its ranges
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+s"(v));
    return v;
}
// the token operands of a step's blocks: row m's values 16 h .. 16 h + 15
template <int TYPE, typename ACTS> __device__ __forceinline__ void i8_tokens(int4v (&t)[2], const ACTS& a, int i, int m, int h) {
    constexpr int SUB = i8_sub<TYPE>();
#pragma unroll
    for (int k = 0; k < SUB; ++k) t[k] = *reinterpret_cast<const int4v*>(a.q(m, SUB * i + k) + 16 * h);
}
// block scales and sums of 4 tokens
template <int TYPE> struct I8Tok4 {
    static constexpr int SUB = i8_sub<TYPE>();
    float d[SUB][4], s[SUB][4];
    template <typename ACTS> __device__ __forceinline__ void load(const ACTS& a, int blk, int t) {
#pragma unroll
        for (int k = 0; k < SUB; ++k) {
            const float4 v = *reinterpret_cast<const float4*>(a.d(blk + k) + t);
            d[k][0] = v.x, d[k][1] = v.y, d[k][2] = v.z, d[k][3] = v.w;
            if constexpr (SUB == 2 || TYPE == SFNX_Q5_1) {
                const float4 u = *reinterpret_cast<const float4*>(a.s(blk + k) + t);
                s[k][0] = u.x, s[k][1] = u.y, s[k][2] = u.z, s[k][3] = u.w;
            }
        }
    }
};
// a step's terms added to the strip's sums cur (tokens past n left out in eights; reading the next eight's scales while one
// is summed takes registers and was 4% slower)
template <int TYPE, int TOK, typename ACTS>
__device__ __forceinline__ void i8_step(const I8Scale<TYPE>& w, const int4v (&a0)[2], const int4v (&b)[2], const ACTS& a, int i, int h, int n,
                                        const int16v& bias, float (&cur)[16]) {
    constexpr int SUB = i8_sub<TYPE>();
    const int blk = SUB * i;
    I8Tok4<TYPE> t;
    t.load(a, blk, 4 * h);   // the first eight's with the products
    int16v lo, hi;
    if constexpr (SUB == 2) {
        lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[0], b[0], bias, 0, 0, 0);
        hi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[1], b[1], bias, 0, 0, 0);
    } else {
        lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[0], b[0], int16v{}, 0, 0, 0);
        if constexpr (TYPE == SFNX_Q4_0) {   // sum (q - 8) a: the -8 a as another product into the same integers
            constexpr int M8 = (int) 0xF8F8F8F8u;
            lo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0[0], int4v{M8, M8, M8, M8}, lo, 0, 0, 0);
        }
    }
    const float k0 = -(w.sc0 * I8_M), k1 = -(w.sc1 * I8_M);
#pragma unroll
    for (int g = 0; g < TOK / 8; ++g) {
        if (8 * g >= opaque(n)) continue;
        if (g) t.load(a, blk, 8 * g + 4 * h);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int q = 4 * g + c;
            if constexpr (SUB == 2) {
                const float pl = fmaf(w.sc0, __int_as_float(lo[q]), k0), ph = fmaf(w.sc1, __int_as_float(hi[q]), k1);
                cur[q] += w.d * (t.d[0][c] * pl + t.d[1][c] * ph) -
                          w.dmin * (t.d[0][c] * (w.m0 * t.s[0][c]) + t.d[1][c] * (w.m1 * t.s[1][c]));
            } else if constexpr (TYPE == SFNX_Q5_1) {
                cur[q] += (w.d * t.d[0][c]) * (float) lo[q] + (w.dmin * t.d[0][c]) * t.s[0][c];
            } else {
                cur[q] += (w.d * t.d[0][c]) * (float) lo[q];
            }
        }
    }
}

// Workgroup b runs on XCD b % 8: a job's row slices and token tiles go to one XCD together, so the second token tile of
// a job finds the weight rows in that XCD's L2 or behind it.  The row slices vary fastest: an XCD hands consecutive
// workgroups to its 4 shader engines in turn, and with the token tiles fastest the empty second tiles of the jobs of at
// most 32 rows all fell to the same two (half the compute units idle: 460 us against 300 for gate|up of 1000 tokens)
constexpr int I8_XG = 4;
__device__ __forceinline__ void i8_unit(int b, int nu, int& u, int& job) {
    const int x = b % XCDS, k = b / XCDS, m = k / nu;
    u = k % nu;
    job = I8_XG * (XCDS * (m / I8_XG) + x) + m % I8_XG;
}
inline int i8_grid(int nu, int njobs_cap) { return nu * ((njobs_cap + XCDS * I8_XG - 1) / (XCDS * I8_XG)) * XCDS * I8_XG; }

// such a job's rows row0 .. row0 + nrows - 1 of the expert, a tile of I8_THREADS / LPR rows at a time
template <int TYPE, int NR, bool DOWN>
__device__ __forceinline__ void few_rows(const uint8_t* mat, int R, int row0, int nrows, int n, const int* ys, const int* outs, unsigned char* lds,
                                         const void* __restrict__ in, float* __restrict__ out) {
    constexpr int LPR = lpr_of<TYPE>(), RPB = I8_THREADS / LPR, C = 512 * NR, FEW = i8_few(TYPE, NR, DOWN);
    const int ln = threadIdx.x % LPR, g = threadIdx.x / LPR, end = min(row0 + nrows, R);
    const Acts a = acts_in(lds, FEW, C);
    if constexpr (DOWN) stage_swiglu(a, (const float*) in, ys, n);
    else stage_q8_1(a, (const uint8_t*) in, ys, n);
    __syncthreads();
    // two tiles' rows in registers, one requested while the other is dotted (4096 columns, Q5_K from 2560: one, two would spill)
    constexpr int ND = NR < (TYPE == SFNX_Q5_K ? 5 : 8) ? 2 : 1;
    typename RowOf<TYPE, NR>::R w[ND];
    if constexpr (ND == 2) RowOf<TYPE, NR>::issue(w[0], mat, R, min(row0 + g, R - 1), C, ln);
    for (int r0 = row0; r0 < end; r0 += ND * RPB)
#pragma unroll
        for (int p = 0; p < ND; ++p) {
            const int row = r0 + p * RPB + g;
            RowOf<TYPE, NR>::issue(w[ND - 1 - p], mat, R, min(ND == 2 ? row + RPB : row, R - 1), C, ln);
            w[p].prepare(ln);
#pragma unroll
            for (int j = 0; j < FEW; ++j)
                if (j < n) {
                    if constexpr (is_kquant(TYPE)) w[p].pin();
                    const float v = group_sum<LPR>(w[p].dot(a, j, ln));
                    if (row < end && ln == 0) out[(size_t) outs[j] * R + row] = v;
                }
        }
}

// A block: TOK tokens of a job x G tiles of 128 rows, 4 wavefronts of 32 rows each.  Gate|up (G = 1): each strip's
// activations come through registers into one of two LDS buffers while the strip before it is summed.  Down: h of the
// block's tokens is made once, every strip in LDS, and serves the G row tiles (h costs ~45 instructions a value).
// Weights stream through a ring of RING register slots, step e + RING requested when step e is unpacked; GS strips of NR
// steps are unrolled together, so that every slot's requests are counted exactly by the compiler's waits.
template <int TYPE, int NR, bool DOWN>
__global__ void __launch_bounds__(I8_THREADS, DOWN && !is_kquant(TYPE) && NR <= 2 ? 3 : 2) k_moe_i8(const uint8_t* __restrict__ A, size_t sa, int R, int G,
                                                         const sfnx_bigjob* __restrict__ jobs, const int* __restrict__ njobs,
                                                         const void* __restrict__ in, float* __restrict__ out) {
    constexpr int LPR = i8_lpr<TYPE>(), SUB = i8_sub<TYPE>(), C = 512 * NR, NB = NR * SUB;
    constexpr int TOK = i8_tok<TYPE, NR, DOWN>();
    using ACTS = I8Acts<TOK, NB>;
    constexpr int GS = NR >= 4 ? 1 : 4 / NR, RING = NR == 5 ? 5 : 4, GE = GS * NR;
    static_assert(GE % RING == 0 && LPR % GS == 0, "a group's steps fill the ring evenly");
    constexpr int ntt = SFNX_PF_JOB / TOK;
    const int nsl = (R + I8_ROWS * G - 1) / (I8_ROWS * G), nj = *njobs;
    int u, ji;
    i8_unit(blockIdx.x, nsl * ntt, u, ji);
    if (ji >= nj) return;
    ji = nj - 1 - ji;   // the shared expert's full jobs, the longest, first
    const int t0 = TOK * (u / nsl), row_base = I8_ROWS * G * (u % nsl);
    const int nall = jobs[ji].n;
    // Q4_K's few rows: each token tile's block takes its share of the weight rows
    constexpr bool SHARE = is_kquant(TYPE) && i8_few(TYPE, NR, DOWN) > 0;
    const bool few = i8_few(TYPE, NR, DOWN) > 0 && nall <= i8_few(TYPE, NR, DOWN);
    const int n = SHARE && few ? nall : min(TOK, nall - t0);
    if (n <= 0) return;
    __shared__ int ys[32], outs[32];
    extern __shared__ __align__(16) unsigned char lds[];
    if (threadIdx.x < 32 && (int) threadIdx.x < n) {
        const int j0 = SHARE && few ? 0 : t0;
        ys[threadIdx.x] = jobs[ji].y[j0 + threadIdx.x];
        outs[threadIdx.x] = jobs[ji].out[j0 + threadIdx.x];
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, nn = lane % 32, h = lane / 32;
    const uint8_t* mat = expert_at(A, sa, jobs[ji].w);
    if constexpr (i8_few(TYPE, NR, DOWN) > 0)
        if (few) {
            __syncthreads();
            constexpr int share = SHARE ? I8_ROWS / ntt : 0;   // (G is 1 where they share)
            if constexpr (SHARE) few_rows<TYPE, NR, DOWN>(mat, R, row_base + share * (t0 / TOK), share, n, ys, outs, lds, in, out);
            else few_rows<TYPE, NR, DOWN>(mat, R, row_base, I8_ROWS * G, n, ys, outs, lds, in, out);
            return;
        }
    const int wrow = row_base + 32 * wave;   // the wavefront's first row
    const I8At<TYPE> at(mat, R, C, wrow, nn, h);
    // row tiles of the wavefront from its first that hold a row (the last one again past them)
    const int last = wrow < R ? (R - 1 - wrow) / I8_ROWS : 0;
    int tile = 0;
    // step e of the strip group at strip k0 (strips past the last: the next row tile's)
    I8W<TYPE> w[RING];
    auto request = [&](I8W<TYPE>& v, int k0, int e) {
        const int k = k0 + e / NR;
        at.load(v, strip_of<LPR>(k % LPR), e % NR, 4 * min(tile + k / LPR, last));
    };
#pragma unroll
    for (int e = 0; e < RING; ++e) {
        request(w[e], 0, e);
        __builtin_amdgcn_sched_barrier(0);   // (in the walk's order, so that its waits count exactly from the first step)
    }
    __syncthreads();
    I8Stage<TYPE, NR> st;
    auto buffer = [&](int b) { return ACTS{lds + b * ACTS::BYTES}; };
    if constexpr (DOWN) {
        stage_h<TYPE, ACTS>(lds, (const float*) in, C, ys, n);
    } else {
        st.init((const uint8_t*) in, ys, n);
        st.load(strip_of<LPR>(0));
        st.store(buffer(0), n);
    }
    lds_barrier();
    int16v bias;
#pragma unroll
    for (int q = 0; q < 16; ++q) bias[q] = I8_MBITS;
    if constexpr (SUB == 2) asm volatile("" : "+v"(bias));   // held in registers, not made again at each step
    float cur[16], p0[16], p1[16], p2[16], p3[16];
    const int m = min(nn, TOK - 1);
    int4v tok[2];   // the next step's token operand
    if constexpr (DOWN) i8_tokens<TYPE>(tok, buffer(strip_of<LPR>(0)), 0, m, h);
    for (; tile < G; ++tile) {
        for (int k0 = 0; k0 < LPR; k0 += GS) {
#pragma unroll
            for (int ks = 0; ks < GS; ++ks) {
                const int k = k0 + ks, l = strip_of<LPR>(k);
                // the next strip's activations, into the other buffer at this strip's end
                if constexpr (!DOWN) {
                    st.load(strip_of<LPR>(min(k + 1, LPR - 1)));
                    i8_tokens<TYPE>(tok, buffer(k & 1), 0, m, h);
                }
#pragma unroll
                for (int q = 0; q < 16; ++q) cur[q] = 0.f;
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    const int e = ks * NR + i;
                    I8W<TYPE>& v = w[e % RING];
                    int4v b[2];
                    i8_unpack<TYPE>(v, l, h, b);
                    I8Scale<TYPE> sc(v, l);
                    // everything of the slot decoded before its refill is requested: a value still to be decoded then
                    // keeps its register, the request gets another, and the copy back waits for the request
                    sc.pin();
                    asm volatile("" : "+v"(b[0]) : : "memory");
                    if constexpr (SUB == 2) asm volatile("" : "+v"(b[1]) : : "memory");
                    request(v, k0, e + RING);
                    const int4v t[2] = {tok[0], tok[1]};
                    if (i + 1 < NR) i8_tokens<TYPE>(tok, buffer(DOWN ? l : k & 1), i + 1, m, h);
                    else if constexpr (DOWN) i8_tokens<TYPE>(tok, buffer(strip_of<LPR>((k + 1) % LPR)), 0, m, h);
                    i8_step<TYPE, TOK>(sc, t, b, buffer(DOWN ? l : k & 1), i, h, n, bias, cur);
                    __builtin_amdgcn_sched_barrier(0);   // (steps interleaved by the scheduler spill)
                }
                // the strip's sums into the butterfly's tree
                auto keep = [&](float (&p)[16]) {
#pragma unroll
                    for (int q = 0; q < 16; ++q) p[q] = cur[q];
                };
                auto merge = [&](const float (&p)[16]) {
#pragma unroll
                    for (int q = 0; q < 16; ++q) cur[q] = p[q] + cur[q];
                };
                if (!(k & 1)) {
                    keep(p0);
                } else {
                    merge(p0);
                    if (!(k & 2)) {
                        keep(p1);
                    } else {
                        merge(p1);
                        if (!(k & 4)) {
                            keep(p2);
                        } else {
                            merge(p2);
                            if constexpr (LPR == 16) {
                                if (!(k & 8)) keep(p3);
                                else merge(p3);
                            }
                        }
                    }
                }
                // the other buffer, which every wavefront left at the last barrier
                if constexpr (!DOWN)
                    if (k + 1 < LPR) {
                        st.store(buffer((k + 1) & 1), n);
                        lds_barrier();
                    }
            }
        }
        const int row = wrow + I8_ROWS * tile + nn;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int t = 8 * (q / 4) + 4 * h + q % 4;
            if (t < n && row < R) out[(size_t) outs[t] * R + row] = cur[q];
        }
    }
}

template <bool DOWN>
void moe_i8(uint32_t type, const void* A, size_t sa, int n_in, int n_out, const sfnx_bigjob* jobs, const int* njobs,
            int njobs_cap, const void* in, float* out, void* st) {
    require(expert_type_ok(type), TYPE_MSG);
    require(n_in > 0 && n_in % 512 == 0, "expert input width must be a multiple of 512");
    require(n_out > 0, "expert rows must be positive");
    require(stride_ok(sa, row_bytes(type, n_in) * (size_t) n_out), "expert stride smaller than a matrix");
    require(njobs_cap >= 0 && njobs_cap <= 65535, "njobs_max out of range");
    if (njobs_cap == 0) return;
    const int nr = n_in / 512;
    require(nr == 1 || nr == 2 || nr == 4 || nr == 5 || nr == 8, "input width must be 512, 1024, 2048, 2560 or 4096");
    // down's row tiles a block: 4 share a block's h, fewer where that leaves under 4 blocks a compute unit (17 tokens, 128
    // experts: 65 us at 4 tiles, 32 at 1; at 1000 tokens, 512 experts 4 is the faster)
    const int tiles = (n_out + I8_ROWS - 1) / I8_ROWS;
    int G = DOWN ? std::min(tiles, 4) : 1;
    while (G > 1 && (long) njobs_cap * ((tiles + G - 1) / G) < 1024) G /= 2;
    auto go = [&](auto kern, int tok, int strip_bytes, int lpr) {
        const size_t lds = std::max((size_t) (DOWN ? lpr : 2) * strip_bytes, acts_bytes(i8_few(type, nr, DOWN), n_in));
        if (lds > 64 * 1024) check(hipFuncSetAttribute((const void*) kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds), "hipFuncSetAttribute");
        kern<<<dim3(i8_grid((tiles + G - 1) / G * (SFNX_PF_JOB / tok), njobs_cap)), I8_THREADS, lds, stream_of(st)>>>(
            (const uint8_t*) A, sa, n_out, G, jobs, njobs, in, out);
    };
#define SFNX_I8K(TY, NRV) go(k_moe_i8<TY, NRV, DOWN>, i8_tok<TY, NRV, DOWN>(), I8Acts<i8_tok<TY, NRV, DOWN>(), NRV * i8_sub<TY>()>::BYTES, i8_lpr<TY>())
#define SFNX_I8(TY)                                \
    switch (nr) {                                  \
        case 1: SFNX_I8K(TY, 1); break;            \
        case 2: SFNX_I8K(TY, 2); break;            \
        case 4: SFNX_I8K(TY, 4); break;            \
        case 5: SFNX_I8K(TY, 5); break;            \
        default: SFNX_I8K(TY, 8); break;           \
    }
    if (type == SFNX_Q4_K) { SFNX_I8(SFNX_Q4_K) }
    else if (type == SFNX_Q5_K) { SFNX_I8(SFNX_Q5_K) }
    else if (type == SFNX_Q4_0) { SFNX_I8(SFNX_Q4_0) }
    else if (type == SFNX_Q5_1) { SFNX_I8(SFNX_Q5_1) }
    else { SFNX_I8(SFNX_Q8_0) }
#undef SFNX_I8
#undef SFNX_I8K
}

}  // namespace
}  // namespace sfnx

using namespace sfnx;

extern "C" int sfnx_moe_gate_up_big(const void* A, size_t sa, uint32_t type, int n_in, int n_out, const sfnx_bigjob* jobs,
                                    const int* njobs, int njobs_cap, const void* xq, float* gu, void* st) {
    return guarded("sfnx_moe_gate_up_big", [&] { moe_i8<false>(type, A, sa, n_in, n_out, jobs, njobs, njobs_cap, xq, gu, st); });
}

extern "C" int sfnx_moe_down_big(const void* A, size_t sa, uint32_t type, int n_in, int n_out, const sfnx_bigjob* jobs,
                                 const int* njobs, int njobs_cap, const float* gu, float* part, void* st) {
    return guarded("sfnx_moe_down_big", [&] { moe_i8<true>(type, A, sa, n_in, n_out, jobs, njobs, njobs_cap, gu, part, st); });
}
