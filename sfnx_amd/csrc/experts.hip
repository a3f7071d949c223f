// The routed experts as grouped matrix x few-vectors products on int8 dot instructions (v_dot4_i32_i8): gate|up of
// the q8_1 activations, and down of h = silu(gate) * up quantized to q8_1 in LDS.  One launch covers every job of a
// layer: blockIdx.y is the job, blockIdx.x a tile of the expert's rows.  A job's activations are staged in LDS once;
// each lane keeps its share of a weight row in registers across the job's rows.  (The prompt path's BigJobs: moe_i8.hip.)
//
// Arithmetic per (row, activation row), identical to the CPU oracle's:
//   Q4_K: 8 lanes a row, lane l8 the 64-value groups l8 + 8 i in order (src/moe_q4k.cuh:30-86), each group
//         d (d8l (sc0 dl) + d8h (sc1 dh)) - dmin (d8l (m0 sl) + d8h (m1 sh)), then xor 4, 2, 1 (src/moe.cuh:224-235).
//   Q5_K: as Q4_K on the 5-bit values.
//   Q4_0 / Q5_1: the Q8_0 lanes; per block (d_w d_a) sum (q - 8) a, or (d_w d_a) sum q a + (m_w d_a) sum a.
//   Q8_0: 16 lanes a row, lane l16 the 32-blocks l16 + 16 i in order, each (d_w d_a) sum(q_w q_a), then xor 8 .. 1.
#include "decode.hpp"

namespace sfnx {
namespace {

constexpr int MV_THREADS = 256;

// ------------------------------------------------------------------------------------------------ the kernel
// Row tiles (256 / lanes a row) a block.  A block of down makes its rows' h itself (silu and the quantization, ~45
// instructions a value), so two tiles, requested together before it, halve that work: a block is 32 rows in every type, the
// K-quants' 8 lanes a row reaching that with one tile.  Down, 512 columns, 512 experts, top 10 plus the shared one, with
// weights from HBM: Q8_0 33.6 -> 28.9 us at 7 rows, 62 -> 50.4 at 16; Q5_1 34.6 -> 26.8, 65 -> 44.4; 1024 columns, 256
// experts: Q8_0 99 -> 81 at 16.  Three and four tiles lost part of it again, K-quants with two took 10% more, and gate|up,
// whose staging is a copy, gained nothing (Q8_0 71 -> 74).  Past 2048 columns two tiles' rows fill the registers.
template <int TYPE, int G, bool DOWN> constexpr int mv_tiles() { return DOWN && !is_kquant(TYPE) && G <= 4 ? 2 : 1; }
// One tile after all where the launch has little beside its longest blocks, the shared job's of T rows: those then last twice
// as long and nothing fills the chip meanwhile.  The line is blocks (of 32 rows) a compute unit per row of the window: below
// it 16 rows take (two tiles / one) Q8_0 31.5 / 27.3 us at 1.03 (2048 rows, top 4), 30.5 / 26.8 at 0.78, Q5_1 30.0 / 26.8 at
// 1.03; above it 31.6 / 31.8 and 29.9 / 32.7 at 1.52, 31.6 / 38.4 and 30.4 / 39.4 at 2.0.  At 2048 columns, whose h is four
// times as long to make, two tiles win from 1.27 (Q8_0, 16 rows 99.6 / 118.4); with 3 rows from 1.08 (Q8_0 12.0 / 13.4; at
// 0.79 8.5 / 7.9).
inline bool mv_two_tiles(int G, int T, int R, int njobs_max) {
    return (long) njobs_max * ((R + 31) / 32) >= (long) (T <= 4 ? 4 : G >= 4 ? 5 : 6) * 64 * T;   // of 256 units
}
// TYPE: SFNX_Q4_K / SFNX_Q5_K (8 lanes a row) or SFNX_Q8_0 (16 lanes a row); G: groups or blocks per lane = C / 512;
// TT: activation rows per pass; DOWN: activations from gu rows through swiglu (else q8_1 rows); NTL: row tiles a block.
template <int TYPE, int G, int TT, bool DOWN, int NTL>
__global__ void __launch_bounds__(MV_THREADS)
k_moe_mv(const uint8_t* __restrict__ A, size_t sa, int R, int C, const sfnx_job* __restrict__ jobs, const int* __restrict__ njobs,
         const void* __restrict__ in, float* __restrict__ out) {
    constexpr int LPR = lpr_of<TYPE>(), RPB = MV_THREADS / LPR;
    // the last job first: with a shared expert it is the shared one, which holds every row of the window; dispatched
    // last, its blocks ran alone at the launch's end
    const int nj = *njobs;
    if ((int) blockIdx.y >= nj) return;
    const int ji = ((int) blockIdx.y + nj - 1) % nj;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ sfnx_job jb;
    load_job(jb, jobs + ji);
    __syncthreads();
    const int r0 = blockIdx.x * NTL * RPB + threadIdx.x / LPR, ln = threadIdx.x % LPR;
    const Acts a = acts_in(lds, TT, C);
    const uint8_t* mat = expert_at(A, sa, jb.w);
    typename RowOf<TYPE, G>::R w[NTL];
#pragma unroll
    for (int i = 0; i < NTL; ++i)
        if (r0 + i * RPB < R) RowOf<TYPE, G>::load(w[i], mat, R, r0 + i * RPB, C, ln);
    for (int j0 = 0; j0 < jb.n; j0 += TT) {
        const int nn = min(TT, jb.n - j0);
        if (j0) __syncthreads();
        if constexpr (DOWN) stage_swiglu(a, (const float*) in, jb.y + j0, nn);
        else stage_q8_1(a, (const uint8_t*) in, jb.y + j0, nn);
        __syncthreads();
        for (int j = 0; j < nn; ++j)
#pragma unroll
            for (int i = 0; i < NTL; ++i) {
                const bool live = r0 + i * RPB < R;
                const float v = group_sum<LPR>(live ? w[i].dot(a, j, ln) : 0.f);
                if (live && ln == 0) out[(size_t) jb.out[j0 + j] * R + r0 + i * RPB] = v;
            }
    }
}

template <int TYPE, int G, int TT, bool DOWN>
void launch_mv(int njobs_max, int T, size_t lds, hipStream_t s, const uint8_t* A, size_t sa, int R, int C, const sfnx_job* jobs,
               const int* njobs, const void* in, float* out) {
    constexpr int rows = MV_THREADS / lpr_of<TYPE>(), NTL = mv_tiles<TYPE, G, DOWN>();
    auto go = [&](auto kern, int tiles) {
        kern<<<dim3((R + tiles * rows - 1) / (tiles * rows), njobs_max), MV_THREADS, lds, s>>>(A, sa, R, C, jobs, njobs, in, out);
    };
    if (NTL > 1 && mv_two_tiles(G, T, R, njobs_max)) go(k_moe_mv<TYPE, G, TT, DOWN, NTL>, NTL);
    else go(k_moe_mv<TYPE, G, TT, DOWN, 1>, 1);
}

template <int TYPE, int TT, bool DOWN>
void launch_g(int G, int njobs_max, int T, size_t lds, hipStream_t s, const uint8_t* A, size_t sa, int R, int C, const sfnx_job* jobs,
              const int* njobs, const void* in, float* out) {
    switch (G) {
        case 1: launch_mv<TYPE, 1, TT, DOWN>(njobs_max, T, lds, s, A, sa, R, C, jobs, njobs, in, out); break;
        case 2: launch_mv<TYPE, 2, TT, DOWN>(njobs_max, T, lds, s, A, sa, R, C, jobs, njobs, in, out); break;
        case 4: launch_mv<TYPE, 4, TT, DOWN>(njobs_max, T, lds, s, A, sa, R, C, jobs, njobs, in, out); break;
        case 5: launch_mv<TYPE, 5, TT, DOWN>(njobs_max, T, lds, s, A, sa, R, C, jobs, njobs, in, out); break;
        case 8: launch_mv<TYPE, 8, TT, DOWN>(njobs_max, T, lds, s, A, sa, R, C, jobs, njobs, in, out); break;
        default: throw std::runtime_error("input width must be 512, 1024, 2048, 2560 or 4096");
    }
}

template <bool DOWN>
void moe_mv(uint32_t type, const void* A, size_t sa, int n_in, int n_out, const sfnx_job* jobs, const int* njobs, int njobs_max,
            int T, const void* in, float* out, void* st) {
    require(expert_type_ok(type), TYPE_MSG);
    require(n_in > 0 && n_in % 512 == 0, "expert input width must be a multiple of 512");
    require(n_out > 0, "expert rows must be positive");
    require(stride_ok(sa, row_bytes(type, n_in) * (size_t) n_out), "expert stride smaller than a matrix");
    require(njobs_max >= 0 && njobs_max <= 65535, "njobs_max out of range");
    if (njobs_max == 0) return;
    const int G = n_in / 512;
    // activation rows staged per pass: up to 16 while they fit 64 KiB of LDS (the kernel loops over the passes)
    int TT = T <= 1 ? 1 : T <= 4 ? 4 : 16;
    if (acts_bytes(TT, n_in) > 64 * 1024) TT = 4;
    const size_t lds = acts_bytes(TT, n_in);
    require(lds <= 64 * 1024, "activation rows do not fit the LDS budget");
    hipStream_t s = stream_of(st);
    const uint8_t* a = (const uint8_t*) A;
#define SFNX_MV(TY, TTV) launch_g<TY, TTV, DOWN>(G, njobs_max, T, lds, s, a, sa, n_out, n_in, jobs, njobs, in, out)
    if (type == SFNX_Q4_K) {
        if (TT == 1) SFNX_MV(SFNX_Q4_K, 1);
        else if (TT == 4) SFNX_MV(SFNX_Q4_K, 4);
        else SFNX_MV(SFNX_Q4_K, 16);
    } else if (type == SFNX_Q5_K) {
        if (TT == 1) SFNX_MV(SFNX_Q5_K, 1);
        else if (TT == 4) SFNX_MV(SFNX_Q5_K, 4);
        else SFNX_MV(SFNX_Q5_K, 16);
    } else if (type == SFNX_Q4_0) {
        if (TT == 1) SFNX_MV(SFNX_Q4_0, 1);
        else if (TT == 4) SFNX_MV(SFNX_Q4_0, 4);
        else SFNX_MV(SFNX_Q4_0, 16);
    } else if (type == SFNX_Q5_1) {
        if (TT == 1) SFNX_MV(SFNX_Q5_1, 1);
        else if (TT == 4) SFNX_MV(SFNX_Q5_1, 4);
        else SFNX_MV(SFNX_Q5_1, 16);
    } else {
        if (TT == 1) SFNX_MV(SFNX_Q8_0, 1);
        else if (TT == 4) SFNX_MV(SFNX_Q8_0, 4);
        else SFNX_MV(SFNX_Q8_0, 16);
    }
#undef SFNX_MV
}

}  // namespace
}  // namespace sfnx

using namespace sfnx;

extern "C" int sfnx_moe_gate_up(const void* A, size_t sa, uint32_t type, int n_in, int n_out, const sfnx_job* jobs,
                                const int* njobs, int njobs_max, int T, const void* xq, float* gu, void* st) {
    return guarded("sfnx_moe_gate_up", [&] {
        require(T >= 1 && T <= SFNX_MAXT, "T out of range (1..16)");
        moe_mv<false>(type, A, sa, n_in, n_out, jobs, njobs, njobs_max, T, xq, gu, st);
    });
}

extern "C" int sfnx_moe_down(const void* A, size_t sa, uint32_t type, int n_in, int n_out, const sfnx_job* jobs,
                             const int* njobs, int njobs_max, int T, const float* gu, float* part, void* st) {
    return guarded("sfnx_moe_down", [&] {
        require(T >= 1 && T <= SFNX_MAXT, "T out of range (1..16)");
        moe_mv<true>(type, A, sa, n_in, n_out, jobs, njobs, njobs_max, T, gu, part, st);
    });
}
