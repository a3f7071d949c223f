#pragma once
#include "topk.hpp"

namespace sfnx {
namespace {

// A decode window's routing from its logits, one workgroup: the top-k of every row, a wavefront a row, then the decode job
// numbering of src/moe.cuh:164-198.  The fused decode runs it between the router and gate|up for windows of several rows
// (at batch 1 its gate|up blocks take the top-k themselves; with more rows each would repeat every row's top-k and the
// numbering), sfnx_router_route after the logits.
// Returns the job count.
constexpr int DR_THREADS = 1024;   // a wavefront per row (T <= 16) and a thread per pick
__device__ __forceinline__ int route_window(int T, int E, int K, int shared, const float* __restrict__ logits,
                                            int* __restrict__ topi_g, float* __restrict__ topw_g, sfnx_job* __restrict__ jg,
                                            sfnx_job* __restrict__ jd, int* __restrict__ njobs_g) {
    constexpr int NW = DR_THREADS / WAVE;
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, p = threadIdx.x, P = T * K;
    __shared__ int ex[MAX_P];
    __shared__ float sw[MAX_P];
    __shared__ unsigned rows[MAX_E];
    __shared__ int jobof[MAX_E], wsum[MAX_P / WAVE];
    for (int t = wave; t < T; t += NW) {
        int pick;
        float w;
        topk_wave_e(logits + (size_t) t * (E + 1), E, K, lane, pick, w);
        if (lane < K) {
            ex[t * K + lane] = pick;
            sw[t * K + lane] = w;
        }
    }
    __syncthreads();
    PickSlot ps;
    const int nr = pick_slots(ex, P, K, rows, jobof, wsum, ps);
    if (p < P) {
        topi_g[p] = ex[p];
        topw_g[p] = sw[p];
        if (ps.e >= 0) {
            const int j = ps.job;
            if (ps.slot == 0) {
                jg[j].w = jd[j].w = ps.e;
                jg[j].n = jd[j].n = ps.cnt;
            }
            jg[j].y[ps.slot] = p / K;
            jg[j].out[ps.slot] = jd[j].y[ps.slot] = jd[j].out[ps.slot] = p;
        }
    }
    if (shared) {
        if (p == 0) {
            jg[nr].w = jd[nr].w = E;
            jg[nr].n = jd[nr].n = T;
        }
        if (p < T) {
            jg[nr].y[p] = p;
            jg[nr].out[p] = jd[nr].y[p] = jd[nr].out[p] = P + p;
        }
    }
    if (p == 0) {
        njobs_g[0] = nr + (shared ? 1 : 0);
        njobs_g[1] = 0;
    }
    return nr + (shared ? 1 : 0);
}

__global__ void __launch_bounds__(DR_THREADS) k_dec_route(int T, int E, int K, int shared, const float* __restrict__ logits,
                                                          int* __restrict__ topi, float* __restrict__ topw,
                                                          sfnx_job* __restrict__ gu, sfnx_job* __restrict__ dn,
                                                          int* __restrict__ njobs) {
    route_window(T, E, K, shared, logits, topi, topw, gu, dn, njobs);
}

}  // namespace
}  // namespace sfnx
