// Device code of the Krylov solve shared by its translation units: block
// reductions and GMRES's norm step.
#pragma once
#include "krylov.hpp"

namespace mp {

constexpr int FIN = 1024;  // threads of the finishing kernels (one block per system)

// Sums of a block's NV values over its rows (WS: the product's shape), stored
// at partial[q * nb + lb] (plain stores: no atomics, the finishing kernel runs
// after the grid): over BLOCK rows, or over one slice (WS == 4, nb and lb then
// count slices; finish_sum adds a block's four in the same order).  Every
// thread of the block must call.
template <int NV, int WS = 1>
__device__ __forceinline__ void block_store(double (&v)[NV], double* __restrict__ partial, int lb,
                                            int nb) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (wid < WS_ROWS<WS> / 64)
#pragma unroll
        for (int q = 0; q < NV; ++q)
            for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_xor(v[q], off);
    if constexpr (WS == 4) {
        if (threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < NV; ++q) partial[(size_t)q * nb + lb] = v[q];
    } else {
        __shared__ double sh[NV][BLOCK / 64];
        if (wid < BLOCK / 64 && lane == 0)
#pragma unroll
            for (int q = 0; q < NV; ++q) sh[q][wid] = v[q];
        __syncthreads();
        if (threadIdx.x < NV) {
            const int q = threadIdx.x;
            double s = sh[q][0];
            for (int t = 1; t < BLOCK / 64; ++t) s += sh[q][t];
            partial[(size_t)q * nb + lb] = s;
        }
    }
}

// Sum of the partials of blocks [b0, b0 + cnt) per value (stride nb), in the
// order of a block of FIN threads whatever the block's size NT: FIN virtual
// threads each sum every FIN-th partial, their wavefronts reduce by shuffles,
// and the wavefronts' sums are added in order.  slices: the partials are per
// slice, four adjacent ones a block (stride 4 nb).  Every thread of the block
// receives the totals.
template <int NV, int NT = FIN>
__device__ __forceinline__ void finish_sum(const double* __restrict__ partial, int nb, int b0,
                                           int cnt, double (&tot)[NV], bool slices = false) {
    typedef double d4 __attribute__((ext_vector_type(4)));
    auto at = [&](int q, int b) {
        if (!slices) return partial[(size_t)q * nb + b0 + b];
        const d4 d = reinterpret_cast<const d4*>(partial)[(size_t)q * nb + b0 + b];
        return ((d.x + d.y) + d.z) + d.w;
    };
    const int lane = threadIdx.x & 63;
    if (cnt <= 64) {
        // one virtual wavefront holds every partial: each wavefront of the block
        // forms its sum on its own (the other fifteen are zeros)
#pragma unroll
        for (int q = 0; q < NV; ++q) tot[q] = lane < cnt ? at(q, lane) : 0.0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int q = 0; q < NV; ++q) tot[q] += __shfl_xor(tot[q], off);
        return;
    }
    __shared__ double sh[NV][FIN / 64];
#pragma unroll
    for (int u = 0; u < FIN / NT; ++u) {
        const int vt = (int)threadIdx.x + u * NT, wid = vt >> 6;
        double acc[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) acc[q] = 0.0;
        if (wid * 64 < cnt) {
            for (int b = vt; b < cnt; b += FIN)
#pragma unroll
                for (int q = 0; q < NV; ++q) acc[q] += at(q, b);
#pragma unroll
            for (int q = 0; q < NV; ++q)
                for (int off = 32; off > 0; off >>= 1) acc[q] += __shfl_xor(acc[q], off);
        }
        if (lane == 0)
#pragma unroll
            for (int q = 0; q < NV; ++q) sh[q][wid] = acc[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        double s = sh[q][0];
        for (int t = 1; t < FIN / 64; ++t) s += sh[q][t];
        tot[q] = s;
    }
}

// Givens rotation (c, s) with c a + s b = r, -s a + c b = 0
__device__ __forceinline__ void gm_givens(double a, double b, double& c, double& s, double& r) {
    if (b == 0.0) {
        c = 1.0;
        s = 0.0;
        r = a;
    } else {
        r = hypot(a, b);
        c = a / r;
        s = b / r;
    }
}

// One GMRES iteration's norm step for system q, by a block of NT threads:
// h_{j+1,j} = |w| from the block partials; the column's rotations, the new
// rotation and the residual estimate; then the stopping tests.
template <int NT>
__device__ __forceinline__ void gm_norm_step(const SegView& sg, int q,
                                             const double* __restrict__ partial, GmState* gm,
                                             GmFlags* fl, int m) {
    GmState* g = gm + q;
    if (g->stop) return;
    const Seg S = seg_at(sg, q);
    double tot[1];
    finish_sum<1, NT>(partial, sg.nrows / BLOCK, S.blk0, S.nblk, tot);
    // the column and the previous rotations into LDS in one parallel load;
    // the rotations themselves are sequential (thread 0)
    __shared__ double h[GM_MAX + 1], cs[GM_MAX], sn[GM_MAX];
    const int j = g->j;
    if ((int)threadIdx.x <= j) h[threadIdx.x] = g->h[threadIdx.x];
    if ((int)threadIdx.x < j) {
        cs[threadIdx.x] = g->cs[threadIdx.x];
        sn[threadIdx.x] = g->sn[threadIdx.x];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 0; i < j; ++i) {
            const double a = h[i], b = h[i + 1];
            h[i] = cs[i] * a + sn[i] * b;
            h[i + 1] = -sn[i] * a + cs[i] * b;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < j) g->R[j * GM_MAX + threadIdx.x] = h[threadIdx.x];
    if (threadIdx.x != 0) return;
    const double eta = sqrt(tot[0]);
    double c, s, r;
    gm_givens(h[j], eta, c, s, r);
    g->cs[j] = c;
    g->sn[j] = s;
    g->R[j * GM_MAX + j] = r;
    g->g[j + 1] = -s * g->g[j];
    g->g[j] = c * g->g[j];
    g->j = j + 1;
    g->iter += 1;
    const double res2 = g->g[j + 1] * g->g[j + 1];
    g->rr = res2;
    g->inv_eta = 1.0 / eta;
    g->sig[j + 1] = g->inv_eta;
    if (!(res2 <= 1.0e300) || !(fabs(r) <= 1.0e300))
        g->done = 5;
    else if (res2 <= g->tol2)
        g->done = 1;
    else if (r == 0.0)
        g->done = 5;  // singular Hessenberg column
    else if (g->iter >= g->maxit)
        g->done = 2;
    else if (g->j >= m)
        g->full = 1;
    // (the product beside this step reads the flag: either value is right for it)
    __hip_atomic_store(&g->stop, (g->done != 0 || g->full) ? 1 : 0, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    fl[q] = GmFlags{g->done, g->full, g->iter, g->cycles};
}

// The norm step of one or more systems, run by extra blocks of another launch
// (sg.nseg == 0: none).
struct GmNorm {
    SegView sg{};
    const double* partial = nullptr;
    GmState* gm = nullptr;
    GmFlags* fl = nullptr;
    int m = 0;
};

}  // namespace mp
