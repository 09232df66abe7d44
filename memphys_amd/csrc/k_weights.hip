// Part (a): batched PHS r^p + polynomial stencil weights, FP64.
//
// One workgroup (256 threads, 4 wavefronts) per stencil.  The saddle-point
// matrix [Phi P; P^T 0] (M = k + m) and the d+1 right-hand sides live in LDS;
// partial-pivot LU runs right-looking with one barrier-separated phase per
// step (pivot search on wave 0, row swap, multipliers, trailing update), then a
// column-oriented back substitution.  The arithmetic order is fixed: each
// matrix entry sees the same fma sequence as the oracle's sequential LU, so
// the weights agree bit for bit with it.
//
// Follows coefficient_computations.cpp:33-328 (shifting_scaling, A and rhs
// assembly, partialPivLu().solve) and cloud.cpp:207-279 (loop over nodes,
// row 0 of the solution is the stencil's weight row).
#include <algorithm>
#include <climits>

#include "mp_internal.hpp"

namespace mp {

namespace {

__device__ __forceinline__ double rpow_d(double r2, int q) {
    if (q >= 1) {
        double v = sqrt(r2);
        for (int s = 0; s < (q - 1) / 2; ++s) v = v * r2;
        return v;
    }
    double v = 1.0 / sqrt(r2);
    for (int s = 0; s < (-q - 1) / 2; ++s) v = v / r2;
    return v;
}

__device__ __forceinline__ double ipow_d(double x, int e) {
    double v = 1.0;
    for (int s = 0; s < e; ++s) v = v * x;
    return v;
}

// Right-hand-side entries of saddle-point row i (columns gx, gy, (gz), lap at
// out[0..dim]) with the oracle's formulas (coefficient_computations.cpp:108-292):
// a stencil row (is_pt) differentiates the PHS kernel between the scaled point
// xi and the scaled centre xc; a polynomial row differentiates the monomial
// with exponents e at xc.  sc holds the per-axis scale factors.
// ONCE: r^(phs-2) and r^(phs-4) are formed once per row, for the register
// kernels.  The LDS kernels form them at each use: held across the loops they
// took 28 registers more, eight wavefronts per SIMD became five or six, and
// 64k mixed stencils of 60 rows went from 14.6 to 19.8 ms, 10k FP64 stencils of
// 26 rows with condition estimates from 1.03 to 1.09 ms.
template <bool ONCE>
__device__ __forceinline__ void rhs_entries(bool is_pt, int dim, int phs, const double* xi,
                                            const double* xc, const double* sc, const int* e,
                                            double* out) {
    const double p = (double)phs;
    if (is_pt) {
        double r2 = 0.0;
        for (int a = 0; a < dim; ++a) {
            double d = xi[a] - xc[a];
            r2 = r2 + d * d;
        }
        double q2 = ONCE ? rpow_d(r2, phs - 2) : 0.0;
        for (int a = 0; a < dim; ++a) {
            double v = (-p) * (xi[a] - xc[a]);
            if (!ONCE) q2 = rpow_d(r2, phs - 2);
            v = v * q2;
            out[a] = v / sc[a];
        }
        double lp = 0.0;
        if (fabs(r2) > 1e-14) {
            double g[3] = {0.0, 0.0, 0.0};
            double q4 = ONCE ? rpow_d(r2, phs - 4) : 0.0;
            for (int a = 0; a < dim; ++a) {
                double d = xi[a] - xc[a];
                double d2 = d * d;
                if (!ONCE) q4 = rpow_d(r2, phs - 4);
                double v = (p * p) * d2 * q4;
                v = v - (2.0 * p) * d2 * q4;
                if (!ONCE) q2 = rpow_d(r2, phs - 2);
                v = v + p * q2;
                g[a] = v / (sc[a] * sc[a]);
            }
            lp = g[0] + g[1];
            if (dim == 3) lp = lp + g[2];
        }
        out[dim] = lp;
        return;
    }
    const double x0 = xc[0], x1 = xc[1], x2 = (dim == 3) ? xc[2] : 0.0;
    for (int a = 0; a < dim; ++a) {
        double v = 0.0;
        if (e[a] > 0) {
            if (a == 1) {
                v = ipow_d(x0, e[0]);
                v = v * (double)e[1];
                v = v * ipow_d(x1, e[1] - 1);
                if (dim == 3) v = v * ipow_d(x2, e[2]);
            } else if (a == 0) {
                v = (double)e[0] * ipow_d(x0, e[0] - 1);
                v = v * ipow_d(x1, e[1]);
                if (dim == 3) v = v * ipow_d(x2, e[2]);
            } else {
                v = (double)e[2] * ipow_d(x2, e[2] - 1);
                v = v * ipow_d(x0, e[0]);
                v = v * ipow_d(x1, e[1]);
            }
            v = v / sc[a];
        }
        out[a] = v;
    }
    double g0 = 0.0, g1 = 0.0, g2 = 0.0;
    if (e[0] > 1) {
        double v = (double)e[0] * ((double)e[0] - 1.0) * ipow_d(x0, e[0] - 2);
        v = v * ipow_d(x1, e[1]);
        if (dim == 3) v = v * ipow_d(x2, e[2]);
        g0 = v / (sc[0] * sc[0]);
    }
    if (e[1] > 1) {
        double v = (double)e[1] * ((double)e[1] - 1.0) * ipow_d(x1, e[1] - 2);
        v = v * ipow_d(x0, e[0]);
        if (dim == 3) v = v * ipow_d(x2, e[2]);
        g1 = v / (sc[1] * sc[1]);
    }
    if (dim == 3 && e[2] > 1) {
        double v = (double)e[2] * ((double)e[2] - 1.0) * ipow_d(x2, e[2] - 2);
        v = v * ipow_d(x0, e[0]);
        v = v * ipow_d(x1, e[1]);
        g2 = v / (sc[2] * sc[2]);
    }
    double lp = g0 + g1;
    if (dim == 3) lp = lp + g2;
    out[dim] = lp;
}

__global__ __launch_bounds__(256) void weights_fp64_kernel(
    int dim, int phs, int m, const int* __restrict__ exps, SellView sv,
    const double* __restrict__ xyz, int npad, double* __restrict__ gx, double* __restrict__ gy,
    double* __restrict__ gz, double* __restrict__ lap, double* __restrict__ cond,
    const int* __restrict__ rows, const int* __restrict__ only, int t0, double* gwork,
    long gstride) {
    extern __shared__ double lds[];
    __shared__ double s_mn[3], s_sc[3];
    __shared__ double s_anorm, s_red[4];
    __shared__ int s_piv, s_jm;
    __shared__ int s_e[MAX_POLY * 3];

    // stencil t of the list (or row t); the work arrays in LDS, or for
    // systems too large for it in this block's share of a global work area
    // (the same operations in the same order either way)
    const int t = t0 + (int)blockIdx.x;
    if (only && !only[t]) return;  // a stencil the register kernel finished
    const int r = rows ? rows[t] : t;
    if (r >= sv.nv || sv.len[r] == 0) return;  // padding rows carry no stencil
    const int tid = threadIdx.x;
    const int k = sv.len[r];
    const int M = k + m;
    const int LDA = M + 1;
    const int nr = dim + 1;
    double* A = gwork ? gwork + (size_t)blockIdx.x * (size_t)gstride : lds;
    double* R = A + M * LDA;
    double* xs = R + M * 4;
    const int base = sell_base(sv.sptr, r);

    for (int i = tid; i < m * dim; i += blockDim.x) s_e[i] = exps[i];
    for (int t = tid; t < k; t += blockDim.x) {
        const int c = sv.col[base + sell_off(t)];
        for (int a = 0; a < dim; ++a) xs[t * 3 + a] = xyz[(size_t)a * npad + c];
    }
    __syncthreads();
    if (tid < dim) {
        double mn = xs[tid], mx = xs[tid];
        for (int t = 0; t < k; ++t) {
            double v = xs[t * 3 + tid];
            if (mn > v) mn = v;
            if (mx < v) mx = v;
        }
        s_mn[tid] = mn;
        s_sc[tid] = mx - mn;
    }
    __syncthreads();
    for (int t = tid; t < k * dim; t += blockDim.x) {
        const int j = t / dim, a = t - j * dim;
        xs[j * 3 + a] = (xs[j * 3 + a] - s_mn[a]) / s_sc[a];
    }
    __syncthreads();

    // ---- assemble A (M x M) ----
    for (int idx = tid; idx < M * M; idx += blockDim.x) {
        const int i = idx / M, j = idx - i * M;
        double v = 0.0;
        if (i < k && j < k) {
            if (i != j) {
                double s = 0.0;
                for (int a = 0; a < dim; ++a) {
                    double d = xs[i * 3 + a] - xs[j * 3 + a];
                    s = s + d * d;
                }
                v = rpow_d(s, phs);
            }
        } else if (i < k || j < k) {
            const int pt = (i < k) ? i : j;
            const int t = (i < k) ? j - k : i - k;
            v = ipow_d(xs[pt * 3 + 0], s_e[t * dim + 0]);
            for (int a = 1; a < dim; ++a) v = v * ipow_d(xs[pt * 3 + a], s_e[t * dim + a]);
        }
        A[i * LDA + j] = v;
    }
    // ---- right-hand sides: gx, gy, (gz), lap ----
    for (int i = tid; i < M; i += blockDim.x)
        rhs_entries<false>(i < k, dim, phs, xs + 3 * (i < k ? i : 0), xs, s_sc,
                    s_e + (i < k ? 0 : i - k) * dim, R + 4 * i);
    __syncthreads();

    // ---- 1-norm of A (for the condition estimate) ----
    int* perm = (int*)xs;  // the scaled coordinates are no longer needed
    if (cond) {
        if (tid == 0) s_anorm = 0.0;
        __syncthreads();
        for (int j = tid; j < M; j += blockDim.x) {
            double sum = 0.0;
            for (int i = 0; i < M; ++i) sum += fabs(A[i * LDA + j]);
            atomicMax((unsigned long long*)&s_anorm, (unsigned long long)__double_as_longlong(sum));
        }
    }
    __syncthreads();
    for (int i = tid; i < M; i += blockDim.x) perm[i] = i;
    __syncthreads();

    // ---- LU with partial pivoting, right-looking ----
    for (int c = 0; c < M; ++c) {
        if (tid < 64) {
            double best = -1.0;
            int bi = M;
            for (int i = c + tid; i < M; i += 64) {
                double v = fabs(A[i * LDA + c]);
                if (v > best) {
                    best = v;
                    bi = i;
                }
            }
            for (int off = 32; off > 0; off >>= 1) {
                double ob = __shfl_xor(best, off);
                int oi = __shfl_xor(bi, off);
                if (ob > best || (ob == best && oi < bi)) {
                    best = ob;
                    bi = oi;
                }
            }
            if (tid == 0) s_piv = bi;
        }
        __syncthreads();
        const int piv = s_piv;
        if (piv != c) {
            if (tid == 0) {
                const int tp = perm[c];
                perm[c] = perm[piv];
                perm[piv] = tp;
            }
            for (int j = tid; j < M + nr; j += blockDim.x) {
                if (j < M) {
                    double t0 = A[c * LDA + j];
                    A[c * LDA + j] = A[piv * LDA + j];
                    A[piv * LDA + j] = t0;
                } else {
                    const int q = j - M;
                    double t0 = R[c * 4 + q];
                    R[c * 4 + q] = R[piv * 4 + q];
                    R[piv * 4 + q] = t0;
                }
            }
            __syncthreads();
        }
        const double d = A[c * LDA + c];
        if (d != 0.0) {
            for (int i = c + 1 + tid; i < M; i += blockDim.x) A[i * LDA + c] = A[i * LDA + c] / d;
            __syncthreads();
            const int nrow = M - c - 1;
            const int ncol = M - c - 1 + nr;
            for (int idx = tid; idx < nrow * ncol; idx += blockDim.x) {
                const int ii = idx / ncol;
                const int jj = idx - ii * ncol;
                const int i = c + 1 + ii;
                const double l = A[i * LDA + c];
                if (jj < nrow) {
                    const int j = c + 1 + jj;
                    A[i * LDA + j] = fma(-l, A[c * LDA + j], A[i * LDA + j]);
                } else {
                    const int q = jj - nrow;
                    R[i * 4 + q] = fma(-l, R[c * 4 + q], R[i * 4 + q]);
                }
            }
        }
        __syncthreads();
    }
    // ---- back substitution (column oriented) ----
    for (int c = M - 1; c >= 0; --c) {
        if (tid < nr) R[c * 4 + tid] = R[c * 4 + tid] / A[c * LDA + c];
        __syncthreads();
        for (int idx = tid; idx < c * nr; idx += blockDim.x) {
            const int i = idx / nr, q = idx - i * nr;
            R[i * 4 + q] = fma(-A[i * LDA + c], R[c * 4 + q], R[i * 4 + q]);
        }
        __syncthreads();
    }
    for (int t = tid; t < k; t += blockDim.x) {
        const size_t slot = (size_t)base + (size_t)sell_off(t);
        gx[slot] = R[t * 4 + 0];
        gy[slot] = R[t * 4 + 1];
        if (dim == 3) gz[slot] = R[t * 4 + 2];
        lap[slot] = R[t * 4 + dim];
    }
    if (!cond) return;
    __syncthreads();
    // ---- Hager (1984) / Higham (1988) estimate of ||A^-1||_1 from the LU factors ----
    double* w = R;          // work vectors reuse the right-hand-side storage
    double* xv = R + M;
    double* yv = R + 2 * M;
    bool singular = false;
    for (int c = 0; c < M; ++c) singular |= (A[c * LDA + c] == 0.0);
    if (singular) {
        if (tid == 0) cond[r] = __builtin_inf();
        return;
    }
    // w = A^-1 v  (v in xv): w = P v, forward with unit L, backward with U
    auto solve = [&](const double* v, double* out) {
        for (int i = tid; i < M; i += blockDim.x) out[i] = v[perm[i]];
        __syncthreads();
        for (int c = 0; c < M; ++c) {
            for (int i = c + 1 + tid; i < M; i += blockDim.x) out[i] = fma(-A[i * LDA + c], out[c], out[i]);
            __syncthreads();
        }
        for (int c = M - 1; c >= 0; --c) {
            if (tid == 0) out[c] = out[c] / A[c * LDA + c];
            __syncthreads();
            for (int i = tid; i < c; i += blockDim.x) out[i] = fma(-A[i * LDA + c], out[c], out[i]);
            __syncthreads();
        }
    };
    // out = A^-T v: U^T then L^T (column oriented), then un-permute
    auto solve_t = [&](const double* v, double* tmpv, double* out) {
        for (int i = tid; i < M; i += blockDim.x) tmpv[i] = v[i];
        __syncthreads();
        for (int c = 0; c < M; ++c) {
            if (tid == 0) tmpv[c] = tmpv[c] / A[c * LDA + c];
            __syncthreads();
            for (int i = c + 1 + tid; i < M; i += blockDim.x) tmpv[i] = fma(-A[c * LDA + i], tmpv[c], tmpv[i]);
            __syncthreads();
        }
        for (int c = M - 1; c >= 0; --c) {
            for (int i = tid; i < c; i += blockDim.x) tmpv[i] = fma(-A[c * LDA + i], tmpv[c], tmpv[i]);
            __syncthreads();
        }
        for (int i = tid; i < M; i += blockDim.x) out[perm[i]] = tmpv[i];
        __syncthreads();
    };
    auto l1 = [&](const double* v) {  // sequential sum on thread 0, broadcast
        if (tid == 0) {
            double sum = 0.0;
            for (int i = 0; i < M; ++i) sum += fabs(v[i]);
            s_red[0] = sum;
        }
        __syncthreads();
        double res = s_red[0];
        __syncthreads();
        return res;
    };
    for (int i = tid; i < M; i += blockDim.x) xv[i] = 1.0 / (double)M;
    __syncthreads();
    double est = 0.0;
    int jlast = -1;
    for (int itn = 0; itn < 5; ++itn) {
        solve(xv, yv);
        est = fmax(est, l1(yv));
        for (int i = tid; i < M; i += blockDim.x) w[i] = (yv[i] >= 0.0) ? 1.0 : -1.0;
        __syncthreads();
        solve_t(w, yv, w);
        if (tid == 0) {
            int jm = 0;
            double zx = 0.0;
            for (int i = 0; i < M; ++i) {
                if (fabs(w[i]) > fabs(w[jm])) jm = i;
                zx += w[i] * xv[i];
            }
            s_jm = (fabs(w[jm]) <= zx || jm == jlast) ? -1 : jm;
        }
        __syncthreads();
        const int jm = s_jm;
        if (jm < 0) break;
        jlast = jm;
        for (int i = tid; i < M; i += blockDim.x) xv[i] = (i == jm) ? 1.0 : 0.0;
        __syncthreads();
    }
    for (int i = tid; i < M; i += blockDim.x)
        xv[i] = ((i % 2) ? -1.0 : 1.0) * (1.0 + (double)i / (double)(M > 1 ? M - 1 : 1));
    __syncthreads();
    solve(xv, yv);
    est = fmax(est, 2.0 * l1(yv) / (3.0 * (double)M));
    if (tid == 0) cond[r] = s_anorm * est;
}


// ---------------------------------------------------------------------------
// FP64 weights with the saddle-point matrix in registers: one wavefront per
// stencil (two for 64 < M <= 96), thread i holding row i.  At pivot step c a
// row keeps its columns c..M-1 in a[0..M-1-c]: the trailing update writes a[j]
// from a[j+1], so the row shifts by one column per step and every register
// index is a compile-time constant.  The update width is rounded up to a
// multiple of 8 (the entries past the row's end are never read back).  Only the
// rows below the pivot are updated, so a finished row keeps its row of U in
// registers; U and the forward-eliminated right-hand sides go to LDS for the
// back substitution.  Every entry sees the oracle's roundings in the oracle's
// order: the same division for each multiplier, fma(-l, u, a) for each update,
// the pivot chosen as the first maximum in position order (a NaN on the
// diagonal position keeps it), and the column-oriented back substitution.  The
// weights are therefore bit-identical to the oracle's and to the LDS kernel's.
//
// One wavefront is bound by its vector instructions (about 80 % busy at three
// wavefronts per SIMD).  183k stencils of 60 rows: 7.3 ms, 10.7 ms with the
// whole of U in LDS (two wavefronts per SIMD), the monomials by loops over their
// exponents, the matrix column by column and the back substitution with four
// divisions per column.  64k stencils of 70 to 80 rows on two wavefronts: 10.3 ms
// (11.1 ms); their steps wait for LDS and the barrier.

// f(integral_constant i) for i in [I, N).
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

__device__ __forceinline__ double readlane_d(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// d = a * b + c, one rounding, as the three-address v_fma_f64: the result may
// go to any register.  (The compiler's own fma becomes the two-address
// v_fmac_f64, which writes over c; for the shifted rows below that register is
// the neighbour's, and every step would end by copying the row back.)
__device__ __forceinline__ double fma3(double a, double b, double c) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

// The same with b in scalar registers (a value that readlane has just fetched).
__device__ __forceinline__ double fma3s(double a, double b, double c) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "s"(b), "v"(c));
    return d;
}

// Maximum of a double over the wavefront (no NaN among the inputs), through
// DPP row shifts and broadcasts: lane 63 ends with the maximum, which every
// lane receives.  Max is exact and order-free, so any combination order gives
// the same value.
__device__ __forceinline__ double wave_max_d(double v) {
    int hi = __double2hiint(v), lo = __double2loint(v);
#define MP_DPP_MAX(ctrl, rows)                                                    \
    {                                                                             \
        const int th = __builtin_amdgcn_update_dpp(hi, hi, ctrl, rows, 0xf, false); \
        const int tl = __builtin_amdgcn_update_dpp(lo, lo, ctrl, rows, 0xf, false); \
        v = fmax(v, __hiloint2double(th, tl));                                    \
        hi = __double2hiint(v);                                                   \
        lo = __double2loint(v);                                                   \
    }
    MP_DPP_MAX(0x111, 0xf)  // row_shr:1
    MP_DPP_MAX(0x112, 0xf)  // row_shr:2
    MP_DPP_MAX(0x114, 0xf)  // row_shr:4
    MP_DPP_MAX(0x118, 0xf)  // row_shr:8: lane 15 of each row holds the row's maximum
    MP_DPP_MAX(0x142, 0xa)  // row_bcast:15 into rows 1 and 3
    MP_DPP_MAX(0x143, 0xc)  // row_bcast:31 into rows 2 and 3: lane 63 holds the maximum
#undef MP_DPP_MAX
    return __hiloint2double(__builtin_amdgcn_readlane(hi, 63), __builtin_amdgcn_readlane(lo, 63));
}

// Maximum of an unsigned over the wavefront, the same way (one instruction per
// step: 0 stands in where no lane is read).
__device__ __forceinline__ unsigned wave_max_u(unsigned v) {
#define MP_DPP_MAXU(ctrl, rows)                                                              \
    v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false));
    MP_DPP_MAXU(0x111, 0xf)
    MP_DPP_MAXU(0x112, 0xf)
    MP_DPP_MAXU(0x114, 0xf)
    MP_DPP_MAXU(0x118, 0xf)
    MP_DPP_MAXU(0x142, 0xa)
    MP_DPP_MAXU(0x143, 0xc)
#undef MP_DPP_MAXU
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Lanes whose |v| is the largest among those with act (none of them NaN): the
// bits of non-negative doubles order as integers, so the high words decide, and
// only lanes that tie there compare their low words.
__device__ __forceinline__ unsigned long long wave_argmax(double v, bool act) {
    const unsigned hi = (unsigned)__double2hiint(v) & 0x7FFFFFFFu;
    const unsigned mh = wave_max_u(act ? hi + 1u : 0u);  // (0: no lane takes part)
    bool top = act && hi + 1u == mh;
    unsigned long long b = __ballot(top);
    if (b & (b - 1)) {  // several lanes: uniform branch
        const unsigned lo = (unsigned)__double2loint(v);
        const unsigned ml = wave_max_u(top ? lo : 0u);
        b = __ballot(top && lo == ml);
    }
    return b;
}

// Minimum and maximum over the lanes that hold a point, each equal to the
// oracle's left-to-right scan (a later value replaces the current one only when
// strictly smaller / larger): the extreme value by DPP reductions, then the
// exact bits of the first lane (lowest index) holding an equal value, which is
// the one the scan keeps among equal values such as -0 and +0.
__device__ __forceinline__ void ordered_minmax(double& mn, double& mx, int& has, int lane) {
    (void)lane;
    const double big = __builtin_inf();
    const double x = mn;
    const double vmax = wave_max_d(has ? x : -big);
    const double vmin = -wave_max_d(has ? -x : -big);
    const unsigned long long bmax = __ballot(has && x == vmax);
    const unsigned long long bmin = __ballot(has && x == vmin);
    mx = bmax ? readlane_d(x, __ffsll((long long)bmax) - 1) : vmax;
    mn = bmin ? readlane_d(x, __ffsll((long long)bmin) - 1) : vmin;
    has = __ballot(has) != 0ull;
}

// First column of U's right strip: the single-wavefront kernel of up to 64 rows
// puts its columns 48.. and then its columns 0..47 in LDS for the back
// substitution, so that a stencil needs about 12 KB and the registers, not LDS,
// set the number of wavefronts in flight (the whole triangle: 18 KB, 8 blocks
// per CU instead of 12).
constexpr int wave_split(int NW, int AW) { return NW == 1 && AW > 48 ? 48 : AW; }

// LDS doubles the register-resident kernel needs for a stencil of M = k + m.
template <int NW, int AW>
constexpr int wave_lds_doubles(int m) {
    const int M = AW, k = AW - m, H = wave_split(NW, AW);
    const int left = H * (H + 1) / 2, right = M * ((M - H) | 1);
    const int cand = NW == 2 ? 4 * (AW + 6) : AW + 2;  // published pivot rows
    const int asm_ = 4 * k + m * k;                    // scaled coordinates and monomials
    int n = 4 * M + left;
    if (H < M && right > left) n = 4 * M + right;
    if (n < cand) n = cand;
    return n > asm_ ? n : asm_;
}

// The pivot steps of one wavefront's rows.  phase<W> runs the steps whose
// trailing width M-1-c lies in (W-8, W] with a fixed update width W, then hands
// over to phase<W-8>: each loop body has one static width, so the shifted row
// stays in the same registers from step to step.
template <int NW, int AW>
struct WaveLu {
    double (&a)[AW + 1];
    double (&r)[4];
    double* pub;         // published pivot rows
    const double* zero;  // AW + 1 zeros
    double* s_cv;
    int* s_cp;
    int M, pos, lane, wv;
    bool valid;
    bool zero_pivot = false;  // a single wavefront met an exactly zero pivot (stencil redone)

    // One wavefront (M <= 64).  The pivot is found with a DPP maximum and a
    // ballot, and only the rows below the pivot are updated (exec mask), so a
    // pivot row keeps its U row in registers until the end (store_u).
    template <int W>
    __device__ __forceinline__ void step1(int c) {
        const bool act = valid && pos >= c;
        const bool isn = !(a[0] == a[0]);
        const unsigned long long tie = wave_argmax(a[0], act && !isn);
        int piv;
        if (__ballot(valid && pos == c && isn) != 0ull || tie == 0ull) {
            piv = c;  // a NaN on the diagonal position keeps it (nothing compares greater)
        } else if (__popcll(tie) == 1) {
            piv = __builtin_amdgcn_readlane(pos, __ffsll((long long)tie) - 1);
        } else {  // exact ties: the first in position order
            int cp = ((tie >> lane) & 1ull) ? pos : INT_MAX;
            for (int off = 32; off > 0; off >>= 1) cp = min(cp, __shfl_xor(cp, off));
            piv = __builtin_amdgcn_readfirstlane(cp);
        }
        if (pos == c) pos = piv;
        else if (pos == piv) pos = c;
        const int pl = __ffsll((long long)__ballot(pos == c)) - 1;  // the pivot row's lane
        // The pivot row reaches the other rows two ways at once: its first
        // quarter through LDS (one lane writes, every lane reads the same
        // address), the rest by readlane into scalar operands.  7.3 ms for 183k
        // stencils of 60 rows with a quarter, 7.4 with a half, 7.8 with three.
        constexpr int L = (W / 4) & ~1;
        if (L > 0) {
            if (pos == c) {
#pragma unroll
                for (int j = 1; j <= L; ++j) pub[j + 1] = a[j];  // (a[1] 16-byte aligned)
            }
            __syncthreads();
        }
        const double* u = pub + 1;
        const double d = readlane_d(a[0], pl);
        if (d == 0.0) {  // a singular column (the oracle skips it): left to the LDS kernel
            zero_pivot = true;
            return;
        }
        // Every readlane runs with the whole wavefront active, in front of the
        // masked fmas that use it: inside the mask the pivot's lane is off, and
        // a spill, a reload or a register move there would leave its copy stale.
        // (Eight columns at a time, or 16 or 24: 18.3 ms for 250k 3D stencils,
        // the time of one masked block with the readlanes inside.)
        const bool below = pos > c;
        const double nl = -(a[0] / d);
        constexpr int T = 8, G = W > L ? (W - L + T - 1) / T : 1;
        static_for<0, G>([&](auto g) {
            constexpr int i = decltype(g)::value, j0 = L + T * i;
            constexpr int n = W - j0 < T ? W - j0 : T;
            double s[T], sr[4];
#pragma unroll
            for (int t = 0; t < n; ++t) s[t] = readlane_d(a[j0 + t + 1], pl);
            if (i == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) sr[q] = readlane_d(r[q], pl);
            }
            if (below) {
                if (i == 0) {
#pragma unroll
                    for (int j = 0; j < L; ++j) a[j] = fma3(nl, u[j + 1], a[j + 1]);
#pragma unroll
                    for (int q = 0; q < 4; ++q) r[q] = fma3s(nl, sr[q], r[q]);
                }
#pragma unroll
                for (int t = 0; t < n; ++t) a[j0 + t] = fma3s(nl, s[t], a[j0 + t + 1]);
            }
        });
    }

    // Two wavefronts: each publishes the candidate among its own rows, whole,
    // and one barrier later both read the winner's, so a step has a single
    // barrier (two buffers in turn: a wavefront one step ahead writes the other).
    template <int W>
    __device__ __forceinline__ void step2(int c) {
        const bool act = valid && pos >= c;
        const bool isn = !(a[0] == a[0]);
        const unsigned long long diag_nan = __ballot(valid && pos == c && isn);
        unsigned long long tie = wave_argmax(a[0], act && !isn);
        double key = -1.0;  // |candidate|; a NaN on the diagonal position wins over all
        int cp = INT_MAX, cl = 64;
        if (diag_nan) {
            cl = __ffsll((long long)diag_nan) - 1;
            key = __builtin_inf();
            cp = -1;
        } else if (tie) {
            cl = __ffsll((long long)tie) - 1;
            key = fabs(readlane_d(a[0], cl));
            cp = __builtin_amdgcn_readlane(pos, cl);
            if (__popcll(tie) > 1) {  // exact ties: the first in position order
                cp = ((tie >> lane) & 1ull) ? pos : INT_MAX;
                for (int off = 32; off > 0; off >>= 1) cp = min(cp, __shfl_xor(cp, off));
                cp = __builtin_amdgcn_readfirstlane(cp);
                cl = __ffsll((long long)__ballot(act && pos == cp)) - 1;
            }
        }
        const int buf = 2 * (c & 1);
        if (lane == cl) {
            double* o = pub + (buf + wv) * (AW + 6);
#pragma unroll
            for (int j = 0; j <= W; ++j) o[j + 1] = a[j];
#pragma unroll
            for (int q = 0; q < 4; ++q) o[AW + 2 + q] = r[q];
        }
        if (lane == 0) {
            s_cv[buf + wv] = key;
            s_cp[buf + wv] = cp;
        }
        __syncthreads();
        const double v0 = s_cv[buf], v1 = s_cv[buf + 1];
        const int p0 = s_cp[buf], p1 = s_cp[buf + 1];
        const bool one = v0 == v1 ? p1 < p0 : v1 > v0;  // wavefront 1 holds the pivot
        const int best = one ? p1 : p0;
        const int piv = best < 0 ? c : best;
        if (pos == c) pos = piv;
        else if (pos == piv) pos = c;
        // A zero pivot leaves the rows below untouched (the oracle skips the
        // column): multiplier -0 against a row of +0 gives x + (-0) = x exactly
        // for every x, so the same instructions run in both cases.
        const double* u = pub + (buf + (one ? 1 : 0)) * (AW + 6) + 1;
        const double* y = u + AW + 1;
        const double d = u[0];
        const bool sing = (d == 0.0);
        if (sing) u = y = zero;
        if (pos > c) {
            const double nl = sing ? -0.0 : -(a[0] / d);
#pragma unroll
            for (int j = 0; j < W; ++j) a[j] = fma3(nl, u[j + 1], a[j + 1]);
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] = fma3(nl, y[q], r[q]);
        }
    }

    // After the last step every row holds its U row (columns pos..M-1 in
    // a[0..M-1-pos]) and its forward-eliminated right-hand sides.  Columns
    // [0, H) go to LDS packed (row p at p*H - p(p-1)/2), columns [H, M) with a
    // row stride of rs.
    __device__ __forceinline__ void store_left(double* U, int H) const {
        if (!valid || pos >= H) return;
        const int b = pos * H - pos * (pos - 1) / 2;
#pragma unroll
        for (int j = 0; j < AW; ++j)
            if (j < H - pos) U[b + j] = a[j];
    }
    __device__ __forceinline__ void store_right(double* U, int H, int rs) const {
        if (!valid) return;
        const int b = pos * rs + pos - H;
#pragma unroll
        for (int j = 0; j < AW; ++j)
            if ((unsigned)(j + pos - H) < (unsigned)(M - H)) U[b + j] = a[j];
    }

    template <int W>
    __device__ __forceinline__ void phase(int& c) {
        for (; c < M && M - 1 - c > W - 8 && !zero_pivot; ++c) {
            if constexpr (NW == 1) step1<W>(c);
            else step2<W>(c);
        }
        if constexpr (W > 0) phase<W - 8>(c);
    }
};

// Back substitution, column oriented.  16 lanes per right-hand side, lane l of
// a group holding its rows 16*b + l, so a column takes one division and its
// quotient reaches the group through one DPP broadcast; the four right-hand
// sides go side by side.  (One lane per row with the four one after the other
// took 38k cycles for 60 rows.)
//
// y / d from the correctly rounded reciprocal of the row's diagonal (Markstein
// 1990): q1 is within one ulp, the remainder y - d*q1 is then exact, and its
// correction with RN(1/d) gives the correctly rounded quotient.  That holds
// while nothing under- or overflows; outside [2^-400, 2^400], for infinities
// and NaN the division itself runs.
struct BackRow {
    double y, d, rd;
    bool dok;  // the diagonal is in range
};

__device__ __forceinline__ double back_quotient(const BackRow& b, bool ask) {
    const double q0 = b.y * b.rd;
    double e = fma(-b.d, q0, b.y);
    const double q1 = fma(e, b.rd, q0);
    e = fma(-b.d, q1, b.y);
    double q = fma(e, b.rd, q1);
    const double ay = fabs(b.y);
    const bool zero = ay == 0.0;
    q = zero ? q0 : q;
    const bool ok = b.dok && (zero || (ay >= 0x1p-400 && ay <= 0x1p400));
    if (__ballot(ask && !ok)) q = b.y / b.d;  // uniform
    return q;
}

// Columns c = 16*B + C .. 16*B (C counts down) of the rows 0..16*B+15: at(p, c)
// is the LDS index of U's entry.
template <int B, int C, int NB, class At>
__device__ __forceinline__ void back_columns(BackRow (&row)[NB], const double* U, int M, int l,
                                             const At& at) {
    constexpr int c = 16 * B + C;
    if (c < M) {
        double u[B + 1];
#pragma unroll
        for (int b = 0; b <= B; ++b) u[b] = b < B || l < C ? U[at(16 * b + l, c)] : 0.0;
        const double q = back_quotient(row[B], l == C);
        const int qh = __double2hiint(q), ql = __double2loint(q);
        const double x = __hiloint2double(
            __builtin_amdgcn_update_dpp(0, qh, 0x150 + C, 0xf, 0xf, true),   // row_newbcast:C
            __builtin_amdgcn_update_dpp(0, ql, 0x150 + C, 0xf, 0xf, true));
#pragma unroll
        for (int b = 0; b < B; ++b) row[b].y = fma(-u[b], x, row[b].y);
        if (l < C) row[B].y = fma(-u[B], x, row[B].y);
        else if (l == C) row[B].y = x;
    }
    if constexpr (C > 0) back_columns<B, C - 1>(row, U, M, l, at);
}

// Column blocks B .. LO.
template <int B, int LO, int NB, class At>
__device__ __forceinline__ void back_blocks(BackRow (&row)[NB], const double* U, int M, int l,
                                            const At& at) {
    back_columns<B, 15>(row, U, M, l, at);
    if constexpr (B > LO) back_blocks<B - 1, LO>(row, U, M, l, at);
}

// Row i of the saddle-point matrix, from the assembly tables in LDS.
struct SaddleRow {
    const double *xs, *P;
    int i, it, ip, k, M, dim, phs;
    double x0, x1, x2;

    // Columns J .. J+T-1, all of them stencil points: their square roots side by side.
    template <int J, int T, int N>
    __device__ __forceinline__ void points(double (&a)[N]) const {
        double sq[T], v[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const double d0 = x0 - xs[4 * (J + t)], d1 = x1 - xs[4 * (J + t) + 1];
            double s = 0.0;
            s = s + d0 * d0;
            s = s + d1 * d1;
            sq[t] = s;
        }
        if (dim == 3) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const double d2 = x2 - xs[4 * (J + t) + 2];
                sq[t] = sq[t] + d2 * d2;
            }
        }
#pragma unroll
        for (int t = 0; t < T; ++t) v[t] = sqrt(sq[t]);
        for (int e = 0; e < (phs - 1) / 2; ++e) {
#pragma unroll
            for (int t = 0; t < T; ++t) v[t] = v[t] * sq[t];
        }
#pragma unroll
        for (int t = 0; t < T; ++t)
            a[J + t] = i < k ? (i == J + t ? 0.0 : v[t]) : P[it * k + J + t];
    }

    __device__ __forceinline__ double entry(int j) const {
        if (j >= M) return 0.0;
        if (j >= k) return i < k ? P[(j - k) * k + ip] : 0.0;
        const double d0 = x0 - xs[j * 4], d1 = x1 - xs[j * 4 + 1];
        double s = 0.0;
        s = s + d0 * d0;
        s = s + d1 * d1;
        if (dim == 3) {
            const double d2 = x2 - xs[j * 4 + 2];
            s = s + d2 * d2;
        }
        const double rb = (i == j) ? 0.0 : rpow_d(s, phs);
        return i < k ? rb : P[it * k + j];
    }

    template <int J, int AW, int N>
    __device__ __forceinline__ void fill(double (&a)[N]) const {
        constexpr int T = J + 24 <= AW ? 4 : 2;  // (the row itself fills the registers by then)
        if (J + T <= k && phs >= 1) {
            points<J, T>(a);
        } else {
#pragma unroll
            for (int t = 0; t < T; ++t) a[J + t] = entry(J + t);
        }
        if constexpr (J + T < AW) fill<J + T, AW>(a);
    }
};

template <int NW, int AW>
__global__ __launch_bounds__(64 * NW, AW <= 32 ? 4 : AW <= 64 ? 3 : 2) void weights_wave_kernel(
    int dim, int phs, int m, const int* __restrict__ exps, SellView sv,
    const double* __restrict__ xyz, int npad, double* __restrict__ gx, double* __restrict__ gy,
    double* __restrict__ gz, double* __restrict__ lap, const int* __restrict__ rows,
    int* __restrict__ redo) {
    extern __shared__ double lds[];
    __shared__ double s_mm[NW][6];
    __shared__ int s_has[NW];
    __shared__ double s_sc[3], s_mn[3];
    __shared__ double s_cv[4];
    __shared__ int s_cp[4];
    __shared__ int s_e[WAVE_MAX_POLY * 3];
    __shared__ double s_zero[NW == 2 ? AW + 1 : 1];

    const int r = rows[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int k = sv.len[r];
    const int M = k + m;
    const int base = sell_base(sv.sptr, r);
    double* Y = lds;                          // forward-eliminated right-hand sides [M][4]
    double* U = lds + 4 * M;                  // rows of U (a strip of columns at a time)
    double* xs = lds;                         // assembly: scaled coordinates [k][4]
    double* P = lds + 4 * k;                  // assembly: monomial t at point j, P[t*k + j]

    for (int i = tid; i < m * dim; i += 64 * NW) s_e[i] = exps[i];
    // ---- shifting_scaling: thread t holds point t ----
    double xp[3] = {0.0, 0.0, 0.0};
    int has = tid < k;
    if (has) {
        const int cidx = sv.col[base + sell_off(tid)];
        for (int a = 0; a < dim; ++a) xp[a] = xyz[(size_t)a * npad + cidx];
    }
    for (int a = 0; a < dim; ++a) {
        double mn = xp[a], mx = xp[a];
        int h = has;
        ordered_minmax(mn, mx, h, lane);
        if (lane == 0) {
            s_mm[wv][2 * a] = mn;
            s_mm[wv][2 * a + 1] = mx;
            s_has[wv] = h;
        }
    }
    __syncthreads();
    if (tid < dim) {
        double mn = s_mm[0][2 * tid], mx = s_mm[0][2 * tid + 1];
        if constexpr (NW == 2) {
            if (s_has[1]) {
                const double mn1 = s_mm[1][2 * tid], mx1 = s_mm[1][2 * tid + 1];
                if (mn > mn1) mn = mn1;
                if (mx < mx1) mx = mx1;
            }
        }
        s_mn[tid] = mn;
        s_sc[tid] = mx - mn;
    }
    __syncthreads();
    if (has) {
        for (int a = 0; a < dim; ++a) {
            xp[a] = (xp[a] - s_mn[a]) / s_sc[a];
            xs[tid * 4 + a] = xp[a];
        }
        // x^e as 1*x*x*..., the first three powers at hand: a loop over each
        // exponent's multiplications cost 25k of the stencil's 250k cycles
        const double p0[2] = {xp[0] * xp[0], xp[0] * xp[0] * xp[0]};
        const double p1[2] = {xp[1] * xp[1], xp[1] * xp[1] * xp[1]};
        const double p2[2] = {xp[2] * xp[2], xp[2] * xp[2] * xp[2]};
        auto pw = [](double x, const double (&p)[2], int e) {
            double v = e <= 0 ? 1.0 : e == 1 ? x : e == 2 ? p[0] : p[1];
            for (int s = 3; s < e; ++s) v = v * x;
            return v;
        };
        for (int t = 0; t < m; ++t) {
            const int* e = s_e + t * dim;
            double v = pw(xp[0], p0, __builtin_amdgcn_readfirstlane(e[0]));
            v = v * pw(xp[1], p1, __builtin_amdgcn_readfirstlane(e[1]));
            if (dim == 3) v = v * pw(xp[2], p2, __builtin_amdgcn_readfirstlane(e[2]));
            P[t * k + tid] = v;
        }
    }
    __syncthreads();

    // ---- row i of A = [Phi P; P^T 0] and its right-hand sides ----
    const int i = tid;
    const bool valid = i < M;
    const int ip = i < k ? i : 0;                     // the row's point (stencil rows)
    const int it = (i >= k && i < M) ? i - k : 0;     // the row's monomial (polynomial rows)
    const double xi0 = xs[ip * 4], xi1 = xs[ip * 4 + 1], xi2 = xs[ip * 4 + 2];
    // (the right-hand sides first, while the row is not in registers yet)
    double rr[4] = {0.0, 0.0, 0.0, 0.0};
    if (valid) rhs_entries<true>(i < k, dim, phs, xs + 4 * ip, xs, s_sc, s_e + it * dim, rr);
    double a[AW + 1];
    // Four columns at a time, their square roots side by side: column by column
    // the chain of each left the vector units idle (50k cycles for 60 rows).
    const SaddleRow sr{xs, P, i, it, ip, k, M, dim, phs, xi0, xi1, xi2};
    sr.fill<0, AW>(a);
    a[AW] = 0.0;
    __syncthreads();  // the assembly tables are overwritten by U from here on

    // ---- LU with partial pivoting, right-looking ----
    if constexpr (NW == 2) {
        for (int j = tid; j <= AW; j += 64 * NW) s_zero[j] = 0.0;
        __syncthreads();
    }
    WaveLu<NW, AW> lu{a, rr, lds, s_zero, s_cv, s_cp, M, valid ? i : (1 << 20), lane, wv, valid};
    int c = 0;
    lu.template phase<AW>(c);
    if (lu.zero_pivot) {  // uniform: the whole wavefront saw the zero pivot
        if (tid == 0) redo[blockIdx.x] = 1;
        return;
    }
    __syncthreads();  // (the published rows are overwritten)
    if (valid) {
#pragma unroll
        for (int q = 0; q < 4; ++q) Y[4 * lu.pos + q] = rr[q];
    }

    // ---- back substitution (wavefront 0) ----
    constexpr int SPLIT = wave_split(NW, AW), NB = AW / 16;
    const int q = lane >> 4, l = lane & 15;
    BackRow row[NB];
    auto load = [&](int b, double d) {  // row 16*b + l, its diagonal entry d
        const int p = 16 * b + l;
        row[b].y = p < M ? Y[4 * p + q] : 0.0;
        row[b].d = p < M ? d : 1.0;
        row[b].rd = 1.0 / row[b].d;
        const double ad = fabs(row[b].d);
        row[b].dok = ad >= 0x1p-400 && ad <= 0x1p400;
    };
    const int H = M < SPLIT ? M : SPLIT;
    if constexpr (SPLIT < AW) {
        const int rs = (M - H) | 1;
        lu.store_right(U, H, rs);
        __syncthreads();
        auto at = [&](int p, int cc) { return p < M ? p * rs + cc - H : 0; };
        row[SPLIT / 16].d = 1.0;
        load(SPLIT / 16, U[at(SPLIT + l, SPLIT + l)]);
#pragma unroll
        for (int b = 0; b < SPLIT / 16; ++b) load(b, 1.0);
        back_blocks<NB - 1, SPLIT / 16>(row, U, M, l, at);
        __syncthreads();
    }
    lu.store_left(U, H);
    __syncthreads();
    if (wv != 0) return;
    {
        auto at = [&](int p, int cc) { return p <= cc ? p * H - p * (p - 1) / 2 + cc - p : 0; };
#pragma unroll
        for (int b = 0; b < SPLIT / 16; ++b) {
            const int p = 16 * b + l;
            const double y = row[b].y;
            load(b, p < H ? U[at(p, p)] : 1.0);
            if (SPLIT < AW) row[b].y = y;
        }
        back_blocks<SPLIT / 16 - 1, 0>(row, U, M, l, at);
    }
    double* out = q == 0 ? gx : q == 1 ? gy : q == 2 && dim == 3 ? gz : lap;
    if (q <= dim) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int p = 16 * b + l;
            if (p < k) out[(size_t)base + (size_t)sell_off(p)] = row[b].y;
        }
    }
}

// Entry (i, j) of the saddle-point matrix from the scaled coordinates, with the
// arithmetic of the FP64 assembly above.
__device__ __forceinline__ double saddle_entry(int i, int j, int k, int dim, int phs,
                                               const double* xs, const int* e) {
    if (i < k && j < k) {
        if (i == j) return 0.0;
        double s = 0.0;
        for (int a = 0; a < dim; ++a) {
            double d = xs[i * 3 + a] - xs[j * 3 + a];
            s = s + d * d;
        }
        return rpow_d(s, phs);
    }
    if (i >= k && j >= k) return 0.0;
    const int pt = (i < k) ? i : j;
    const int t = (i < k) ? j - k : i - k;
    double v = ipow_d(xs[pt * 3 + 0], e[t * dim + 0]);
    for (int a = 1; a < dim; ++a) v = v * ipow_d(xs[pt * 3 + a], e[t * dim + a]);
    return v;
}

// FP32 LU + FP64 iterative refinement.  The LU factors (FP32) and the FP64
// right-hand sides live in LDS; each refinement forms r = b - A x in FP64 with
// A's entries recomputed from the coordinates, solves the correction with the
// FP32 factors and adds it in FP64.  Stops once the correction reaches the
// FP64 floor; a stencil that has not converged after `max_ref` rounds is
// flagged for the FP64 kernel.
constexpr int MIX_THREADS = 256;  // four wavefronts per stencil (one: 8 per CU by LDS, 43 % slower)
__global__ __launch_bounds__(MIX_THREADS) void weights_mixed_kernel(
    int dim, int phs, int m, const int* __restrict__ exps, SellView sv,
    const double* __restrict__ xyz, int npad, double* __restrict__ gx, double* __restrict__ gy,
    double* __restrict__ gz, double* __restrict__ lap, const int* __restrict__ rows,
    int* __restrict__ flag, int max_ref) {
    extern __shared__ double lds[];
    __shared__ double s_mn[3], s_sc[3];
    __shared__ float s_bestf;
    __shared__ int s_piv, s_conv;
    __shared__ double s_red[2];
    __shared__ int s_e[WAVE_MAX_POLY * 3];
    const int r = rows[blockIdx.x];
    const int tid = threadIdx.x;
    const int k = sv.len[r];
    const int M = k + m;
    const int LDA = M + 1;
    const int nr = dim + 1;
    double* B = lds;                       // FP64 right-hand sides [M][4]
    double* X = B + M * 4;                 // FP64 solution [M][4]
    double* xs = X + M * 4;                // scaled coordinates [k][3]
    float* Af = (float*)(xs + k * 3);      // FP32 LU factors [M][LDA]
    float* W = Af + M * LDA;               // FP32 work [M][4]
    int* perm = (int*)(W + M * 4);         // row permutation [M]
    const int base = sell_base(sv.sptr, r);
    (void)s_bestf;

    for (int i = tid; i < m * dim; i += blockDim.x) s_e[i] = exps[i];
    for (int t = tid; t < k; t += blockDim.x) {
        const int c = sv.col[base + sell_off(t)];
        for (int a = 0; a < dim; ++a) xs[t * 3 + a] = xyz[(size_t)a * npad + c];
    }
    __syncthreads();
    if (tid < dim) {
        double mn = xs[tid], mx = xs[tid];
        for (int t = 0; t < k; ++t) {
            double v = xs[t * 3 + tid];
            if (mn > v) mn = v;
            if (mx < v) mx = v;
        }
        s_mn[tid] = mn;
        s_sc[tid] = mx - mn;
    }
    __syncthreads();
    for (int t = tid; t < k * dim; t += blockDim.x) {
        const int j = t / dim, a = t - j * dim;
        xs[j * 3 + a] = (xs[j * 3 + a] - s_mn[a]) / s_sc[a];
    }
    __syncthreads();
    for (int i = tid >> 6; i < M; i += MIX_THREADS / 64)
        for (int j = tid & 63; j < M; j += 64)
            Af[i * LDA + j] = (float)saddle_entry(i, j, k, dim, phs, xs, s_e);
    // FP64 right-hand sides (same formulas as the FP64 kernel)
    for (int i = tid; i < M; i += blockDim.x) {
        for (int q = 0; q < 4; ++q) B[i * 4 + q] = 0.0;
        rhs_entries<false>(i < k, dim, phs, xs + 3 * (i < k ? i : 0), xs, s_sc,
                    s_e + (i < k ? 0 : i - k) * dim, B + 4 * i);
        perm[i] = i;
    }
    __syncthreads();
    // FP32 LU with partial pivoting
    bool singular = false;
    for (int c = 0; c < M; ++c) {
        if (tid < 64) {
            float best = -1.0f;
            int bi = M;
            for (int i = c + tid; i < M; i += 64) {
                float v = fabsf(Af[i * LDA + c]);
                if (v > best) {
                    best = v;
                    bi = i;
                }
            }
            for (int off = 32; off > 0; off >>= 1) {
                float ob = __shfl_xor(best, off);
                int oi = __shfl_xor(bi, off);
                if (ob > best || (ob == best && oi < bi)) {
                    best = ob;
                    bi = oi;
                }
            }
            if (tid == 0) s_piv = bi;
        }
        __syncthreads();
        const int piv = s_piv;
        if (piv != c) {
            if (tid == 0) {
                const int tp = perm[c];
                perm[c] = perm[piv];
                perm[piv] = tp;
            }
            for (int j = tid; j < M; j += blockDim.x) {
                float t0 = Af[c * LDA + j];
                Af[c * LDA + j] = Af[piv * LDA + j];
                Af[piv * LDA + j] = t0;
            }
            __syncthreads();
        }
        const float d = Af[c * LDA + c];
        if (d == 0.0f) {
            singular = true;
            __syncthreads();
            continue;
        }
        for (int i = c + 1 + tid; i < M; i += blockDim.x) Af[i * LDA + c] = Af[i * LDA + c] / d;
        __syncthreads();
        // trailing update: the wavefronts take the rows in turn, the lanes the
        // columns (no index division; every entry sees the same single fma)
        for (int i = c + 1 + (tid >> 6); i < M; i += MIX_THREADS / 64) {
            const float l = Af[i * LDA + c];
            for (int j = c + 1 + (tid & 63); j < M; j += 64)
                Af[i * LDA + j] = fmaf(-l, Af[c * LDA + j], Af[i * LDA + j]);
        }
        __syncthreads();
    }
    // W (FP32) holds the current right-hand side; X accumulates in FP64
    for (int t = tid; t < M * 4; t += blockDim.x) {
        const int i = t >> 2, q = t & 3;
        W[t] = (float)B[perm[i] * 4 + q];
        X[t] = 0.0;
    }
    __syncthreads();
    int converged = 0;
    double dprev = 1e300;
    for (int it = 0; it <= max_ref && !singular; ++it) {
        // forward (unit L) and backward (U) substitution on the nr columns of W
        // (four columns per row, t = 4 i + q; column q >= nr is not used)
        for (int c = 0; c < M; ++c) {
            for (int t = tid; t < (M - c - 1) * 4; t += blockDim.x) {
                const int i = c + 1 + (t >> 2), q = t & 3;
                if (q < nr) W[i * 4 + q] = fmaf(-Af[i * LDA + c], W[c * 4 + q], W[i * 4 + q]);
            }
            __syncthreads();
        }
        for (int c = M - 1; c >= 0; --c) {
            if (tid < nr) W[c * 4 + tid] = W[c * 4 + tid] / Af[c * LDA + c];
            __syncthreads();
            for (int t = tid; t < c * 4; t += blockDim.x) {
                const int i = t >> 2, q = t & 3;
                if (q < nr) W[i * 4 + q] = fmaf(-Af[i * LDA + c], W[c * 4 + q], W[i * 4 + q]);
            }
            __syncthreads();
        }
        // x += dx; size of the correction relative to x
        if (tid == 0) {
            s_red[0] = 0.0;
            s_red[1] = 0.0;
        }
        __syncthreads();
        double dmax = 0.0, xmax = 0.0;
        for (int t = tid; t < M * 4; t += blockDim.x) {
            if ((t & 3) >= nr) continue;
            const double dx = (double)W[t];
            const double xn = X[t] + dx;
            X[t] = xn;
            dmax = fmax(dmax, fabs(dx));
            xmax = fmax(xmax, fabs(xn));
        }
        for (int off = 32; off > 0; off >>= 1) {
            dmax = fmax(dmax, __shfl_xor(dmax, off));
            xmax = fmax(xmax, __shfl_xor(xmax, off));
        }
        if ((tid & 63) == 0) {
            atomicMax((unsigned long long*)&s_red[0], (unsigned long long)__double_as_longlong(dmax));
            atomicMax((unsigned long long*)&s_red[1], (unsigned long long)__double_as_longlong(xmax));
        }
        __syncthreads();
        // converged: the correction is at the FP64 rounding floor (<= 1e-13 of x),
        // or it has stopped shrinking below 1e-11 of x (residual noise ~ cond * eps64)
        const double dcur = s_red[0], xcur = s_red[1];
        if (dcur <= 1e-13 * xcur || (it > 0 && dcur <= 1e-11 * xcur && dcur >= 0.5 * dprev)) {
            converged = 1;
            break;
        }
        if (it == max_ref || !(dcur == dcur)) break;
        dprev = dcur;
        // r = b - A x in FP64 (entries recomputed), permuted into W as FP32
        for (int i = tid; i < M; i += blockDim.x) {
            const int pi = perm[i];
            double acc[4] = {B[pi * 4 + 0], B[pi * 4 + 1], B[pi * 4 + 2], B[pi * 4 + 3]};
            for (int j = 0; j < M; ++j) {
                const double a = saddle_entry(pi, j, k, dim, phs, xs, s_e);
                if (a != 0.0)
                    for (int q = 0; q < 4; ++q) acc[q] = fma(-a, X[j * 4 + q], acc[q]);
            }
            for (int q = 0; q < 4; ++q) W[i * 4 + q] = (float)acc[q];
        }
        __syncthreads();
    }
    if (tid == 0) s_conv = converged;
    __syncthreads();
    if (!s_conv) {
        if (tid == 0) flag[r] = 1;
        return;
    }
    for (int t = tid; t < k; t += blockDim.x) {
        const size_t slot = (size_t)base + (size_t)sell_off(t);
        gx[slot] = X[t * 4 + 0];
        gy[slot] = X[t * 4 + 1];
        if (dim == 3) gz[slot] = X[t * 4 + 2];
        lap[slot] = X[t * 4 + dim];
    }
}

}  // namespace

size_t weights_mixed_lds(int max_len, int m) {
    const int M = max_len + m;
    return sizeof(double) * ((size_t)M * 8 + (size_t)max_len * 3) +
           sizeof(float) * ((size_t)M * (M + 1) + (size_t)M * 4) + sizeof(int) * M;
}

void launch_weights_mixed(hipStream_t s, int dim, int phs, int m, const int* exps_dev,
                          const SellView& sv, const double* xyz_soa, int npad, double* gx,
                          double* gy, double* gz, double* lap, const int* rows, int nrows,
                          int* flag, int max_len, int max_ref) {
    if (nrows == 0) return;
    if (m > WAVE_MAX_POLY || weights_mixed_lds(max_len, m) > WEIGHTS_LDS_MAX)
        throw std::runtime_error("launch_weights_mixed: system too large for the mixed kernel");
    const size_t lds = weights_mixed_lds(max_len, m);
    if (lds > 64 * 1024)
        MP_HIP(hipFuncSetAttribute((const void*)weights_mixed_kernel,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(weights_mixed_kernel, dim3(nrows), dim3(MIX_THREADS), lds, s, dim, phs, m, exps_dev,
                       sv, xyz_soa, npad, gx, gy, gz, lap, rows, flag, max_ref);
    MP_HIP(hipGetLastError());
}

void launch_weights_fp64(hipStream_t s, int dim, int phs, int m, const int* exps_dev,
                         const SellView& sv, const double* xyz_soa, int npad, double* gx,
                         double* gy, double* gz, double* lap, double* cond, int max_len,
                         const int* rows, int nrows, const int* only) {
    if (rows && nrows == 0) return;
    const int n = rows ? nrows : sv.nv;
    const int M = max_len + m;
    const size_t doubles = (size_t)M * (M + 1) + (size_t)M * 4 + (size_t)max_len * 3;
    const size_t lds = sizeof(double) * doubles;
    if (lds <= WEIGHTS_LDS_MAX) {
        if (lds > 64 * 1024)
            MP_HIP(hipFuncSetAttribute((const void*)weights_fp64_kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(weights_fp64_kernel, dim3(n), dim3(256), lds, s, dim, phs, m, exps_dev,
                           sv, xyz_soa, npad, gx, gy, gz, lap, cond, rows, only, 0,
                           (double*)nullptr, 0L);
        MP_HIP(hipGetLastError());
        return;
    }
    // systems too large for LDS (high polynomial degrees): a global work area
    // of `doubles` per block, in launches of at most 256 MiB of it
    const long stride = (long)((doubles + 31) & ~(size_t)31);
    const int chunk = (int)std::max<long>(1, std::min<long>(n, (256L << 20) / 8 / stride));
    DevBuf<double> work;
    work.alloc((size_t)chunk * (size_t)stride);
    for (int t0 = 0; t0 < n; t0 += chunk) {
        const int cnt = std::min(chunk, n - t0);
        hipLaunchKernelGGL(weights_fp64_kernel, dim3(cnt), dim3(256), 0, s, dim, phs, m, exps_dev,
                           sv, xyz_soa, npad, gx, gy, gz, lap, cond, rows, only, t0, work.p,
                           stride);
        MP_HIP(hipGetLastError());
    }
    MP_HIP(hipStreamSynchronize(s));  // (the work area is freed on return)
}


template <int NW, int AW>
void launch_wave(hipStream_t s, int dim, int phs, int m, const int* exps_dev, const SellView& sv,
                 const double* xyz_soa, int npad, double* gx, double* gy, double* gz, double* lap,
                 const int* rows, int nrows, int* redo) {
    if (nrows == 0) return;
    const size_t lds = sizeof(double) * (size_t)wave_lds_doubles<NW, AW>(m);
    if (lds > 64 * 1024)
        MP_HIP(hipFuncSetAttribute((const void*)weights_wave_kernel<NW, AW>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((weights_wave_kernel<NW, AW>), dim3(nrows), dim3(64 * NW), lds, s, dim,
                       phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, rows, redo);
    MP_HIP(hipGetLastError());
}

void launch_weights_fp64_rows(hipStream_t s, int dim, int phs, int m, const int* exps_dev,
                              const SellView& sv, const double* xyz_soa, int npad, double* gx,
                              double* gy, double* gz, double* lap, const std::vector<int>& rows,
                              const std::vector<int>& lens, DevBuf<int>& dev_rows) {
    static const int cls[WAVE_CLASSES] = {32, 48, 64, 80, 96};
    std::vector<int> bucket[WAVE_CLASSES + 1];
    int max_long = 0;
    for (size_t t = 0; t < rows.size(); ++t) {
        const int M = lens[t] + m;
        int b = 0;
        while (b < WAVE_CLASSES && M > cls[b]) ++b;
        if (m > WAVE_MAX_POLY) b = WAVE_CLASSES;  // (the register kernels' monomial table)
        bucket[b].push_back(rows[t]);
        if (b == WAVE_CLASSES) max_long = std::max(max_long, lens[t]);
    }
    std::vector<int> all;
    all.reserve(rows.size());
    int off[WAVE_CLASSES + 2];
    for (int b = 0; b <= WAVE_CLASSES; ++b) {
        off[b] = (int)all.size();
        all.insert(all.end(), bucket[b].begin(), bucket[b].end());
    }
    off[WAVE_CLASSES + 1] = (int)all.size();
    if (all.empty()) return;
    // the grouped row list, then one flag per row (set by a single-wavefront
    // stencil that met an exactly zero pivot)
    const size_t nall = all.size();
    dev_rows.alloc(2 * nall);
    MP_HIP(hipMemcpyAsync(dev_rows.p, all.data(), sizeof(int) * nall, hipMemcpyHostToDevice, s));
    MP_HIP(hipMemsetAsync(dev_rows.p + nall, 0, sizeof(int) * nall, s));
    auto n = [&](int b) { return off[b + 1] - off[b]; };
    const int* d = dev_rows.p;
    int* redo = dev_rows.p + nall;
    launch_wave<1, 32>(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, d + off[0],
                       n(0), redo + off[0]);
    launch_wave<1, 48>(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, d + off[1],
                       n(1), redo + off[1]);
    launch_wave<1, 64>(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, d + off[2],
                       n(2), redo + off[2]);
    launch_wave<2, 80>(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, d + off[3],
                       n(3), redo + off[3]);
    launch_wave<2, 96>(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, d + off[4],
                       n(4), redo + off[4]);
    // single-wavefront stencils with a zero pivot: the LDS kernel, which
    // follows the oracle through the singular column
    const int n1 = off[3] - off[0];
    if (n1 > 0)
        launch_weights_fp64(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, nullptr,
                            64 - m, d + off[0], n1, redo + off[0]);
    if (n(WAVE_CLASSES) > 0)
        launch_weights_fp64(s, dim, phs, m, exps_dev, sv, xyz_soa, npad, gx, gy, gz, lap, nullptr,
                            max_long, d + off[WAVE_CLASSES], n(WAVE_CLASSES));
}

}  // namespace mp
