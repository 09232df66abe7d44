// Internal declarations shared by the HIP translation units of libmemphys_hip.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/memphys_hip.h"
#include "parallel.hpp"

namespace mp {

constexpr int SLICE = 64;       // rows per SELL slice (one wavefront)
constexpr int SGROUP = 4;       // neighbours of a row stored side by side in a slice
constexpr int SIGMA = 4096;     // rows per length-sorting window
constexpr int BLOCK = 256;      // threads per block of the row kernels
// Largest stencil (k) and monomial count (m) accepted: the reference's
// parameter range (poly_deg up to 15, parameters.cpp:84-88, 122-130) gives
// m = 136 in 2D; stencils of M = k + m above what LDS holds run from a global
// work area.  The register-resident weights kernels and the mixed kernel see
// m <= WAVE_MAX_POLY only (their stencils have M <= 96, and M >= 3m).
constexpr int MAX_STENCIL = 512;
constexpr int MAX_POLY = 136;
constexpr int WAVE_MAX_POLY = 35;
// dynamic LDS the weights kernel's per-stencil system may use (of 160 KB per CU,
// leaving room for its static arrays)
constexpr size_t WEIGHTS_LDS_MAX = 150 * 1024;

struct HipError {
    hipError_t code;
    const char* what;
};

#define MP_HIP(call)                                         \
    do {                                                     \
        hipError_t _e = (call);                              \
        if (_e != hipSuccess) throw ::mp::HipError{_e, #call}; \
    } while (0)

template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    void alloc(size_t count) {
        free();
        if (count == 0) count = 1;
        MP_HIP(hipMalloc((void**)&p, count * sizeof(T)));
        n = count;
    }
    void free() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    ~DevBuf() { free(); }
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), n(o.n) {
        o.p = nullptr;
        o.n = 0;
    }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) {
            free();
            p = o.p;
            n = o.n;
            o.p = nullptr;
            o.n = 0;
        }
        return *this;
    }
};

// Number of XCDs of the MI355X: the dispatcher hands workgroup b to XCD b % 8.
constexpr int NXCD = 8;

// XCD-aware block numbering: launch grid_xcd(G) blocks; block b works on
// logical block (b % 8) * ceil(G/8) + b / 8, so each XCD (and its L2) owns a
// contiguous range of rows.  Returns -1 for the padding blocks.
__host__ __device__ inline int grid_xcd(int g) { return ((g + NXCD - 1) / NXCD) * NXCD; }
__device__ __forceinline__ int xcd_block(int g, int block) {
    const int per = (g + NXCD - 1) / NXCD;
    const int lb = (block % NXCD) * per + block / NXCD;
    return lb < g ? lb : -1;
}
__device__ __forceinline__ int xcd_block(int g) { return xcd_block(g, (int)blockIdx.x); }

// SELL-64x4 slot numbering: slice s holds rows 64s..64s+63; neighbour j of
// slice row l sits at sptr[s] + 256*(j/4) + 4*l + j%4, so each lane reads its
// row's neighbours four at a time (one 16-byte load of columns or FP32
// values) and the wavefront still covers 256 consecutive slots per group.
// Slice widths are padded to a multiple of 4; padding slots hold the row's
// own column and value 0.
__host__ __device__ inline int sell_base(const int* sptr, int r) {
    return sptr[r >> 6] + ((r & 63) << 2);
}
__host__ __device__ inline int sell_off(int j) { return ((j >> 2) << 8) + (j & 3); }
__host__ __device__ inline int sell_width4(int w) { return (w + 3) & ~3; }

template <typename T>
struct Vec4 {
    typedef T type __attribute__((ext_vector_type(4)));
};

// Compressed columns: a slice whose columns fall into at most CW_COUNT
// windows of 2^CW_BITS consecutive ids stores each slot's column in 16 bits,
// (window << CW_BITS) | (column - base[window]), with the slice's window bases
// in cbase[CW_COUNT * s ...]; cbase[CW_COUNT * s] < 0 marks a slice that keeps
// its 32-bit columns.  The decode is exact, so either form gives the same sums.
constexpr int CW_BITS = 13;
constexpr int CW_COUNT = 8;

__device__ __forceinline__ int col_decode(uint32_t e, const int (&b)[CW_COUNT]) {
    const uint32_t w = e >> CW_BITS;
    const int t0 = (w & 1u) ? b[1] : b[0];
    const int t1 = (w & 1u) ? b[3] : b[2];
    const int t2 = (w & 1u) ? b[5] : b[4];
    const int t3 = (w & 1u) ? b[7] : b[6];
    const int u0 = (w & 2u) ? t1 : t0;
    const int u1 = (w & 2u) ? t3 : t2;
    return ((w & 4u) ? u1 : u0) + (int)(e & ((1u << CW_BITS) - 1u));
}

// Loads of the matrix: non-temporal (NT) keep the gathered vector in L2; the
// small systems' matrices stay in L2 themselves between two products.
template <bool NT, typename V>
__device__ __forceinline__ V load_stream(const V* p) {
    if constexpr (!NT || sizeof(V) > 16)
        return *p;
    else
        return __builtin_nontemporal_load(p);
}

// The neighbour loop of one slice row (groups of four slots from slot b0 +
// 4 lane, w4 groups): load(g) fetches group g's stored columns and decode()
// turns them into column ids.  A row's sum is four fma chains, chain p over the
// groups p, p + 4, ..., added as (0 + 1) + (2 + 3).  PARTS == 1: one wavefront
// forms all four; the stored columns and the values of U4 groups are requested
// before the first decode, so their loads overlap.  PARTS == 4: this wavefront
// forms chain `part` alone and returns it (two groups in flight); the caller
// adds the four.  Either way the row's sum has the same bits.
template <int PARTS, int U4, typename T, typename TM, typename LD, typename DC, typename FV,
          typename FX>
__device__ __forceinline__ T sell4_loop(int b0, int w4, int lane, int part,
                                        const TM* __restrict__ a, LD load, DC decode, FV fv,
                                        FX fx) {
    typedef typename Vec4<TM>::type v4;
    typedef decltype(load(0)) raw4;
    const v4* ap = reinterpret_cast<const v4*>(a + b0) + lane;
    // acc += the products of N groups g, g + step, ... (chain by chain)
    auto groups = [&](auto n, int g, int step, T* acc, int astep) {
        constexpr int N = decltype(n)::value;
        raw4 e[N];
        v4 v[N];
        T xv[4 * N];
#pragma unroll
        for (int u = 0; u < N; ++u) e[u] = load(g + u * step);
#pragma unroll
        for (int u = 0; u < N; ++u) v[u] = load_stream<PARTS == 1>(ap + (g + u * step) * SLICE);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const typename Vec4<int>::type c = decode(e[u]);
            xv[4 * u + 0] = fx(c.x);
            xv[4 * u + 1] = fx(c.y);
            xv[4 * u + 2] = fx(c.z);
            xv[4 * u + 3] = fx(c.w);
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            T& s = acc[u * astep];
            s = fma(fv(v[u].x), xv[4 * u + 0], s);
            s = fma(fv(v[u].y), xv[4 * u + 1], s);
            s = fma(fv(v[u].z), xv[4 * u + 2], s);
            s = fma(fv(v[u].w), xv[4 * u + 3], s);
        }
    };
    if constexpr (PARTS == 4) {
        T acc = (T)0;
        int g = part;
        for (; g + 4 < w4; g += 8) groups(std::integral_constant<int, 2>{}, g, 4, &acc, 0);
        if (g < w4) groups(std::integral_constant<int, 1>{}, g, 4, &acc, 0);
        return acc;
    } else {
        // U4 == 2 forms chains 0 and 1, then 2 and 3 (two accumulators live)
        static_assert(PARTS == 1 && (U4 == 2 || U4 == 4), "");
        T sum[4 / U4];
#pragma unroll
        for (int h = 0; h < 4; h += U4) {
            T acc[U4];
#pragma unroll
            for (int u = 0; u < U4; ++u) acc[u] = (T)0;
            int g = h;
            for (; g + U4 <= w4; g += 4) groups(std::integral_constant<int, U4>{}, g, 1, acc, 1);
#pragma unroll
            for (int u = 0; u + 1 < U4; ++u)
                if (g + u < w4) groups(std::integral_constant<int, 1>{}, g + u, 1, acc + u, 1);
            if constexpr (U4 == 4)
                sum[0] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            else
                sum[h / 2] = acc[0] + acc[1];
        }
        if constexpr (U4 == 4)
            return sum[0];
        else
            return sum[0] + sum[1];
    }
}

// Where a slice's slots start, its groups, and its column windows (base[0] < 0:
// 32-bit columns).  A slice past the matrix has no groups.
struct SellHead {
    int b0, w4;
    int base[CW_COUNT];
};

// Sum over the neighbours of one slice row of fv(value) * fx(column) (PARTS == 4:
// chain `part` of it; see sell4_loop): the slice of head h, lane = slice row.  The
// four neighbours of a group come in one vector load of columns (16-bit
// compressed ones when col16 is given and the slice has them) and one of
// values; U4 groups are loaded before their gathers.  With PARTS == 1 columns
// and values up to 4 bytes use non-temporal loads so the gathered vector stays
// cached; FP64 values (32 bytes a lane, fetched as two 16-byte halves) use ordinary loads,
// which keep the line in cache between the halves.
template <int PARTS, int U4, typename T, typename TM, typename FV, typename FX>
__device__ __forceinline__ T sell4_accumulate(const SellHead& h, const int* __restrict__ col,
                                              const uint16_t* __restrict__ col16,
                                              const TM* __restrict__ a, int lane, int part,
                                              FV fv, FX fx) {
    typedef typename Vec4<int>::type c4;
    typedef typename Vec4<uint16_t>::type e4;
    if (h.base[0] >= 0) {
        const e4* ep = reinterpret_cast<const e4*>(col16 + h.b0) + lane;
        return sell4_loop<PARTS, U4, T>(
            h.b0, h.w4, lane, part, a, [&](int g) { return load_stream<PARTS == 1>(ep + g * SLICE); },
            [&](e4 e) {
                c4 c;
                c.x = col_decode(e.x, h.base);
                c.y = col_decode(e.y, h.base);
                c.z = col_decode(e.z, h.base);
                c.w = col_decode(e.w, h.base);
                return c;
            },
            fv, fx);
    }
    const c4* cp = reinterpret_cast<const c4*>(col + h.b0) + lane;
    return sell4_loop<PARTS, U4, T>(
        h.b0, h.w4, lane, part, a, [&](int g) { return load_stream<PARTS == 1>(cp + g * SLICE); },
        [](c4 c) { return c; }, fv, fx);
}

// Where a SELL-64x4 matrix keeps its slots' columns: 32-bit, compressed to 16
// bits where a slice allows (col16, cbase; may be null), and, for large
// matrices, per block of BLOCK rows: uptr[b] .. uptr[b+1]-1 index the block's
// distinct columns ucol (ascending), loc holds each slot's place among them,
// max_u their largest number (0: not built).
struct Slots {
    int nslices = 0;
    const int* sptr = nullptr;
    const int* col = nullptr;
    const uint16_t* col16 = nullptr;
    const int* cbase = nullptr;
    const int* uptr = nullptr;
    const int* ucol = nullptr;
    const uint16_t* loc = nullptr;
    int max_u = 0;
};

// The shapes of a product's blocks (WS):
//   1   BLOCK threads over BLOCK rows: a wavefront per slice, four chains each;
//   2   as 1, with the block's distinct gathered entries staged in LDS first
//       (dynamic LDS: max_u of them);
//   4   BLOCK threads over one slice: a wavefront per chain;
//   16  4 * BLOCK threads over BLOCK rows: a wavefront per chain.
// Shape 2 is for large systems: a CU serves a gather of 64 entries from L2 in
// about 50 cycles, and a row block of a compact cluster reads each of its
// distinct columns (4-6 per row of 42) about nine times; gathered once, in
// ascending order, and read back from LDS, the product streams its matrix.
// One against staged: 1M-node cube, GMRES product 66.8 and 53.1 us (5.3 TB/s),
// level-0 residual 58.9 and 42.5, T_0 35 and 24, FP64 residual 126 and 92; 64 2D
// cavities of 665k nodes 31.5, 26.6, 15.5, 58 and 26.5, 21.3, 12.8, 47 us.
// The wide shapes (4, 16) are for systems whose slices leave SIMDs idle: the row's
// serial chain of loads is a quarter as long, and (4) the gathers, which a CU
// serves one wavefront at a time, spread over four times the CUs.
template <int WS>
constexpr int WS_THREADS = WS == 16 ? 4 * BLOCK : BLOCK;
template <int WS>
constexpr int WS_ROWS = WS == 4 ? SLICE : BLOCK;

// This wavefront's slice and chain in logical block lb.
template <int WS>
__device__ __forceinline__ int ws_slice(int lb) {
    const int wid = (int)(threadIdx.x >> 6);
    return __builtin_amdgcn_readfirstlane(WS == 4 ? lb : lb * (BLOCK / SLICE) + (wid & 3));
}
template <int WS>
__device__ __forceinline__ int ws_part() {
    const int wid = (int)(threadIdx.x >> 6);
    return __builtin_amdgcn_readfirstlane(WS == 4 ? wid : wid >> 2);
}
// This thread's row in logical block lb; past every row for the threads beyond
// the block's rows.
template <int WS>
__device__ __forceinline__ int block_row(int lb) {
    return (int)threadIdx.x < WS_ROWS<WS> ? lb * WS_ROWS<WS> + (int)threadIdx.x : INT_MAX;
}

__device__ __forceinline__ SellHead sell4_head(int nslices, const int* __restrict__ sptr,
                                               const uint16_t* __restrict__ col16,
                                               const int* __restrict__ cbase, int s) {
    SellHead h{0, 0, {-1, 0, 0, 0, 0, 0, 0, 0}};
    if (s < nslices) {
        h.b0 = sptr[s];
        h.w4 = (sptr[s + 1] - h.b0) >> 8;
        if (col16 != nullptr)
#pragma unroll
            for (int k = 0; k < CW_COUNT; ++k) h.base[k] = cbase[CW_COUNT * s + k];
    }
    return h;
}

// The four chains of a block's rows, one from each wavefront, added up: row t
// of the block to the threads of wavefront t / 64 and those that share its rows.
template <int WS, typename T>
__device__ __forceinline__ T add_chains(T acc, int part) {
    __shared__ T red[4][WS_ROWS<WS>];
    const int t = (int)(threadIdx.x & (WS_ROWS<WS> - 1));
    red[part][t] = acc;
    __syncthreads();
    return (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
}

// The row sums of one block (logical block lb): row block_row<WS>(lb) to its
// thread (zero past nslices); every thread must call.
template <int WS, int U4, typename T, typename TM, typename FV, typename FX>
__device__ __forceinline__ T sell4_block(const Slots& m, const TM* __restrict__ a, int lb, FV fv,
                                         FX fx) {
    const int lane = (int)(threadIdx.x & 63);
    if constexpr (WS == 2) {
        typedef decltype(fx(0)) TX;
        typedef typename Vec4<uint16_t>::type e4;
        typedef typename Vec4<int>::type c4;
        extern __shared__ __align__(16) char stage_lds[];
        TX* xs = reinterpret_cast<TX*>(stage_lds);
        const int s = ws_slice<1>(lb);
        const int b0 = s < m.nslices ? m.sptr[s] : 0;
        const int w4 = s < m.nslices ? (m.sptr[s + 1] - b0) >> 8 : 0;
        const int u0 = m.uptr[lb], nu = m.uptr[lb + 1] - u0;
        for (int t = (int)threadIdx.x; t < nu; t += 4 * BLOCK) {
            int c[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (t + q * BLOCK < nu) c[q] = m.ucol[u0 + t + q * BLOCK];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (t + q * BLOCK < nu) xs[t + q * BLOCK] = fx(c[q]);
        }
        __syncthreads();
        const e4* ep = reinterpret_cast<const e4*>(m.loc + b0) + lane;
        return sell4_loop<1, U4, T>(
            b0, w4, lane, 0, a, [&](int g) { return load_stream<true>(ep + g * SLICE); },
            [](e4 e) { return c4{e.x, e.y, e.z, e.w}; }, fv, [xs](int i) { return (T)xs[i]; });
    } else {
        const SellHead h = sell4_head(m.nslices, m.sptr, m.col16, m.cbase, ws_slice<WS>(lb));
        const int part = ws_part<WS>();
        T acc = sell4_accumulate<(WS == 1 ? 1 : 4), U4, T>(
            h, m.col, m.col16, a, lane, part, fv, [&](int c) { return (T)fx(c); });
        if constexpr (WS != 1) acc = add_chains<WS>(acc, part);
        return acc;
    }
}

// sell4_block<4> for gathered entries fin(raw), raw = pre(column) loaded from
// the vectors: the columns, values and raw entries of the chain's first two
// groups are requested before mid() runs, which may hold barriers and returns
// whether to go on (the same on every thread), so mid's latency and theirs
// overlap.  ok receives mid's answer.
template <typename T, typename TM, typename PRE, typename MID, typename FIN>
__device__ __forceinline__ T sell4_block_early(const Slots& m, const TM* __restrict__ a, int lb,
                                               PRE pre, MID mid, FIN fin, bool& ok) {
    typedef typename Vec4<TM>::type v4;
    typedef typename Vec4<int>::type c4;
    typedef typename Vec4<uint16_t>::type e4;
    typedef decltype(pre(0)) raw;
    const SellHead h = sell4_head(m.nslices, m.sptr, m.col16, m.cbase, ws_slice<4>(lb));
    const int lane = (int)(threadIdx.x & 63), part = ws_part<4>();
    const v4* ap = reinterpret_cast<const v4*>(a + h.b0) + lane;
    auto columns = [&](int g) {
        c4 c;
        if (h.base[0] >= 0) {
            const e4 e = (reinterpret_cast<const e4*>(m.col16 + h.b0) + lane)[g * SLICE];
            c.x = col_decode(e.x, h.base);
            c.y = col_decode(e.y, h.base);
            c.z = col_decode(e.z, h.base);
            c.w = col_decode(e.w, h.base);
        } else {
            c = (reinterpret_cast<const c4*>(m.col + h.b0) + lane)[g * SLICE];
        }
        return c;
    };
    T acc = (T)0;
    auto add = [&](v4 v, raw r0, raw r1, raw r2, raw r3) {
        acc = fma((T)v.x, fin(r0), acc);
        acc = fma((T)v.y, fin(r1), acc);
        acc = fma((T)v.z, fin(r2), acc);
        acc = fma((T)v.w, fin(r3), acc);
    };
    v4 v[2];
    raw r[2][4];
    c4 c[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (part + 4 * u < h.w4) {
            c[u] = columns(part + 4 * u);
            v[u] = ap[(part + 4 * u) * SLICE];
        }
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (part + 4 * u < h.w4) {
            r[u][0] = pre(c[u].x);
            r[u][1] = pre(c[u].y);
            r[u][2] = pre(c[u].z);
            r[u][3] = pre(c[u].w);
        }
    ok = mid();
    if (!ok) return (T)0;
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (part + 4 * u < h.w4) add(v[u], r[u][0], r[u][1], r[u][2], r[u][3]);
    for (int g = part + 8; g < h.w4; g += 4) {
        const c4 cc = columns(g);
        const v4 vv = ap[g * SLICE];
        add(vv, pre(cc.x), pre(cc.y), pre(cc.z), pre(cc.w));
    }
    return add_chains<4>(acc, part);
}

// Blocks of BLOCK rows up to which a product runs with a wavefront per chain.
// Shapes 1, 16 and 4: level-0 residual of a 64k-node cube (249 blocks) 11.7, 9.3
// and 6.9 us, FP64 product of a 110k-node cube (414 blocks) 18.2, 16.0 and 13.6.
// Whole iterations with a wavefront per chain (and the fused launches that go
// with it) against staged entries, us:
//                    FP64 Jacobi BiCGSTAB   mixed multigrid   FP64 multigrid
//   3D  249 blocks      34.3    38.2           53.9   61.4       57.3   65.0
//   3D  430             45.7    50.1           74.4   75.9       78.3   81.0
//   3D  648             59.3    60.4           87.4   85.0       90.9   91.3
//   3D  842             74.2    68.6           99.7   94.4      104.2  102.5
//   2D  265             27.9    30.8           63.8   64.1       57.8   62.2
//   2D  426             37.5    38.1           63.7   62.9       62.1   66.4
//   2D  625             47.5    47.1           74.5   68.4       72.9   72.1
//   2D  723             52.2    49.1           75.1   68.7       75.8   74.2
// The line lies where most of them cross (the 2D mixed multigrid would cross at
// about 430 blocks).
constexpr int SPLIT_MAX_BLOCKS = 640;

// SELL-64x4 view of the stencil set in device order.
struct SellView {
    int nv;            // real rows
    int nslices;
    const int* sptr;   // [nslices+1] first slot of each slice
    const int* col;    // [slots] device column ids
    const int* len;    // [nslices*64] row lengths (0 on ghost rows)
    const uint16_t* col16 = nullptr;  // [slots] compressed column ids (or null)
    const int* cbase = nullptr;       // [nslices*CW_COUNT] window bases
    const int* uptr = nullptr;        // distinct columns per row block (see Slots; or null)
    const int* ucol = nullptr;
    const uint16_t* loc = nullptr;
    int max_u = 0;
    long nuniq = 0;     // entries of ucol
    double reuse = 0;   // slots per entry of ucol
    __host__ __device__ Slots slots() const { return Slots{nslices, sptr, col, col16, cbase, uptr, ucol, loc, max_u}; }
};

// The predictor, right-hand side and corrector read staged entries: large clouds
// whose row blocks' distinct columns are listed (see Slots), when DIM vectors of
// them fit 64 KB of LDS (the limit without an attribute) and a staged entry
// serves at least 1.25 slots; the gathers of one entry per weight otherwise
// bound these kernels.  1M-node cube (reuse 9), gathered and staged: predictor
// 460 (plus 15 for the interleaved copy it gathers from) and 323 us, right-hand
// side 296 and 198, corrector 275 and 241.  At the LDS limit, 600k 2D rows of 20
// and 32 entries, 4,092 and 2,952 columns in the largest block, reuse 1.27 and
// 2.8: 123, 84, 89 and 114, 87, 70 us; 174, 126, 117 and 130, 92, 86.  600k rows
// of 12 and 16 entries whose columns lie anywhere, reuse 1.0: 81, 47, 55 and 96,
// 75, 51; 106, 67, 76 and 127, 102, 71.
template <int DIM>
bool staged_steps(const SellView& sv) {
    return sv.max_u > 0 && DIM * sv.max_u <= 8192 && sv.reuse >= 1.25;
}

// Host: the compressed columns of slots sptr/col (see CW_BITS above): c16 per
// slot, cb CW_COUNT window bases per slice (-1: the slice keeps 32-bit columns).
void compress_columns(const std::vector<int>& sptr, const std::vector<int>& col, int nslices,
                      std::vector<uint16_t>& c16, std::vector<int>& cb);

// Host: the distinct columns of every block of BLOCK rows and each slot's place
// among them (see Slots); false when a block has more than STAGE_MAX (48 KB of
// FP64 entries), which the LDS form is not for.  Up to there it is the faster
// one for the products, whatever the reuse and also when a single block sets
// every block's LDS.  600k rows, FP64, FP32 operator in BiCGSTAB and in GMRES,
// gathered and staged: 32 entries, 5,892 columns in the largest block, reuse
// 1.4: 83, 68, 49 and 55, 50, 41 us; reuse 22 with one block of 5,869: 42, 38, 33
// and 37, 30, 31; 20 entries anywhere (5,049, reuse 1.0): 68, 65, 60 and 62, 57,
// 48.
constexpr int STAGE_MAX = 6144;
bool stage_columns(const std::vector<int>& sptr, const std::vector<int>& col, int nslices,
                   std::vector<int>& uptr, std::vector<int>& ucol, std::vector<uint16_t>& loc,
                   int& max_u);

// Device-side Krylov scalars (FP64) of one system.  Written only by the
// single-block finishing kernels, read by every block of the following kernels.
struct KScalars {
    double rho, rho_old, alpha, omega, beta;
    double r0sq, bb, rr, tol2, eps2, tol_rel;
    double red[4];  // results of the last residual reduction
    // 0 running, 1 converged, 2 iteration cap, 3 restart needed, 4 zero
    // right-hand side, 5 breakdown / non-finite, 6 not part of this solve
    int done;
    int iter, maxit, restarts;
    // fused iterations: 1 when the last iteration's r.r and r0.r still wait in
    // the partial sums; which of the two buffers holds p and v
    int pending, par;
};

// One independent system of a batch: real rows [row0, row0 + nv), its border
// unknown (full-Neumann Lagrange multiplier) at row row0 + nv when border != 0,
// and the row blocks [blk0, blk0 + nblk) of BLOCK rows it owns.  Systems start
// on block boundaries, so a block never mixes two systems.
struct Seg {
    int row0, nv, blk0, nblk, border;
};

struct SegView {
    int nseg, nrows;    // systems; rows of all systems incl. padding (multiple of BLOCK)
    const Seg* seg;     // [nseg]
    const int* bseg;    // [nrows / BLOCK] system of each row block
    Seg one;            // the system, when there is only one: it comes with the
                        // kernel's arguments, two dependent loads (about 1 us
                        // of a small system's kernel) sooner
};
#ifdef __HIPCC__
// System of logical block lb (block-uniform scalar load), and its rows.
__device__ __forceinline__ int block_seg(const SegView& sg, int lb) {
    return sg.nseg == 1 ? 0 : __builtin_amdgcn_readfirstlane(sg.bseg[lb]);
}
__device__ __forceinline__ Seg seg_at(const SegView& sg, int q) {
    Seg s = sg.one;
    if (sg.nseg != 1) s = sg.seg[q];
    return s;
}
#endif

// Per-system controls of one Krylov run (uploaded before it starts).
struct SegCtl {
    int active, maxit;
    double tol_rel;
};

// ---- launchers (defined in the .hip files) ----
// rows == nullptr: every row; otherwise the listed device rows.
// FP64 weights of the device rows `rows` (stencil lengths `lens`): the
// register-resident kernel for systems of M = k + m <= 96 (one or two
// wavefronts per stencil), the LDS kernel beyond.  dev_rows receives the
// grouped row list and must stay allocated until the launches complete.
constexpr int WAVE_CLASSES = 5;
void launch_weights_fp64_rows(hipStream_t s, int dim, int phs, int m, const int* exps_dev,
                              const SellView& sv, const double* xyz_soa, int npad, double* gx,
                              double* gy, double* gz, double* lap, const std::vector<int>& rows,
                              const std::vector<int>& lens, DevBuf<int>& dev_rows);
void launch_weights_fp64(hipStream_t s, int dim, int phs, int m, const int* exps_dev,
                         const SellView& sv, const double* xyz_soa, int npad, double* gx,
                         double* gy, double* gz, double* lap, double* cond, int max_len,
                         const int* rows = nullptr, int nrows = 0, const int* only = nullptr);
// Dynamic LDS of the mixed kernel for stencils of up to max_len points.
size_t weights_mixed_lds(int max_len, int m);
// FP32 LU + FP64 refinement for the listed rows; flag[r] = 1 where it did not converge.
void launch_weights_mixed(hipStream_t s, int dim, int phs, int m, const int* exps_dev,
                          const SellView& sv, const double* xyz_soa, int npad, double* gx,
                          double* gy, double* gz, double* lap, const int* rows, int nrows,
                          int* flag, int max_len, int max_ref);

template <int DIM>
void launch_predictor(hipStream_t s, const SellView& sv, const double* gx, const double* gy,
                      const double* gz, const double* lap, const double* u, const double* v,
                      const double* w, double* uh, double* vh, double* wh, double* S_new,
                      const double* S_oo, int npad, double rho, double mu, double dt, int euler,
                      double* upk, double* uhpk, const int* bprob = nullptr,
                      const double* prm = nullptr, const double* force = nullptr);
// upk, uhpk: the velocity before and after the predictor interleaved per node
// (2 doubles per node in 2D, 4 in 3D: u, v, w, 0); the predictor packs u, v, w
// into upk for its gathers and writes uhpk beside uh, vh, wh for the
// right-hand side's gathers.
template <int DIM>
void launch_ppe_rhs(hipStream_t s, const SellView& sv, const double* gx, const double* gy,
                    const double* gz, const double* uh, const double* vh, const double* wh,
                    const double* uhpk, const double* u, const double* v, const double* w,
                    const double* p_old,
                    const uint8_t* bnd, const uint8_t* pdir, const double* normal_soa,
                    int npad, double rho, double dt, double* b, const int* bprob = nullptr,
                    const double* prm = nullptr);
template <int DIM>
void launch_corrector(hipStream_t s, const SellView& sv, const double* gx, const double* gy,
                      const double* gz, const double* p, const double* uh, const double* vh,
                      const double* wh, double* un, double* vn, double* wn, int npad, double rho,
                      double dt, const int* bprob = nullptr, const double* prm = nullptr);
template <int DIM>
void launch_boundary_fix(hipStream_t s, const SellView& sv, const int* brows, int nb,
                         const double* gx, const double* gy, const double* gz,
                         const double* normal_soa, int npad, const uint8_t* pdir,
                         const uint8_t* udir, const uint8_t* vdir, const uint8_t* wdir,
                         const double* u_old, const double* v_old, const double* w_old,
                         double* un, double* vn, double* wn);
void launch_spmv(hipStream_t s, const SellView& sv, const double* val, const double* x, double* y);
template <int DIM>
void launch_divergence(hipStream_t s, const SellView& sv, const double* gx, const double* gy,
                       const double* gz, const double* u, const double* v, const double* w,
                       const uint8_t* bnd, double* partial, int nblocks);

// Pressure operator in SELL slots: value arrays from the stencil weights.
void launch_build_operator(hipStream_t s, const SellView& sv, int dim, const double* gx,
                           const double* gy, const double* gz, const double* lap,
                           const double* normal_soa, int npad, const uint8_t* bnd,
                           const uint8_t* dir, double unsteady, double conv, double diff,
                           double* aval, double* diag);

// Largest-magnitude eigenvalue of a stencil operator (k_eig.hip); returns the
// Arnoldi restarts used.
// kNN stencils of host points into host CSR (row_ptr is filled from the
// stencil sizes); throws std::invalid_argument on bad sizes.
void knn_stencils(hipStream_t st, int nv, int dim, const double* xyz, const uint8_t* boundary,
                  const int* k_per_node, int* row_ptr, int* col);

// Reverse Cuthill-McKee order of a host CSR graph (order[old] = new); the
// number of BFS levels goes to *levels (may be null).
void rcm_order(hipStream_t st, int nv, const int* row_ptr, const int* col, int* order,
               int* levels);

int largest_eigenvalue(hipStream_t s, const SellView& sv, const double* val, int m, double tol,
                       int max_restarts, double* re, double* im);

// Krylov building blocks (k_krylov.hip).
void launch_fill(hipStream_t s, double* x, double v, int n);
void launch_copy(hipStream_t s, double* dst, const double* src, int n);

// Projection guess (k_project.hip): rings of PROJ_MAX stored pressures and
// their products with the pressure operator (vectors of ld doubles each); the
// device record holds the newest slot, the entries held and the last
// coefficients.
constexpr int PROJ_MAX = 24;
struct ProjState {
    int head;
    int count;
    double beta[PROJ_MAX];
};
size_t proj_partial_size();
// out = the combination of the newest k stored pressures (k <= PROJ_MAX, at
// most the entries held) with the smallest residual against b, over n rows
void launch_proj_guess(hipStream_t s, int k, int n, const double* hp, const double* hw, size_t ld,
                       ProjState* ps, const double* b, double* partial, double* out);
// stores p and A p = b - r as the newest entry
void launch_proj_store(hipStream_t s, int n, const double* p, const double* b, const double* r,
                       double* hp, double* hw, size_t ld, ProjState* ps);
void launch_proj_reset(hipStream_t s, ProjState* ps);

}  // namespace mp
