// Reverse Cuthill-McKee order on the GPU (cuthill_mckee_ordering and
// reverse_cuthill_mckee_ordering, general_functions.cpp:807-879, as called by
// CLOUD::re_order_points_reverse_cuthill_mckee, cloud.cpp:315-331), level by
// level.  Sequentially, the queue takes each node in turn, claims its not yet
// visited stencil neighbours in stencil order and appends them sorted by
// (degree, index).  A node reached from level L is therefore claimed by the
// level-L node of lowest queue position whose stencil holds it, and level L+1
// is each level-L node's claimed neighbours, in queue order, sorted by (degree,
// index).  Per level:
//   claim   a wavefront per node: atomicMin of (queue position, entry) on every
//           unvisited column, so each column belongs to one stencil entry;
//   count   the node's columns that kept its claim;
//   scan    offsets of the nodes' groups, the next level's bounds;
//   place   a column's rank inside its group by comparing keys across the
//           wavefront; its queue position.
// The levels' bounds live on the device, so the host launches several levels
// between two looks at them.  A 250k-node cube (about 60 levels): 1.1 ms of kernels
// where one thread per node, a radix sort and a synchronisation per level took
// 5.9 ms of kernels and about 2 ms of gaps.
// Nodes the start cannot reach restart the search at the
// lowest-index unvisited node of minimum degree: while components are short,
// the device finds their roots itself between levels (see rcm_order).
// order[old] = new, reversed.
#include <algorithm>
#include <climits>
#include <stdexcept>
#include <string>
#include <vector>

#include "mp_internal.hpp"

namespace mp {

namespace {

// The search's progress: the current level is queue positions a .. b-1 (empty
// once its component is done); roots: components begun.
struct RcmState {
    int a, b, levels, roots;
};

// key of the lowest (degree, index) unvisited node, reduced into *best, when the
// current level is empty and nodes are left
__global__ __launch_bounds__(BLOCK) void k_rcm_start(const RcmState* s, int nv,
                                                     const int* __restrict__ rp,
                                                     const int* __restrict__ pos, int idx_bits,
                                                     unsigned long long* best) {
    if (s->a != s->b || s->b >= nv) return;
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    unsigned long long k = ~0ull;
    if (i < nv && pos[i] < 0)
        k = ((unsigned long long)(rp[i + 1] - rp[i]) << idx_bits) | (unsigned long long)i;
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long v = __shfl_xor(k, o);
        k = v < k ? v : k;
    }
    if ((threadIdx.x & 63) == 0 && k != ~0ull) atomicMin(best, k);
}

// The node k_rcm_start found becomes the next component's root (*best: ~0 when it
// did not run, and again afterwards).
__global__ void k_rcm_root(unsigned long long* best, unsigned long long mask,
                           int* __restrict__ numbering, int* __restrict__ pos, RcmState* s) {
    const unsigned long long k = *best;
    if (k == ~0ull) return;
    *best = ~0ull;
    const int v = (int)(k & mask), at = s->b;
    numbering[at] = v;
    pos[v] = at;
    s->a = at;
    s->b = at + 1;
    s->levels += 1;
    s->roots += 1;
}

// smallest entry whose column is outside 0 .. nv-1 (LLONG_MAX: none)
__global__ __launch_bounds__(BLOCK) void k_rcm_check(long nnz, int nv, const int* __restrict__ col,
                                                     unsigned long long* bad) {
    for (long e = (long)blockIdx.x * BLOCK + threadIdx.x; e < nnz; e += (long)gridDim.x * BLOCK)
        if (col[e] < 0 || col[e] >= nv) {
            atomicMin(bad, (unsigned long long)e);
            return;
        }
}

constexpr int RCM_WAVES = BLOCK / 64;
constexpr int RCM_BLOCKS = 2048;  // grid of the per-level kernels: 8192 nodes at a time
constexpr int RCM_FEW_BLOCKS = 256;  // and while components are short

// every stencil entry of the level's nodes claims its unvisited column
__global__ __launch_bounds__(BLOCK) void k_rcm_claim(const RcmState* s, const int* __restrict__ rp,
                                                     const int* __restrict__ col,
                                                     const int* __restrict__ numbering,
                                                     const int* __restrict__ pos,
                                                     unsigned long long* __restrict__ claim) {
    const int b = s->b, lane = threadIdx.x & 63;
    for (int t = s->a + (int)blockIdx.x * RCM_WAVES + (int)(threadIdx.x >> 6); t < b;
         t += (int)gridDim.x * RCM_WAVES) {
        const int v = numbering[t], e0 = rp[v], e1 = rp[v + 1];
        for (int e = e0 + lane; e < e1; e += 64) {
            const int c = col[e];
            if (pos[c] < 0)
                atomicMin(claim + c, ((unsigned long long)t << 32) | (unsigned)(e - e0));
        }
    }
}

// entry e (of queue position t's row from e0) holds an unvisited column it claimed
__device__ __forceinline__ bool rcm_owns(int c, int t, int k, const int* __restrict__ pos,
                                         const unsigned long long* __restrict__ claim) {
    return pos[c] < 0 && claim[c] == (((unsigned long long)t << 32) | (unsigned)k);
}

__global__ __launch_bounds__(BLOCK) void k_rcm_count(const RcmState* s, const int* __restrict__ rp,
                                                     const int* __restrict__ col,
                                                     const int* __restrict__ numbering,
                                                     const int* __restrict__ pos,
                                                     const unsigned long long* __restrict__ claim,
                                                     int* __restrict__ cnt) {
    const int a = s->a, b = s->b, lane = threadIdx.x & 63;
    for (int t = a + (int)blockIdx.x * RCM_WAVES + (int)(threadIdx.x >> 6); t < b;
         t += (int)gridDim.x * RCM_WAVES) {
        const int v = numbering[t], e0 = rp[v], e1 = rp[v + 1];
        int n = 0;
        for (int e = e0; e < e1; e += 64) {
            const bool own = e + lane < e1 && rcm_owns(col[e + lane], t, e + lane - e0, pos, claim);
            n += __popcll(__ballot(own));
        }
        if (lane == 0) cnt[t - a] = n;
    }
}

// cnt -> exclusive offsets over the level; the next level's bounds go to out
// (k_rcm_place still reads the current ones)
__global__ __launch_bounds__(1024) void k_rcm_scan(const RcmState* s, RcmState* out,
                                                   int* __restrict__ cnt) {
    __shared__ int wsum[16];
    const int n = s->b - s->a, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int carry = 0;
    for (int i0 = 0; i0 < n; i0 += 1024) {
        const int i = i0 + (int)threadIdx.x;
        const int v = i < n ? cnt[i] : 0;
        int x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == 63) wsum[wid] = x;
        __syncthreads();
        int before = carry, total = carry;
        for (int w = 0; w < 16; ++w) {
            before += w < wid ? wsum[w] : 0;
            total += wsum[w];
        }
        if (i < n) cnt[i] = before + x - v;
        carry = total;
        __syncthreads();
    }
    if (threadIdx.x == 0)
        *out = RcmState{s->b, s->b + carry, s->levels + (carry > 0 ? 1 : 0), s->roots};
}

// numbers each claimed column: its group's offset plus the columns of the
// group with a smaller (degree, index).  A row of more than MAX_STENCIL entries
// comes in that order already (comparing its columns pairwise would take its
// length squared): there it is the number of claimed columns in front.
__global__ __launch_bounds__(BLOCK) void k_rcm_place(const RcmState* s, const int* __restrict__ rp,
                                                     const int* __restrict__ col,
                                                     int* __restrict__ numbering,
                                                     int* __restrict__ pos,
                                                     const unsigned long long* __restrict__ claim,
                                                     const int* __restrict__ off, int idx_bits) {
    const int a = s->a, b = s->b, lane = threadIdx.x & 63;
    for (int t = a + (int)blockIdx.x * RCM_WAVES + (int)(threadIdx.x >> 6); t < b;
         t += (int)gridDim.x * RCM_WAVES) {
        const int v = numbering[t], e0 = rp[v], e1 = rp[v + 1];
        // (a column's claim stays its owner's after it is numbered, so the test
        // for the others reads the claim alone)
        auto mine = [&](int e, int& c) {
            c = e < e1 ? col[e] : 0;
            return e < e1 && claim[c] == (((unsigned long long)t << 32) | (unsigned)(e - e0));
        };
        if (e1 - e0 > MAX_STENCIL) {
            int at = b + off[t - a];
            for (int e = e0; e < e1; e += 64) {
                int c;
                const bool own = mine(e + lane, c);
                const unsigned long long m = __ballot(own);
                if (own) {
                    const int p = at + __popcll(m & ((1ull << lane) - 1ull));
                    numbering[p] = c;
                    pos[c] = p;
                }
                at += __popcll(m);
            }
            continue;
        }
        for (int e = e0; e < e1; e += 64) {
            int c;
            const bool own = mine(e + lane, c);
            const unsigned long long key =
                own ? ((unsigned long long)(rp[c + 1] - rp[c]) << idx_bits) | (unsigned)c : ~0ull;
            if (__ballot(own) == 0) continue;
            int rank = 0;
            for (int f = e0; f < e1; f += 64) {
                int d = c;
                bool other = own;
                unsigned long long k = key;
                if (f != e) {
                    other = mine(f + lane, d);
                    k = other ? ((unsigned long long)(rp[d + 1] - rp[d]) << idx_bits) | (unsigned)d
                              : ~0ull;
                }
                for (unsigned long long m = __ballot(other); m; m &= m - 1)
                    rank += __shfl(k, __ffsll(m) - 1) < key ? 1 : 0;
            }
            if (own) {
                const int at = b + off[t - a] + rank;
                numbering[at] = c;
                pos[c] = at;
            }
        }
    }
}

__global__ __launch_bounds__(BLOCK) void k_rcm_reverse(int nv, const int* __restrict__ numbering,
                                                       int* __restrict__ order) {
    const int p = blockIdx.x * BLOCK + threadIdx.x;
    if (p < nv) order[numbering[p]] = nv - 1 - p;
}

// pos = -1 (unvisited), claim = none
__global__ __launch_bounds__(BLOCK) void k_rcm_init(int nv, int* __restrict__ pos,
                                                    unsigned long long* __restrict__ claim,
                                                    RcmState* s, unsigned long long* best) {
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i < nv) {
        pos[i] = -1;
        claim[i] = ~0ull;
    }
    if (i == 0) {
        s[0] = s[1] = RcmState{0, 0, 0, 0};
        best[0] = best[1] = ~0ull;
    }
}

int bits_for(long v) {  // bits to hold 0..v
    int b = 1;
    while ((1L << b) <= v) ++b;
    return b;
}

}  // namespace

void rcm_order(hipStream_t st, int nv, const int* row_ptr, const int* col, int* order,
               int* levels_out) {
    if (nv <= 0) throw std::invalid_argument("rcm: nv must be positive");
    if (row_ptr[0] != 0) throw std::invalid_argument("rcm: row_ptr[0] must be 0");
    int max_deg = 0;
    for (int i = 0; i < nv; ++i) {
        if (row_ptr[i + 1] < row_ptr[i]) throw std::invalid_argument("rcm: row_ptr decreases");
        max_deg = std::max(max_deg, row_ptr[i + 1] - row_ptr[i]);
    }
    const long nnz = row_ptr[nv];
    const int idx_bits = bits_for(nv - 1);
    const int deg_bits = bits_for(max_deg);
    if (2 * idx_bits + deg_bits > 64)
        throw std::invalid_argument("rcm: graph too large for 64-bit sort keys");
    const unsigned long long mask = (1ull << idx_bits) - 1ull;
    // rows of more than MAX_STENCIL entries in (degree, index) order (the order
    // inside a row does not change the numbering; see k_rcm_place)
    std::vector<int> sorted;
    if (max_deg > MAX_STENCIL) {
        sorted.assign(col, col + nnz);
        for (int i = 0; i < nv; ++i) {
            int *c0 = sorted.data() + row_ptr[i], *c1 = sorted.data() + row_ptr[i + 1];
            if (c1 - c0 <= MAX_STENCIL) continue;
            // (a row with a bad column stays as it is for k_rcm_check)
            if (std::any_of(c0, c1, [nv](int c) { return c < 0 || c >= nv; })) continue;
            std::sort(c0, c1, [row_ptr](int x, int y) {
                const int dx = row_ptr[x + 1] - row_ptr[x], dy = row_ptr[y + 1] - row_ptr[y];
                return dx != dy ? dx < dy : x < y;
            });
        }
    }
    const int* const up_col = sorted.empty() ? col : sorted.data();

    DevBuf<int> drp, dcol, numbering, pos, cnt, dorder;
    DevBuf<unsigned long long> claim, best;  // best: [0] the start's key, [1] the column check
    DevBuf<RcmState> state;  // two: the current level and the next
    drp.alloc((size_t)nv + 1);
    dcol.alloc(std::max<long>(nnz, 1));
    numbering.alloc(nv);
    pos.alloc(nv);
    claim.alloc(nv);
    cnt.alloc(nv);
    dorder.alloc(nv);
    best.alloc(2);
    state.alloc(2);
    MP_HIP(hipMemcpyAsync(drp.p, row_ptr, sizeof(int) * (nv + 1), hipMemcpyHostToDevice, st));
    if (nnz > 0)
        MP_HIP(hipMemcpyAsync(dcol.p, up_col, sizeof(int) * nnz, hipMemcpyHostToDevice, st));
    const int nb = (nv + BLOCK - 1) / BLOCK;
    hipLaunchKernelGGL(k_rcm_init, dim3(nb), dim3(BLOCK), 0, st, nv, pos.p, claim.p, state.p,
                       best.p);
    hipLaunchKernelGGL(k_rcm_check, dim3(RCM_BLOCKS), dim3(BLOCK), 0, st, nnz, nv, dcol.p,
                       best.p + 1);
    MP_HIP(hipGetLastError());
    struct Polled {
        RcmState s;
        unsigned long long bad;
    };
    Polled* h = nullptr;
    MP_HIP(hipHostMalloc((void**)&h, sizeof(Polled), 0));
    try {
        MP_HIP(hipMemcpyAsync(&h->bad, best.p + 1, sizeof(h->bad), hipMemcpyDeviceToHost, st));
        MP_HIP(hipStreamSynchronize(st));
        if (h->bad != ~0ull)
            throw std::invalid_argument("rcm: column " + std::to_string(col[h->bad]) +
                                        " out of range");
        int cur = 0;
        auto root = [&]() {
            hipLaunchKernelGGL(k_rcm_start, dim3(nb), dim3(BLOCK), 0, st,
                               (const RcmState*)(state.p + cur), nv, drp.p, pos.p, idx_bits,
                               best.p);
            hipLaunchKernelGGL(k_rcm_root, dim3(1), dim3(1), 0, st, best.p, mask, numbering.p,
                               pos.p, state.p + cur);
        };
        h->s = RcmState{0, 0, 0, 0};
        // 16 levels between two looks: those past the component's last are
        // empty (four launches of 2 to 4 us each).  After a component of at most
        // 8 levels the device looks for a root in front of every level (two
        // launches more), for as long as components keep ending that soon: 4000
        // single nodes take 85 ms, 1000 cliques of 30 nodes 45, where a look for
        // every component took 980 and 260 ms.
        bool many = false;
        while (h->s.b < nv) {
            const RcmState before = h->s;
            if (!many && before.a == before.b) root();
            const dim3 grid(many ? RCM_FEW_BLOCKS : RCM_BLOCKS);
            for (int l = 0; l < 16; ++l) {
                if (many) root();
                RcmState *s = state.p + cur, *next = state.p + (cur ^ 1);
                hipLaunchKernelGGL(k_rcm_claim, grid, dim3(BLOCK), 0, st, s, drp.p, dcol.p,
                                   numbering.p, pos.p, claim.p);
                hipLaunchKernelGGL(k_rcm_count, grid, dim3(BLOCK), 0, st, s, drp.p, dcol.p,
                                   numbering.p, pos.p, claim.p, cnt.p);
                hipLaunchKernelGGL(k_rcm_scan, dim3(1), dim3(1024), 0, st, s, next, cnt.p);
                hipLaunchKernelGGL(k_rcm_place, grid, dim3(BLOCK), 0, st, s, drp.p, dcol.p,
                                   numbering.p, pos.p, claim.p, cnt.p, idx_bits);
                cur ^= 1;
            }
            MP_HIP(hipGetLastError());
            MP_HIP(hipMemcpyAsync(&h->s, state.p + cur, sizeof(RcmState), hipMemcpyDeviceToHost,
                                  st));
            MP_HIP(hipStreamSynchronize(st));
            many = h->s.roots - before.roots > 1 ||
                   (h->s.a == h->s.b && h->s.levels - before.levels <= 8);
        }
        hipLaunchKernelGGL(k_rcm_reverse, dim3(nb), dim3(BLOCK), 0, st, nv, numbering.p,
                           dorder.p);
        MP_HIP(hipGetLastError());
        MP_HIP(hipMemcpyAsync(order, dorder.p, sizeof(int) * nv, hipMemcpyDeviceToHost, st));
        MP_HIP(hipStreamSynchronize(st));
    } catch (...) {
        (void)hipHostFree(h);
        throw;
    }
    const int levels = h->s.levels;
    (void)hipHostFree(h);
    if (levels_out) *levels_out = levels;
}

}  // namespace mp
