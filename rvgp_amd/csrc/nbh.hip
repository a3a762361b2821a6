// a3 (part 1)  Geodesic neighbourhoods: the truncated Dijkstra of
// RVGP/lib/ptu_dijkstra.pyx:361-394 driven by the Fibonacci heap of
// pyx:440-690.
//
// Which K+1 nodes form a neighbourhood is decided by the heap's pop order
// among equal hop distances, so the heap is emulated operation for
// operation: the same sibling-list splices, the same linking order, the same
// choice of the new minimum.  Instead of the reference's N heap nodes per
// source (re-initialised N times, an O(N^2) total), a search keeps a private
// pool of only the nodes it touches; node identity (the reference compares
// pointers) becomes pool-slot identity.  A wavefront owns one source with the
// pool in LDS; a search that outgrows the largest LDS pool is redone by one
// lane with a pool in memory, its nodes found through a hash table.
#include "common.h"
#include "nbh_heap.h"

namespace rvgp {

// One wavefront per source, a pool of P nodes.  The search is one chain of
// dependent heap steps, so its time is the latency of the heap's storage: LDS
// here, where a lane per source with the pool in memory also paid for 64
// diverging searches and for clearing its hash table.  Lane 0 runs the heap;
// the lanes look up a pop's edges together (hash table in LDS), and only those
// that insert or decrease go to lane 0, in their order.  26 bytes a node and
// 2 table entries: 32 wavefronts a CU at P = 128, 21 at 256, 10 at 512.
// K = 15, k = 10 on a surface: 1950 -> 176 us at n = 5000, 5.5 -> 2.5 ms at
// 100000; K = 30, k = 20 on a 3-torus, n = 100000: 20.9 -> 8.9 ms; K = 100 at
// n = 5000 (P = 512): 23.7 -> 1.5 ms.
template <int P>
__global__ __launch_bounds__(64) void geo_nbh_wave_kernel(const int* __restrict__ rowptr,
                                                          const int* __restrict__ cols,
                                                          const double* __restrict__ w, int n, int K,
                                                          int* __restrict__ nbh,
                                                          const int* __restrict__ src_list,
                                                          int* __restrict__ ovf_list,
                                                          int* __restrict__ status) {
    constexpr unsigned kMask = 2 * P - 1;
    __shared__ LNode N[P];
    __shared__ short tab[2 * P];  // slot or -1, open addressing by node id
    __shared__ int roots[kMaxRank];
    const int lane = threadIdx.x;
    const int nsrc = src_list != nullptr ? src_list[0] : n;
    for (int si = blockIdx.x; si < nsrc; si += gridDim.x) {
        const int src = src_list != nullptr ? src_list[1 + si] : si;
        int* out = nbh + (size_t)src * (K + 1);
        for (int q = lane; q < P; q += 64) reinterpret_cast<int*>(tab)[q] = -1;
        __syncthreads();
        // the heap's scalars are lane 0's
        HeapOf<LNode> h{N, roots, -1, -1, -1};
        int used = 0, good = 1;
        auto put = [&](int c, double v, unsigned hp) {
            LNode& nd = N[used];
            nd.val = v;
            nd.gidx = c;
            nd.rank = 0;
            nd.parent = nd.children = nd.last = -1;
            tab[hp] = (short)used;
            insert_node(h, used++);
        };
        if (lane == 0) put(src, 0.0, hash_of(src, kMask));
        int scanned = 0;
        while (scanned <= K && __builtin_amdgcn_readfirstlane(h.min_node) != -1) {
            int j = 0;
            double vv = 0.0;
            if (lane == 0) {
                bool o = true;
                const int v = remove_min(h, o);
                good = o;
                j = N[v].gidx;
                vv = N[v].val;
                N[v].val = -HUGE_VAL;  // scanned: above no distance, so never touched again
                if (o) out[scanned] = j;
            }
            if (!__builtin_amdgcn_readfirstlane(good)) break;
            j = __builtin_amdgcn_readfirstlane(j);
            vv = bcast(vv, 0);
            if (++scanned > K) break;
            const int e1 = rowptr[j + 1];
            for (int e0 = rowptr[j]; e0 < e1; e0 += 64) {
                const bool in = e0 + lane < e1;
                const int c = in ? cols[e0 + lane] : 0;
                const double nv = vv + (in ? w[e0 + lane] : 0.0);
                unsigned hp = hash_of(c, kMask);
                int slot = -1;
                bool act = false;
                __syncthreads();  // lane 0's writes
                if (in) {
                    while ((slot = tab[hp]) != -1 && N[slot].gidx != c) hp = (hp + 1) & kMask;
                    act = slot == -1 || N[slot].val > nv;
                }
                for (unsigned long long m = __ballot(act); m != 0; m &= m - 1) {
                    const int l = __builtin_ctzll(m);
                    const int cl = __builtin_amdgcn_readlane(c, l);
                    const double vl = bcast(nv, l);
                    unsigned hl = __builtin_amdgcn_readlane((int)hp, l);
                    if (lane == 0 && good) {
                        // again: an earlier edge may have taken the place, or be its twin
                        int s;
                        while ((s = tab[hl]) != -1 && N[s].gidx != cl) hl = (hl + 1) & kMask;
                        if (s != -1) {
                            if (N[s].val > vl) decrease_val(h, s, vl);
                        } else if (used < P) {
                            put(cl, vl, hl);
                        } else {
                            good = 0;
                        }
                    }
                }
                if (!__builtin_amdgcn_readfirstlane(good)) break;
            }
            if (!__builtin_amdgcn_readfirstlane(good)) break;
        }
        if (lane == 0) {
            if (!good) {
                if (ovf_list != nullptr) ovf_list[1 + atomicAdd(&ovf_list[0], 1)] = src;
                else atomicMax(status, RVGP_ST_POOL_OVERFLOW);
            } else if (scanned <= K) {
                atomicMax(status, RVGP_ST_SHORT_COMPONENT);
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void geo_nbh_kernel(const int* __restrict__ rowptr,
                                                      const int* __restrict__ cols,
                                                      const double* __restrict__ w, int n, int K,
                                                      int batch, int pool, int hsize,
                                                      size_t lane_bytes, int* __restrict__ nbh,
                                                      char* __restrict__ ws,
                                                      const int* __restrict__ src_list,
                                                      int* __restrict__ status) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nsrc = src_list[0];  // sources src_list[1 .. nsrc]
    if (t >= batch || t >= nsrc) return;
    char* base = ws + (size_t)t * lane_bytes;
    NbhLane L;
    L.N = reinterpret_cast<HNode*>(base);
    // hash table entries (node id, pool slot) side by side: one probe, one line
    L.tab = reinterpret_cast<int2*>(L.N + pool);
    L.hposv = reinterpret_cast<int*>(L.tab + hsize);  // table position of each slot
    L.roots = L.hposv + pool;
    L.pool = pool;
    L.mask = (unsigned)hsize - 1u;
    for (int q = 0; q < hsize; ++q) L.tab[q] = make_int2(-1, -1);
    const int Kp1 = K + 1;

    for (int si = t; si < nsrc; si += batch) {
        const int src = src_list[1 + si];
        int scanned = 0;
        const bool ok = nbh_search(rowptr, cols, w, K, src, L, nbh + (size_t)src * Kp1, &scanned);
        if (!ok) {
            atomicMax(status, RVGP_ST_POOL_OVERFLOW);
            return;
        }
        if (scanned < Kp1) atomicMax(status, RVGP_ST_SHORT_COMPONENT);
    }
}

static int next_pow2(int v) {
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

static size_t lane_bytes_for(int pool) {
    const int hsize = next_pow2(2 * pool);
    size_t b = sizeof(HNode) * (size_t)pool + sizeof(int2) * (size_t)hsize +
               sizeof(int) * ((size_t)pool + kMaxRank);
    return (b + 255) & ~(size_t)255;
}

__global__ void nbh_clear_count_kernel(int* __restrict__ a, int* __restrict__ b) {
    if (threadIdx.x == 0 && a != nullptr) a[0] = 0;
    if (threadIdx.x == 0 && b != nullptr) b[0] = 0;
}

// Every source first with an LDS pool for the usual search, those that
// outgrow it (a list) with the largest LDS pool, what is left with the
// worst-case pool 1 + K * max_degree in memory by kNbhBigLanes lanes; a pass
// whose pool holds the worst case is the last.  All run the same heap
// operations, so which one finishes a source does not change its
// neighbourhood.  On k-nearest-neighbour graphs with K = 1.5 k a search
// touches 3 K nodes on a surface, 4 K to 6 K (7 K at most) on a 3-torus: the
// first pool is the smallest that holds 7 K.
constexpr int kNbhPool = 512;
constexpr int kNbhBigLanes = 2048;
constexpr int kNbhGrid = 16384;

static int nbh_first_pool(int K) { return 7 * (long long)K <= 128 ? 128 : 7 * (long long)K <= 256 ? 256 : kNbhPool; }

// Workspace: kNbhPool-node states of `batch` lanes (of which the first list
// takes the front), worst-case states of b2 lanes, the second list.
static void nbh_plan(int n, int batch, int pool, int& p1, int& b2, size_t& o2, size_t& o3,
                     size_t& total) {
    p1 = pool < kNbhPool ? pool : kNbhPool;
    b2 = batch < kNbhBigLanes ? batch : kNbhBigLanes;
    const size_t a = lane_bytes_for(p1) * (size_t)batch;
    const size_t b = p1 < pool ? lane_bytes_for(pool) * (size_t)b2 : 0;
    const size_t c = p1 < pool ? sizeof(int) * ((size_t)n + 1) : 0;
    o2 = a;
    o3 = a + b;
    total = a + b + ((c + 255) & ~(size_t)255);
}

}  // namespace rvgp

using namespace rvgp;

extern "C" size_t rvgp_geo_nbh_ws_bytes(int n, int batch, int pool) {
    if (n < 1 || batch < 1 || pool < 1) return 0;
    int p1, b2;
    size_t o2, o3, total;
    nbh_plan(n, batch, pool, p1, b2, o2, o3, total);
    return total;
}

extern "C" int rvgp_geo_nbh(const int* rowptr, const int* cols, const double* w, int n, int K,
                            int batch, int pool, int* nbh, void* ws, size_t ws_bytes, int* status,
                            void* stream) {
    RVGP_CHECK_ARG(n >= 1 && K >= 0, "rvgp_geo_nbh: need n >= 1, K >= 0");
    RVGP_CHECK_ARG(K < n, "Geodesic neighborhood size must be less than the total number of samples");
    RVGP_CHECK_ARG(batch >= 1 && pool >= K + 1, "rvgp_geo_nbh: bad batch/pool");
    RVGP_CHECK_ARG(ws_bytes >= rvgp_geo_nbh_ws_bytes(n, batch, pool),
                   "rvgp_geo_nbh: workspace too small");
    int p1, b2;
    size_t o2, o3, total;
    nbh_plan(n, batch, pool, p1, b2, o2, o3, total);
    char* base = static_cast<char*>(ws);
    hipStream_t st = as_stream(stream);
    const int grid = n < kNbhGrid ? n : kNbhGrid;
    const int first = nbh_first_pool(K);
    // a smaller pool first where its list of leftovers has room (or none can be)
    const bool fits = pool <= first;
    const bool small = first < kNbhPool && (fits || sizeof(int) * ((size_t)n + 1) <= o2);
    int* ovf1 = small && !fits ? reinterpret_cast<int*>(base) : nullptr;
    int* ovf2 = p1 < pool ? reinterpret_cast<int*>(base + o3) : nullptr;
    if (ovf1 != nullptr || ovf2 != nullptr) {
        hipLaunchKernelGGL(nbh_clear_count_kernel, dim3(1), dim3(64), 0, st, ovf1, ovf2);
        RVGP_LAUNCH_CHECK();
    }
    if (small) {
        const auto kern = first == 128 ? geo_nbh_wave_kernel<128> : geo_nbh_wave_kernel<256>;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(64), 0, st, rowptr, cols, w, n, K, nbh, nullptr, ovf1,
                           status);
        RVGP_LAUNCH_CHECK();
    }
    if (!small || !fits) {
        hipLaunchKernelGGL(geo_nbh_wave_kernel<kNbhPool>, dim3(grid), dim3(64), 0, st, rowptr, cols, w,
                           n, K, nbh, ovf1, ovf2, status);
        RVGP_LAUNCH_CHECK();
    }
    if (ovf2 != nullptr) {
        const int l2 = b2 < n ? b2 : n;
        hipLaunchKernelGGL(geo_nbh_kernel, dim3(cdiv(l2, 256)), dim3(256), 0, st, rowptr, cols, w, n, K,
                           l2, pool, next_pow2(2 * pool), lane_bytes_for(pool), nbh, base + o2, ovf2,
                           status);
        RVGP_LAUNCH_CHECK();
    }
    return RVGP_OK;
}
