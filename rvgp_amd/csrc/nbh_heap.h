// Fibonacci-heap emulation of RVGP/lib/ptu_dijkstra.pyx:440-690 and the
// per-source truncated Dijkstra of pyx:361-394, shared by the neighbourhood
// kernels (nbh.hip) and the host build that runs the same
// code under AddressSanitizer / UndefinedBehaviorSanitizer
// (tests/sanitize/nbh_host.hip).  Every function compiles for both sides.
#ifndef RVGP_NBH_HEAP_H
#define RVGP_NBH_HEAP_H

#include <hip/hip_runtime.h>

namespace rvgp {

enum : int { kScanned = 0, kNotInHeap = 1, kInHeap = 2 };
constexpr int kMaxRank = 32;

// A heap node; HNode's links index a pool of any size, LNode's (24 bytes, for
// pools in LDS) one below 32768.  `last` is the rightmost child.
template <class Idx>
struct __align__(8) NodeOf {
    double val;
    int gidx;
    short rank, state;
    Idx parent, left, right, children, last;
};
using HNode = NodeOf<int>;

// LNode has no state: the wave's search keeps it in a mask.
struct __align__(8) LNode {
    double val;
    int gidx;
    short rank, parent, left, right, children, last;
};

// The root list is the sibling list holding min_node.  Its two ends are kept
// in head / tail, and every node knows its rightmost child, so appending a
// root or a child and finding the leftmost root are O(1) instead of walks
// over the list: the reference walks it (pyx:526-536, 642-660), but the walks
// only locate its ends, and the list itself -- every link, every order -- is
// the same.
template <class Node>
struct HeapOf {
    Node* N;
    int* roots;
    int min_node;
    int head, tail;
};
using Heap = HeapOf<HNode>;

template <class Node>
__host__ __device__ inline int leftmost_sibling(const Node* N, int a) {
    while (N[a].left != -1) a = N[a].left;
    return a;
}

// A root leaves the root list (pyx:542-560 where the parent is -1); its own
// links are the caller's to set.
template <class Node>
__host__ __device__ inline void root_unlink(HeapOf<Node>& h, int a, int left, int right) {
    if (a == h.head) h.head = right;
    if (a == h.tail) h.tail = left;
    if (left != -1) h.N[left].right = right;
    if (right != -1) h.N[right].left = left;
}

// A child leaves its parent (pyx:542-560).
template <class Node>
__host__ __device__ inline void child_remove(HeapOf<Node>& h, int a) {
    Node* N = h.N;
    const int p = N[a].parent, l = N[a].left, r = N[a].right;
    N[p].rank -= 1;
    N[p].children = l != -1 ? l : r;
    if (N[p].last == a) N[p].last = l;
    if (l != -1) N[l].right = r;
    if (r != -1) N[r].left = l;
    N[a].parent = -1;
}

// add_sibling(min_node, s) for the root list (pyx:526-536): s goes after
// the rightmost root; a root's parent is -1, so no rank changes.
template <class Node>
__host__ __device__ inline void root_append(HeapOf<Node>& h, int s) {
    Node* N = h.N;
    N[h.tail].right = s;
    N[s].left = h.tail;
    N[s].right = -1;
    h.tail = s;
}

// pyx:579-589, of a node without parent
template <class Node>
__host__ __device__ inline void insert_node(HeapOf<Node>& h, int a) {
    if (h.min_node != -1) {
        root_append(h, a);
        if (h.N[a].val < h.N[h.min_node].val) h.min_node = a;
    } else {
        h.N[a].left = h.N[a].right = -1;
        h.min_node = a;
        h.head = h.tail = a;
    }
}

template <class Node>
__host__ __device__ inline void decrease_val(HeapOf<Node>& h, int a, double v) {  // pyx:595-608
    Node* N = h.N;
    N[a].val = v;
    if (N[a].parent != -1 && N[N[a].parent].val >= v) {
        child_remove(h, a);
        insert_node(h, a);
    } else if (N[h.min_node].val > v) {
        h.min_node = a;
    }
}

// pyx:642-690 with the linking of pyx:614-636.  The reference clears
// roots_by_rank[0..100); ranks here are bounded by kMaxRank (checked), so
// clearing [0, kMaxRank) is equivalent.  The children of the minimum become
// roots as one splice of their list: its order is the one that appending them
// from the leftmost on gives.  Two linked roots have the same rank r, and the
// parent's is r + 1 after it, so ranks and values of the running root stay in
// registers.
template <class Node>
__host__ __device__ inline int remove_min(HeapOf<Node>& h, bool& ok) {
    Node* N = h.N;
    const int m = h.min_node;
    if (N[m].children != -1) {
        const int first = leftmost_sibling(N, N[m].children), last = N[m].last;
        for (int c = first; c != -1; c = N[c].right) N[c].parent = -1;
        N[h.tail].right = first;
        N[first].left = h.tail;
        h.tail = last;
        N[m].children = -1;
        N[m].rank = 0;
    }
    int t = h.head;  // leftmost_sibling(m)
    if (t == m) {
        t = N[m].right;
        if (t == -1) {
            h.min_node = -1;
            h.head = h.tail = -1;
            return m;
        }
    }
    root_unlink(h, m, N[m].left, N[m].right);
    int mn = t;
    double mv = N[t].val;
    for (int i = 0; i < kMaxRank; ++i) h.roots[i] = -1;
    while (t != -1) {
        int a = t, r = N[t].rank;
        double va = N[t].val;
        const int tr = N[t].right;
        if (va < mv) {
            mn = t;
            mv = va;
        }
        for (;;) {
            if (r >= kMaxRank) {
                ok = false;
                h.min_node = mn;
                return m;
            }
            const int ln = h.roots[r];
            if (ln == -1) {
                h.roots[r] = a;
                break;
            }
            h.roots[r] = -1;
            const double vl = N[ln].val;
            const Node na = N[a], nl = N[ln];
            const bool keep = va < vl || a == mn;
            const int par = keep ? a : ln, ch = keep ? ln : a;
            root_unlink(h, ch, keep ? nl.left : na.left, keep ? nl.right : na.right);
            const int pc = keep ? na.children : nl.children, pl = keep ? na.last : nl.last;
            N[ch].parent = par;  // add_child (pyx:507-520)
            N[ch].right = -1;
            if (pc != -1) {
                N[pl].right = ch;
                N[ch].left = pl;
            } else {
                N[par].children = ch;
                N[ch].left = -1;
            }
            N[par].last = ch;
            N[par].rank = ++r;
            a = par;
            va = keep ? va : vl;
        }
        t = tr;
    }
    h.min_node = mn;
    return m;
}

__host__ __device__ inline unsigned hash_of(int g, unsigned mask) {
    return ((unsigned)g * 2654435761u) & mask;
}


// One lane's private state: `pool` heap nodes, an open-addressing table of
// 2^m >= 2 pool entries (node id, pool slot), each slot's table position and
// the roots-by-rank array.  The table must hold (-1, -1) everywhere on entry;
// nbh_search leaves it that way.
struct NbhLane {
    HNode* N;
    int2* tab;
    int* hposv;
    int* roots;
    int pool;
    unsigned mask;
};

// The K+1 nodes popped by the truncated Dijkstra from `src` (pyx:361-394),
// written to out[0 .. *scanned).  Returns false when the search needs more
// than `pool` nodes (out is then incomplete).
__host__ __device__ inline bool nbh_search(const int* rowptr, const int* cols, const double* w,
                                           int K, int src, const NbhLane& L, int* out,
                                           int* scanned_out) {
    HNode* N = L.N;
    int2* tab = L.tab;
    const unsigned mask = L.mask;
    int used = 0;
    bool ok = true;
    auto new_node = [&](int g, unsigned hp) -> int {
        int s = used++;
        HNode& nd = N[s];
        nd.val = 0.0;
        nd.gidx = g;
        nd.rank = 0;
        nd.state = kNotInHeap;
        nd.parent = nd.left = nd.right = nd.children = nd.last = -1;
        L.hposv[s] = (int)hp;
        tab[hp] = make_int2(g, s);
        return s;
    };
    Heap h{N, L.roots, -1, -1, -1};
    {
        unsigned hp = hash_of(src, mask);
        while (tab[hp].x != -1) hp = (hp + 1) & mask;
        insert_node(h, new_node(src, hp));
    }
    int scanned = 0;
    while (h.min_node != -1 && scanned <= K) {
        int v = remove_min(h, ok);
        if (!ok) break;
        N[v].state = kScanned;
        out[scanned++] = N[v].gidx;
        if (scanned <= K) {
            const int j = N[v].gidx;
            const double vv = N[v].val;
            for (int e = rowptr[j]; e < rowptr[j + 1]; ++e) {
                const int c = cols[e];
                unsigned hp = hash_of(c, mask);
                int sc = -1;
                for (int2 te = tab[hp]; te.x != -1; te = tab[hp]) {
                    if (te.x == c) { sc = te.y; break; }
                    hp = (hp + 1) & mask;
                }
                if (sc != -1 && N[sc].state == kScanned) continue;
                const double nv = vv + w[e];
                if (sc == -1 || N[sc].state == kNotInHeap) {
                    if (sc == -1) {
                        if (used >= L.pool) { ok = false; break; }
                        sc = new_node(c, hp);
                    }
                    N[sc].state = kInHeap;
                    N[sc].val = nv;
                    insert_node(h, sc);
                } else if (N[sc].val > nv) {
                    decrease_val(h, sc, nv);
                }
            }
            if (!ok) break;
        }
    }
    for (int s = 0; s < used; ++s) tab[L.hposv[s]] = make_int2(-1, -1);
    *scanned_out = scanned;
    return ok;
}

}  // namespace rvgp

#endif  // RVGP_NBH_HEAP_H
