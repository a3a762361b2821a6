"""Locality renumbering of graph nodes for the block SpMM.

Points arrive in arbitrary order (the synthetic generators draw them
uniformly at random), so the block columns of a block row are scattered over
the whole operator and every gathered X row misses the caches.  Before the
eigensolve the nodes are renumbered along a Morton (Z-order) curve of their
leading principal coordinates: neighbours on the manifold get nearby
indices, consecutive block rows share most of their neighbours, and the
X rows a workgroup gathers stay resident in L2.

The permuted operator P A P^T has the same spectrum; eigenvector block rows
are mapped back through the permutation when the eigensolver writes its
output (rvgp_evecs_finish).  Node identity is never
renumbered anywhere else (the heap neighbourhoods, whose tie-breaking
depends on node order, run on the original numbering).
"""
import torch

from . import _lib

BOX_DIMS = 6  # box coordinates per point (blocks.h)


class SpatialOrder:
    """The points X (n, D) along a Morton curve of their top min(D, dims)
    principal coordinates (own_axes: of their own coordinates, D <= dims):
    perm (new position -> old node), and the coordinates the curve was made
    from, which bound distances from below."""

    def __init__(self, X, dims=BOX_DIMS, own_axes=False):
        P = min(X.shape[1], dims)
        self.X, self.P = X, P
        self.Y, self.kept = (X, None) if own_axes else _principal(X, P)
        self.lo, self.hi = torch.aminmax(self.Y, dim=0)
        keys = torch.empty(X.shape[0], dtype=torch.int64, device=X.device)
        _lib.call("rvgp_morton_keys", _lib.ptr(self.Y), self.Y.stride(0), X.shape[0], P,
                  _lib.ptr(self.lo), _lib.ptr(self.hi), _lib.ptr(keys), _lib.stream())
        self.perm = torch.sort(keys, stable=True).indices

    def blocks(self, transposed):
        """The points' spatial blocks (rvgp_blocks) as one byte tensor."""
        n, D = self.X.shape
        size = _lib.lib().rvgp_blocks_bytes(n, D, int(transposed))
        out = torch.empty(size, dtype=torch.uint8, device=self.X.device)
        _lib.call("rvgp_blocks", _lib.ptr(self.X), n, D, _lib.ptr(self.Y), self.Y.stride(0), self.P,
                  _lib.ptr(self.lo), _lib.ptr(self.hi), _lib.ptr(self.perm), int(transposed),
                  _lib.ptr(out), size, _lib.stream())
        return out

    def prunes(self, blocks, scalar):
        """(float(scalar), whether a neighbour search can skip most of the
        blocks), in one trip to the host.  It can where the box coordinates
        hold nearly all of the distances and the boxes are small against the
        points' range: a 3-torus in R^32 (n = 12,000, k = 20) keeps 0.999 of
        the variance and its boxes span 0.39 of the range on average (1.5
        against the plain scan's 1.9 ms); 20,000 Gaussian points in R^32 keep
        0.2, nothing is skipped and the plain scan is twice as fast (2.8
        against 5.4 ms)."""
        n = self.X.shape[0]
        nb = -(-n // 64)
        box = blocks[256:256 + 64 * nb].view(torch.float32).reshape(nb, 2, 8)
        span = (box[:, 1, :self.P] - box[:, 0, :self.P]).mean(0).max().double() / 2.0
        kept = torch.ones_like(span) if self.kept is None else self.kept
        v, kept, span = torch.stack([scalar.double(), kept, span]).tolist()
        return v, kept >= 0.9 and span <= 0.5


def _principal(X, P):
    """The top-P principal coordinates of the points, and the share of the
    total variance they keep (device scalar)."""
    from . import dense
    Xc = (X - X.mean(0, keepdim=True)).contiguous()
    C = dense.gemm_sym(Xc, Xc)
    w, V = dense.syev(C)
    return dense.gemm(Xc, V[:, -P:].contiguous()), w[-P:].sum() / w.sum()


def morton_perm(X, max_dims=6):
    """Permutation (new position -> old node) sorting nodes by the Morton
    code of their top-P principal coordinates (P = min(D, max_dims))."""
    return SpatialOrder(X, max_dims).perm


def bsr_permutation(rowptr, cols, perm):
    """The structure of P A P^T for a block-CSR pattern (rowptr, cols) and
    perm[new] = old block row: (new rowptr int32, new cols int32, order) with
    order[e] = the stored block that lands at position e.  Operators on one
    graph (the scalar and the connection Laplacian) share it."""
    dev = rowptr.device
    nb = rowptr.numel() - 1
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(nb, device=dev, dtype=perm.dtype)
    rp = rowptr.long()
    lens = rp[1:] - rp[:-1]
    rows = torch.repeat_interleave(torch.arange(nb, device=dev), lens)
    new_r = inv[rows]
    new_c = inv[cols.long()]
    order = torch.sort(new_r * nb + new_c, stable=True).indices
    new_rp = torch.zeros(nb + 1, dtype=torch.int64, device=dev)
    new_rp[1:] = torch.cumsum(lens[perm], 0)
    return new_rp.to(torch.int32), new_c[order].to(torch.int32), order


def permute_bsr(A, perm, plan=None):
    """B = P A P^T for a BSR operator; perm[new] = old block row.  plan: the
    result of bsr_permutation for A's pattern, when already computed."""
    from .sparse import BSR
    rp, cols, order = plan if plan is not None else bsr_permutation(A.rowptr, A.cols, perm)
    bb = A.b * A.b
    v64 = A.vals64.reshape(-1, bb)[order].reshape(-1).contiguous()
    v32 = None if A.vals32 is None else A.vals32.reshape(-1, bb)[order].reshape(-1).contiguous()
    return BSR(rp, cols, v64, v32, A.b)
