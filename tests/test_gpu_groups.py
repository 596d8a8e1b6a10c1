"""Grouping of FD nodes for the projections: whatever list the nodes come in
(brick order, shuffled, far apart, with repeats) and whatever grid side they
are cut from, a node's bounds and moments are the same bits, and H v agrees
with the FP64 oracle (1e-12 FP64; 2e-6 with FP32 storage, the bound of one
FP32 rounding per value through H)."""
import numpy as np
import pytest

import helpers as H
from sqdft_amd.configs import smooth_veff
from sqdft_amd.sq import SpectralQuadrature

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed", "mixed_lanczos"])
@pytest.mark.parametrize("elem,n", [("al", 7), ("al", 9), ("lih", 13)])
def test_moments_do_not_depend_on_the_list(elem, n, prec):
    print(elem, n, prec, flush=True)
    S = (H.small_al if elem == "al" else H.small_lih)(n_cell=n)[0]
    veff = smooth_veff(S)
    sq = SpectralQuadrature(S, precision=prec)
    whole = sq.node_moments(veff, np.arange(S.nn))
    rng = np.random.Generator(np.random.PCG64(n))
    for nodes in (rng.permutation(S.nn)[: 3 * n], np.arange(0, S.nn, 2 * n + 1), np.array([5, 5, 0, S.nn - 1, 5])):
        part = sq.node_moments(veff, nodes)
        for k in ("chi", "zee", "mu", "iters"):
            assert np.array_equal(part[k], whole[k][nodes]), k


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("elem", ["al", "lih"])
def test_hsub_of_scattered_nodes(elem, prec, tol):
    print(elem, prec, flush=True)
    S, Rcut, T = (H.small_al if elem == "al" else H.small_lih)(n_cell=9)
    veff, o = smooth_veff(S), H.oracle_for(S, Rcut, T)
    rng = np.random.Generator(np.random.PCG64(3))
    nodes = np.concatenate([np.arange(11), rng.integers(0, S.nn, 6), [4, 4]])
    sq = SpectralQuadrature(S, precision=prec)
    v = rng.standard_normal((nodes.size, sq.M, sq.M, sq.M))
    hv = sq.HsubTimesVec(veff, nodes, v)
    for b, nd in enumerate(nodes):
        ref = o.hsub(veff, int(nd), v[b].reshape(-1))
        assert H.rel(hv[b].reshape(-1), ref) < tol


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("elem", ["al", "lih"])
def test_hsub_of_pairs_in_any_order(elem, prec):
    """Two nodes share a group up to one plane and several rows or columns
    apart, and either may come first; next to them, pairs too far away to join.
    Every product is the one that the node gives alone."""
    print(elem, prec, flush=True)
    S = (H.small_al if elem == "al" else H.small_lih)(n_cell=13)[0]
    n, veff, nodes, at = 13, smooth_veff(S), [], 0
    for dx, dy in [(0, 1), (0, 2), (1, 2), (0, 3), (0, 5), (0, 6), (3, 3), (6, 0), (-2, 2), (-3, 1)]:
        for dz in (0, 1):
            a = [3, 1, 5 * (at % 3)]
            b = [3 + dx, 1 + dy, a[2] + dz]
            at += 1
            nodes += [(p[2] * n + p[1]) * n + p[0] for p in ([b, a] if at % 4 < 3 else [a, b])]
    nodes = np.array(nodes)
    sq = SpectralQuadrature(S, precision=prec)
    rng = np.random.Generator(np.random.PCG64(8))
    v = rng.standard_normal((nodes.size, sq.M, sq.M, sq.M))
    hv = sq.HsubTimesVec(veff, nodes, v)
    for b, nd in enumerate(nodes):
        one = sq.HsubTimesVec(veff, nodes[b:b + 1], v[b:b + 1])
        assert np.array_equal(hv[b].reshape(-1), one.reshape(-1)), (b, nd)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("elem,n", [("al", 9), ("lih", 9)])
def test_shares_of_a_group_sum_alike(elem, n, prec):
    """The images of a group go to one, two or four workgroups by the number of
    groups in the call: the same nodes give the same bits in calls of 9 (four
    shares), 100 (two), 150 and 300 isolated nodes (one, two) and repeated."""
    print(elem, n, prec, flush=True)
    S = (H.small_al if elem == "al" else H.small_lih)(n_cell=n)[0]
    veff = smooth_veff(S)
    sq = SpectralQuadrature(S, precision=prec)
    rng = np.random.Generator(np.random.PCG64(21))
    # alternately from the lowest and the highest planes: groups of one node each
    lo, hi = rng.integers(0, n * n, 150), S.nn - 1 - rng.integers(0, n * n, 150)
    nodes = np.stack([lo, hi], axis=1).reshape(-1)
    v = rng.standard_normal((nodes.size, sq.M, sq.M, sq.M))
    whole = sq.HsubTimesVec(veff, nodes, v).reshape(nodes.size, -1)
    for cnt in (9, 100, 150):
        part = sq.HsubTimesVec(veff, nodes[:cnt], v[:cnt]).reshape(cnt, -1)
        assert np.array_equal(part, whole[:cnt]), cnt
