"""Projections where their usual walk does not fit: the systems are chosen by what
they make of the LDS and of the register slots, not as materials.  A block of
nodes that share a group and single ones against the FP64 oracle: H v at 1e-12
(2e-6 with FP32 storage, one FP32 rounding per value through H), Lanczos bounds
and moments at 1e-10, and the block bit for bit what its nodes give alone."""
import os

import numpy as np
import pytest

import helpers as H
from sqdft_amd.configs import smooth_veff
from sqdft_amd.sq import SpectralQuadrature
from sqdft_amd.system import AtomType, System

pytestmark = pytest.mark.gpu


def system(elem, n, h, nloc, frac, npl=8):
    """Atoms at frac (fractions of the cell) on an n^3 grid with cubes of 2 nloc + 1."""
    sym, Z, lloc = {"al": ("Al", 3, 1), "li": ("Li", 1, 0)}[elem]
    xyz = np.asarray(frac) * n * h
    types = [AtomType(sym, Z, lloc, os.path.join(H.PSD, f"psd_{sym}.pot"), xyz)]
    Rcut = (nloc - 0.5) * h
    return System.build(n=n, L_box=n * h, types=types, Rcut=Rcut, npl=npl, T=58000.0, h=h), Rcut, 58000.0


def scattered(natom, seed):
    return np.random.Generator(np.random.PCG64(seed)).uniform(0.0, 1.0, (natom, 3))


def on_faces(n, left, right, middle, x0, x1, hi, seed):
    """left and right atoms on the grid planes x0 and x1, middle ones between."""
    rng = np.random.Generator(np.random.PCG64(seed))
    p = rng.uniform(1.0, hi - 1.0, (left + right + middle, 3))
    p[:left, 0], p[left:left + right, 0] = x0, x1
    return p / n


def list_length(S, nodes):
    """Images with projectors whose box meets the cube of any of the nodes."""
    n, im = S.n, S.images()
    ti = [S.type_info(t) for t in range(S.info["n_typ"])]
    R = S.info["nloc"] + np.array([t["nlocc"] for t in ti])[im["type"]]
    has = np.array([t["nproj"] > 0 for t in ti])[im["type"]]
    hit = np.zeros(has.size, dtype=bool)
    for nd in nodes:
        r = np.array([nd % n, (nd // n) % n, nd // (n * n)])
        hit |= np.all(np.abs(im["nn"] - r) <= R[:, None], axis=1)
    return int(np.sum(hit & has))


def slots(S, nodes, planes, waves):
    """Register slots a walk of the nodes' images takes: image li of the z-sorted list
    is wave li mod waves', and holds a slot from the slab where it enters the union of
    the cubes to the one where it leaves."""
    n, im, nloc = S.n, S.images(), S.info["nloc"]
    c = S.type_info(0)["nlocc"]
    r = np.array([[nd % n, (nd // n) % n, nd // (n * n)] for nd in nodes])
    lo, hi = r.min(axis=0) - nloc, r.max(axis=0) + nloc
    z = np.sort(im["nn"][np.all((im["nn"] + c >= lo) & (im["nn"] - c <= hi), axis=1), 2])
    enter, leave = np.maximum(z - c, lo[2]) // planes, np.minimum(z + c, hi[2]) // planes
    return max(int(np.sum(leave[w:i:waves] >= enter[i])) + 1 for i in range(z.size) for w in [i % waves])


def block(n, x, y, z, dx=4, dy=2):
    return np.array([(z * n + y + j) * n + x + i for j in range(dy) for i in range(dx)], dtype=np.int32)


def check(S, Rcut, T, nodes, precs=("fp64", "mixed"), moments=True):
    veff, o = smooth_veff(S), H.oracle_for(S, Rcut, T)
    for prec in precs:
        sq = SpectralQuadrature(S, precision=prec)
        v = np.random.Generator(np.random.PCG64(2)).standard_normal((nodes.size, sq.M ** 3))
        hv = sq.HsubTimesVec(veff, nodes, v).reshape(nodes.size, -1)
        for b, nd in enumerate(nodes):
            assert H.rel(hv[b], o.hsub(veff, int(nd), v[b])) < (2e-6 if prec == "mixed" else 1e-12), (prec, b)
            assert np.array_equal(sq.HsubTimesVec(veff, nodes[b:b + 1], v[b:b + 1]).reshape(-1), hv[b]), (prec, b)
        if moments:
            got = sq.node_moments(veff, nodes)
            one = sq.node_moments(veff, nodes[:1])
            for k in ("chi", "zee", "mu", "iters"):
                assert np.array_equal(got[k][:1], one[k]), k
            if prec == "fp64":
                ref = o.moments_nodes(veff, nodes, nthreads=0)
                assert np.array_equal(got["iters"], ref["iters"])
                for k in ("chi", "zee", "mu"):
                    assert H.rel(got[k], np.asarray(ref[k]).reshape(got[k].shape)) < 1e-10, k
        sq.close()


def test_rows_without_padding():
    """35^3 cubes with boxes of 5^3: the padded slab leaves no room for the columns."""
    S, Rcut, T = system("al", 16, 1.5, 17, scattered(6, 1))
    nodes = block(16, 4, 4, 4)
    assert S.type_info(0)["nlocc"] == 2 and 80 < list_length(S, nodes) <= 121
    print("unpadded", list_length(S, nodes), flush=True)
    check(S, Rcut, T, nodes)


def test_images_shared_out():
    """33^3 cubes with boxes of 3^3: the columns leave no room for the longest list."""
    S, Rcut, T = system("al", 12, 2.7, 16, scattered(14, 2))
    nodes = block(12, 4, 4, 4)
    assert S.type_info(0)["nlocc"] == 1 and 330 < list_length(S, nodes) <= 451
    print("shares", list_length(S, nodes), flush=True)
    check(S, Rcut, T, nodes)


def test_staged_images_shared_out():
    """43^3 cubes with a group list too long for k_projs' slab: most atoms lie on
    planes that the cubes of the block's first or last nodes alone reach."""
    n = 64
    S, Rcut, T = system("al", n, 0.98, 21, on_faces(n, 310, 310, 130, 60.0, 47.0, 44.0, 3))
    nodes = block(n, 20, 20, 20)
    assert S.type_info(0)["nlocc"] == 3 and list_length(S, nodes) > 710
    assert max(list_length(S, nodes[i:i + 1]) for i in range(8)) <= 512
    print("staged shares", list_length(S, nodes), flush=True)
    check(S, Rcut, T, nodes, precs=("fp64",), moments=False)


@pytest.mark.parametrize("n,h,nloc,natom", [(16, 1.5, 14, 40), (12, 1.5, 3, 140), (12, 1.2, 10, 30)])
def test_dense_tables_of_several_projectors(n, h, nloc, natom):
    """Matrix-core walks of groups with long lists: a deep slab whose images are
    shared out (29^3 cubes, 402 images), and slabs of one plane where the deep one
    keeps more images alive than there are slots (7^3 with 151, 21^3 with 418)."""
    S, Rcut, T = system("li", n, h, nloc, scattered(natom, 5))
    nodes = block(n, 4, 4, 4)
    assert list_length(S, nodes) == {14: 402, 3: 151, 10: 418}[nloc]
    print("dense", S.info["nloc"], flush=True)
    check(S, Rcut, T, nodes, precs=("fp64", "mixed_lanczos"), moments=True)


def test_nonlocal_apply_without_the_column_table():
    """43^3 cubes of a dense p-channel table: the nonlocal apply's rows fill the LDS."""
    S, Rcut, T = system("li", 40, 1.2, 21, scattered(250, 7))
    nodes = block(40, 0, 3, 10)
    gl = list_length(S, nodes)
    rows = 4 * 3 * S.images()["type"].size + gl * 3 * 80
    print("columns", gl, rows, flush=True)
    assert rows <= 160 * 1024 < rows + 4 * 46 ** 2
    assert max(list_length(S, nodes[i:i + 1]) for i in range(8)) <= 512
    check(S, Rcut, T, nodes, precs=("fp64", "mixed"), moments=False)


@pytest.mark.parametrize("n,h,nloc,natom,waves,need", [(16, 0.8, 8, 20, 12, range(1, 5)), (12, 1.2, 7, 20, 8, range(6, 11)),
                                                       (12, 1.2, 7, 40, 8, range(11, 17))])
def test_every_compiled_slot_count(n, h, nloc, natom, waves, need):
    """s-channel walks of twelve waves with 4 slots and of eight with 10 and 16, for
    slabs of one FP64 and two FP32 planes."""
    S, Rcut, T = system("al", n, h, nloc, scattered(natom, 5))
    nodes = block(n, 4, 4, 4)
    assert all(slots(S, nodes, planes, waves) in need for planes in (1, 2))
    assert waves == 12 or slots(S, nodes, 1, 12) > 4
    print("slots", slots(S, nodes, 1, waves), slots(S, nodes, 2, waves), flush=True)
    check(S, Rcut, T, nodes, precs=("fp64", "mixed", "mixed_lanczos"))
