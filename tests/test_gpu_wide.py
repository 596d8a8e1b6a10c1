"""Sizes past the first tile of a kernel: Lanczos runs longer than the rows that
its eigenvalue kernel keeps on chip, and adjoint rows longer than sixteen nodes,
against the FP64 oracle at 1e-10 (its summation order differs; the suite's bound
for FP64 bounds and derivatives)."""
import numpy as np
import pytest

import helpers as H
from sqdft_amd.configs import smooth_veff
from sqdft_amd.sq import SpectralQuadrature

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elem", ["al", "lih"])
def test_extremes_of_500_lanczos_passes(elem):
    from oracle import OracleSystem

    print("500 passes", elem, flush=True)
    S, Rcut, T = (H.small_al if elem == "al" else H.small_lih)(npl=8)
    i, veff = S.info, smooth_veff(S)
    o = OracleSystem(i["n"], i["L"], H.types_of(S), Rcut, i["npl"], T, h=i["h"], lanczos_tol=-1.0,
                     fermi_tol=i["fermi_tol"], fermi_alg=i["fermi_alg"])
    nodes = np.array([0, 7, S.nn // 2, S.nn - 1], dtype=np.int32)
    ref = o.moments_nodes(veff, nodes, nthreads=0)
    sq = SpectralQuadrature(S, precision="fp64", lanczos_tol=-1.0)
    sq.density(veff, scf_iter=1)
    nd = sq.node_data()
    assert np.array_equal(nd["iters"][nodes], ref["iters"])
    for k in ("chi", "zee"):
        assert H.rel(nd[k][nodes], ref[k]) < 1e-10, k


@pytest.mark.parametrize("n", [17, 20])
def test_adjoint_on_longer_rows(n):
    print("adjoint", n, flush=True)
    S, Rcut, T = H.small_al(npl=8, n_cell=n)
    veff, o = smooth_veff(S), H.oracle_for(S, Rcut, T)
    sq = SpectralQuadrature(S, precision="fp64", ckpt_interval=3)
    d = sq.density(veff, scf_iter=1)
    nd = sq.node_data()
    w = np.random.Generator(np.random.PCG64(n)).normal(size=S.nn)
    g = sq.adjoint_veff(w, fixed_n=1)
    ref = o.adjoint_veff(veff, nd["chi"], nd["zee"], nd["mu"].reshape(-1), d["lambda_f"], w, fixed_n=1)
    assert H.rel(g, ref) < 1e-10
