"""The adjoint's gather where the grid is wider than the node cube (24 to 36 nodes
a side against cubes of 9^3), in one batch and in batches of a few planes, against
the FP64 oracle at 1e-10 (the suite's bound for FP64 derivatives)."""
import numpy as np
import pytest

import helpers as H
from sqdft_amd.configs import smooth_veff
from sqdft_amd.sq import SpectralQuadrature

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncell,n_cell,Rcut", [(2, 12, 2.5), (3, 9, 3.0), (3, 12, 2.5)])
def test_adjoint_on_grids_wider_than_the_cube(ncell, n_cell, Rcut):
    S, Rc, T = H.small_al(ncell=ncell, n_cell=n_cell, Rcut=Rcut, npl=8)
    veff, o = smooth_veff(S), H.oracle_for(S, Rc, T)
    w = np.random.Generator(np.random.PCG64(S.n)).normal(size=S.nn)
    ref = None
    for planes in (S.n, 5):
        print("adjoint", S.n, S.info["nloc"], planes, flush=True)
        sq = SpectralQuadrature(S, precision="fp64", ckpt_interval=3, batch_nodes=planes * S.n ** 2)
        d = sq.density(veff, scf_iter=1)
        nd = sq.node_data()
        if ref is None:
            ref = o.adjoint_veff(veff, nd["chi"], nd["zee"], nd["mu"].reshape(-1), d["lambda_f"], w, fixed_n=1)
        assert H.rel(sq.adjoint_veff(w, fixed_n=1), ref) < 1e-10
        sq.close()
