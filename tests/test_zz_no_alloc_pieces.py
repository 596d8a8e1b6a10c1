"""sqg_hsub_apply_batch_noalloc on nodes so scattered that their group lists do
not fit the scratch array beside the batch's vectors: the call runs as pieces,
bit for bit the product that sqg_hsub_apply_batch gives."""
import numpy as np
import pytest

import helpers as H
from sqdft_amd import _lib as L
from sqdft_amd.configs import smooth_veff
from sqdft_amd.sq import SpectralQuadrature
from test_zz_no_alloc import DevArray, noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case,prec", [("small_al", "fp64"), ("small_lih", "fp64"), ("small_al", "mixed"),
                                       ("small_lih", "mixed_lanczos")])
def test_pieces_match_hsub(case, prec):
    print("noalloc pieces", case, prec, flush=True)
    S = getattr(H, case)()[0]
    sq = SpectralQuadrature(S, precision=prec)
    M3, rs = sq.M ** 3, 4 if prec == "mixed" else 8
    n_ip = sum(S.type_info(int(t))["nproj"] for t in S.images()["type"])
    vec = M3 * rs * (3 if prec == "mixed" else 1) + 8 * n_ip
    nb = int(0.97 * (64 << 20) / (vec + 4 * (512 + 2 + 1025 / 8)))   # below the limit in full groups
    assert nb * (vec + 4 * 1027) > (64 << 20)                         # above it in groups of one node
    rng = np.random.Generator(np.random.PCG64(5))
    n2 = S.n ** 2
    lo, hi = rng.integers(0, n2, nb), S.nn - 1 - rng.integers(0, n2, nb)
    nodes = np.where(np.arange(nb) % 2 == 0, lo, hi).astype(np.int32)
    v = rng.normal(size=(nb, M3))
    veff = smooth_veff(S)
    ref = sq.HsubTimesVec(veff, nodes, v).reshape(nb, M3)
    veff_d, v_d, hv_d = DevArray(veff), DevArray(v), DevArray(np.full((nb, M3), np.nan))
    for _ in range(2):
        code = noalloc(sq, veff_d, nodes, v_d, hv_d)
        assert code == 0, L.STATUS.get(code, code)
        assert np.array_equal(hv_d.get(), ref)
    for d in (veff_d, v_d, hv_d):
        d.free()
    sq.close()
