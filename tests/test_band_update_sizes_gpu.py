"""Band products at the edges of the update's block widths (32, 64, 128
columns) and of the overlap's tiles, with few and with many plane waves."""
import numpy as np
import pytest

from amdkiit_amd.context import KSContext
from tests.common import random_bands, small_setup

pytestmark = pytest.mark.gpu


def overlap(a, b):
    return 2.0 * (a.conj() @ b.T).real - np.outer(a[:, 0].real, b[:, 0].real)


# FP32 products are summed in FP32 over 32 terms and in FP64 beyond: a few
# 2^-24 of the largest term
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("nb", [1, 16, 17, 31, 32, 33, 63, 64, 65, 128, 129])
@pytest.mark.parametrize("box,ecut", [(7.0, 20.0), (10.0, 30.0)])
def test_lagrange_and_ortho(box, ecut, nb, prec, tol):
    pw = small_setup(box, ecut)
    if nb > pw.ngpw // 2:
        pytest.skip("more bands than the sphere can hold")
    print(f"case=band_update nb={nb} npw={pw.ngpw} prec={prec}", flush=True)
    c = random_bands(pw, nb, seed=nb)
    ctx = KSContext(pw, nb, prec)
    s = overlap(c, c)
    inv = np.linalg.inv(np.linalg.cholesky(s).T)
    want = inv.T @ c
    want[:, 0] = want[:, 0].real
    got = ctx.ortho(c)
    assert np.abs(got - want).max() < 1e-10 * np.abs(want).max()
    assert np.abs(overlap(got, got) - np.eye(nb)).max() < 1e-12
    c2 = random_bands(pw, nb, seed=nb + 500)
    g, gemax, cnorm = ctx.lagrange(got, c2, np.full(nb, 2.0))
    ref = c2 - overlap(c2, got).T @ got
    ref[:, 0] = ref[:, 0].real
    assert np.abs(g - ref).max() < tol * np.abs(c2).max() * max(1.0, np.sqrt(nb))
    assert abs(gemax - np.abs(ref).max()) < 10 * tol * np.abs(c2).max()
    ctx.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("nb", [5, 18, 50, 66])
@pytest.mark.parametrize("box,ecut", [(6.0, 8.0), (10.0, 30.0)])
def test_lagrange_with_empty_bands(box, ecut, nb, prec, tol):
    """One-launch and split-K overlaps with bands that take no part."""
    pw = small_setup(box, ecut)
    if nb > pw.ngpw // 2:
        pytest.skip("more bands than the sphere can hold")
    print(f"case=empty_bands nb={nb} npw={pw.ngpw} prec={prec}", flush=True)
    ctx = KSContext(pw, nb, prec)
    c = ctx.ortho(random_bands(pw, nb, seed=nb))
    c2 = random_bands(pw, nb, seed=nb + 500)
    occ = np.full(nb, 2.0)
    occ[1::4] = 0.0
    g, _, _ = ctx.lagrange(c, c2, occ)
    lam = overlap(c2, c) * np.outer(occ != 0, occ != 0)
    ref = c2 - lam.T @ c
    ref[:, 0] = ref[:, 0].real
    assert np.abs(g - ref).max() < tol * np.abs(c2).max() * max(1.0, np.sqrt(nb))
    ctx.close()
