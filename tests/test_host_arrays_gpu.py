"""Host arrays on both sides of the sizes where their check moves to the
device and their way out to several threads: values, padding and refusals."""
import numpy as np
import pytest

from amdkiit_amd import lib as L
from amdkiit_amd.context import KSContext
from amdkiit_amd.pwgrid import Cell, PWSetup
from tests.common import random_bands, smooth_potential

pytestmark = pytest.mark.gpu

# bands of 13,601 plane waves (0.22 MB each): 0.2, 1.3, 10.2, 14.4, 33.3 and 38.1 MB
COUNTS = (1, 6, 47, 66, 153, 175)


@pytest.fixture(scope="module")
def setup():
    return PWSetup(Cell.cubic(14.0), 70.0)


def padded(c, pad, fill):
    out = np.full((c.shape[0], c.shape[1] + pad), fill, np.complex128)
    out[:, : c.shape[1]] = c
    return out


@pytest.mark.parametrize("nb", COUNTS)
@pytest.mark.parametrize("pad", [0, 5])
def test_bands_in_and_out(setup, nb, pad):
    pw = setup
    print(f"case=bands nb={nb} pad={pad} MB={16e-6 * nb * pw.ngpw:.1f}", flush=True)
    ctx = KSContext(pw, nb, "fp64")
    c = random_bands(pw, nb, seed=nb)
    host = padded(c, pad, 7.0 + 7.0j)
    occ = np.full(nb, 2.0)
    ld = pw.ngpw + pad
    ctx._chk(ctx.lib.amdk_wfn_load(ctx.h, L.dptr(host.view(np.float64).reshape(-1)), ld, L.dptr(occ), nb))
    out = np.full_like(host, -3.0)
    ctx._chk(ctx.lib.amdk_wfn_store(ctx.h, L.dptr(out.view(np.float64).reshape(-1)), ld))
    assert np.array_equal(out[:, : pw.ngpw], c)
    assert (out[:, pw.ngpw:] == -3.0).all()
    ctx.close()


@pytest.mark.parametrize("nb", COUNTS)
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_refusals_leave_the_state(setup, nb, bad):
    pw = setup
    print(f"case=refusal nb={nb} bad={bad}", flush=True)
    ctx = KSContext(pw, nb, "fp64")
    c = random_bands(pw, nb, seed=nb)
    occ = np.full(nb, 2.0)
    ctx.wfn_load(c, occ)
    for b, g, pad in ((0, 0, 0), (nb - 1, pw.ngpw - 1, 0), (nb // 2, 777, 0), (nb - 1, pw.ngpw + 1, 3)):
        host = padded(c, pad, 0.0)
        host[b, g] = complex(0.0, bad) if g % 2 else complex(bad, 0.0)
        rc = ctx.lib.amdk_wfn_load(ctx.h, L.dptr(host.view(np.float64).reshape(-1)), pw.ngpw + pad, L.dptr(occ), nb)
        assert rc == L.ERR_NONFINITE
        assert np.array_equal(ctx.wfn_store(), c)
    ctx.close()


@pytest.mark.parametrize("n", [(20, 20, 20), (72, 72, 72), (120, 120, 120)], ids=str)
def test_grids(n):
    """64 kB, 3 MB and 13.8 MB of V(r) and rho(r)."""
    pw = PWSetup(Cell(np.diag([0.25 * k for k in n])), 6.0, n=n)
    ctx = KSContext(pw, 1, "fp64")
    print(f"case=grids n={n}", flush=True)
    v = smooth_potential(pw)
    ctx.set_vks(v)
    bad = v.copy()
    bad[n[2] - 1, 3, n[0] - 1] = np.nan
    with pytest.raises(L.AmdkError) as ei:
        ctx.set_vks(bad)
    assert ei.value.code == L.ERR_NONFINITE
    # a single plane wave: |psi|^2 is known everywhere
    c = np.zeros((1, pw.ngpw), np.complex128)
    k = int(np.flatnonzero((pw.mill_pw == [1, 0, 0]).all(1))[0])
    c[0, k] = 1.0
    x = 2.0 * np.pi * np.arange(n[0]) / n[0]
    rho = ctx.eval_density(c, np.array([2.0]))
    want = 2.0 / pw.cell.omega * (2.0 * np.cos(x)) ** 2
    assert np.abs(rho - want).max() < 1e-12 * want.max()
    ctx.close()
