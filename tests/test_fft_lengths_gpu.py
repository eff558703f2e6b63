"""H|psi> and the density at every transform length of the register passes
that the other tests leave out: three at a time, one per axis (separate y and
z passes), with equal y and z lengths (both in one kernel), and with a
wavefunction sphere wider than a quarter of the grid, where no frequency run
may be left out."""
import numpy as np
import pytest

from amdkiit_amd import psp, systems
from amdkiit_amd.context import KSContext
from amdkiit_amd.pwgrid import Cell, PWSetup
from oracle import pw_oracle as O
from oracle.ks_oracle import KSOracle
from tests.common import random_bands, smooth_potential

pytestmark = pytest.mark.gpu

GRIDS = [(32, 40, 50), (54, 64, 80), (90, 96, 120), (128, 150, 20), (24, 160, 162), (192, 36, 30), (30, 20, 192),
         (162, 128, 32), (50, 90, 64), (40, 54, 96), (64, 32, 90), (80, 48, 54), (96, 50, 40), (120, 80, 48), (150, 24, 60)]


LENGTHS = (20, 24, 30, 32, 36, 40, 48, 50, 54, 60, 64, 72, 80, 90, 96, 100, 108, 120, 128, 144, 150, 160, 162, 180, 192)
SQUARE = [(24, k, k) for k in LENGTHS] + [(k, 20, 20) for k in LENGTHS if k >= 32]


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def sphere_to_the_edge(n):
    """A box whose density sphere reaches the largest |m| < n/2 of each axis."""
    return PWSetup(Cell(np.diag([0.25 * k for k in n])), 0.24 * (2 * np.pi / 0.5) ** 2, n=n)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("n", GRIDS + SQUARE, ids=lambda n: "x".join(map(str, n)))
def test_lengths(n, prec, tol):
    pw = sphere_to_the_edge(n)
    nb = 3
    print(f"case=lengths n={n} ngpw={pw.ngpw} R={np.abs(pw.mill_pw).max(0)} prec={prec}", flush=True)
    c = random_bands(pw, nb, seed=3)
    occ = np.array([2.0, 1.0, 2.0])
    v = smooth_potential(pw)
    ctx = KSContext(pw, nb, prec)
    ctx.set_vks(v)
    assert rel(ctx.vpsi(c, occ), O.vpsi(c, occ, v, pw.mill_pw, pw.n, pw.cell.g)) < tol
    assert rel(ctx.eval_density(c, occ), O.eval_density(c, occ, pw.mill_pw, pw.n, pw.cell.omega)) < tol
    ctx.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("n", [(30, 32, 36), (40, 50, 54), (64, 60, 72), (100, 24, 80)], ids=lambda n: "x".join(map(str, n)))
def test_sphere_wider_than_a_quarter_of_the_grid(n, prec, tol):
    pw = sphere_to_the_edge(n)
    pw.mill_pw, pw.ngpw = pw.mill_rho, pw.ngrho  # |m| up to n/2 - 1
    assert (4 * np.abs(pw.mill_pw).max(0) > np.array(n)).all()
    nb = 10  # density in pair groups too
    print(f"case=wide n={n} ngpw={pw.ngpw} R={np.abs(pw.mill_pw).max(0)} prec={prec}", flush=True)
    c = random_bands(pw, nb, seed=4)
    occ = np.full(nb, 2.0)
    v = smooth_potential(pw)
    ctx = KSContext(pw, nb, prec)
    ctx.set_vks(v)
    assert rel(ctx.vpsi(c, occ), O.vpsi(c, occ, v, pw.mill_pw, pw.n, pw.cell.g)) < tol
    assert rel(ctx.eval_density(c, occ), O.eval_density(c, occ, pw.mill_pw, pw.n, pw.cell.omega)) < tol
    ctx.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("nb", [1, 2, 9, 33])
def test_one_kernel_matches_separate_passes(nb, prec, tol, monkeypatch):
    """The y-z kernels against the separate passes: pair groups and pairs per
    block at several band counts, one pair chunk and several."""
    pw = sphere_to_the_edge((30, 36, 36))
    c = random_bands(pw, nb, seed=6)
    occ = np.linspace(2.0, 0.0, nb)
    v = smooth_potential(pw)
    out = {}
    for fft, budget in (("passes", None), ("", None), ("", "1")):
        monkeypatch.setenv("AMDK_FFT", fft)
        if budget:
            monkeypatch.setenv("AMDK_PAIR_BUDGET_MB", budget)
        print(f"case=one_kernel nb={nb} prec={prec} fft={fft!r} budget={budget}", flush=True)
        ctx = KSContext(pw, nb, prec)
        ctx.set_vks(v)
        out[fft, budget] = (ctx.vpsi(c, occ), ctx.eval_density(c, occ))
        ctx.close()
    for key in (("", None), ("", "1")):
        assert rel(out[key][0], out["passes", None][0]) < tol
        assert rel(out[key][1], out["passes", None][1]) < tol
    assert np.array_equal(out["", None][0], out["", "1"][0])


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("n,nb", [(72, 65), (90, 70), (100, 64), (108, 66), (120, 65), (144, 67), (180, 257)])
def test_many_pairs_in_one_kernel(n, nb, prec, tol, monkeypatch):
    """The density from the y-z kernel at the lengths and band counts where it
    is used: pair groups that divide the pairs and that do not, an odd band
    count, and pairs in several chunks with a short last one (which the chunk
    before accumulates into)."""
    pw = sphere_to_the_edge((20, n, n))
    c = random_bands(pw, nb, seed=7)
    occ = np.linspace(2.0, 0.5, nb)
    v = smooth_potential(pw)
    want = O.eval_density(c, occ, pw.mill_pw, pw.n, pw.cell.omega)
    want2 = O.vpsi(c, occ, v, pw.mill_pw, pw.n, pw.cell.g)
    for budget in (None, "40"):
        if budget:
            monkeypatch.setenv("AMDK_PAIR_BUDGET_MB", budget)
        print(f"case=many_pairs n={n} nb={nb} prec={prec} budget={budget}", flush=True)
        ctx = KSContext(pw, nb, prec)
        ctx.set_vks(v)
        assert rel(ctx.eval_density(c, occ), want) < tol
        assert rel(ctx.vpsi(c, occ), want2) < tol
        ctx.close()


@pytest.mark.parametrize("n,nb,edge,precs", [(72, 65, 0.24, ("mixed",)), (80, 65, 0.24, ("mixed",)), (90, 65, 0.24, ("mixed", "fp64")),
                                             (100, 67, 0.24, ("mixed", "fp64")), (108, 65, 0.24, ("fp64",)),
                                             (120, 65, 0.24, ("fp64",)), (144, 129, 0.24, ("mixed",)),
                                             (144, 65, 0.11, ("fp64",)), (160, 129, 0.24, ("mixed",)),
                                             (180, 131, 0.24, ("mixed",)), (192, 129, 0.205, ("mixed",))])
def test_density_lengths_of_one_kernel(n, nb, edge, precs):
    """Every length and precision that takes the density from the y-z kernel,
    at the band counts from which it does (192^3, and 144^3 in double
    precision, only on a smaller sphere), and none that does not."""
    pw = PWSetup(Cell(np.diag([5.0, 0.25 * n, 0.25 * n])), edge * (2 * np.pi / 0.5) ** 2, n=(20, n, n))
    c = random_bands(pw, nb, seed=9)
    occ = np.linspace(2.0, 0.5, nb)
    want = O.eval_density(c, occ, pw.mill_pw, pw.n, pw.cell.omega)
    for prec, tol in (("fp64", 1e-12), ("mixed", 2e-6)):
        print(f"case=density_lengths n={n} nb={nb} R={np.abs(pw.mill_pw).max(0)} prec={prec}", flush=True)
        ctx = KSContext(pw, nb, prec)
        ctx.profile(True)
        assert rel(ctx.eval_density(c, occ), want) < tol
        assert ("yz_rho" in ctx.profile_names()) == (prec in precs)
        ctx.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
def test_several_pairs_per_block(prec, tol, monkeypatch):
    """67 pairs at 100^3: three (FP32) or six (FP64) to a block of H|psi> and
    one over, which work on the same planes in LDS in turn, and the density in
    groups that do not divide them."""
    pw = sphere_to_the_edge((100, 100, 100))
    nb = 133
    c = random_bands(pw, nb, seed=10)
    occ = np.linspace(2.0, 0.5, nb)
    v = smooth_potential(pw)
    out = {}
    for fft in ("passes", ""):
        monkeypatch.setenv("AMDK_FFT", fft)
        print(f"case=several_pairs prec={prec} fft={fft!r}", flush=True)
        ctx = KSContext(pw, nb, prec)
        ctx.set_vks(v)
        ctx.profile(True)
        out[fft] = (ctx.vpsi(c, occ), ctx.eval_density(c, occ))
        assert ({"yz_vpsi", "yz_rho"} <= set(ctx.profile_names())) == (fft == "")
        ctx.close()
    for got, want in zip(out[""], out["passes"]):
        assert rel(got, want) < tol


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
def test_potential_of_a_step_in_a_later_hpsi(prec, tol):
    """An SCF step by the separate passes leaves V(r) x fastest; an H|psi> by
    the y-z kernels after it reorders that potential, after one more step the
    new one, and after a V_KS of its own that."""
    s = systems.water_box((1, 1, 2), 10.0, 20.0, "PBE")
    nb = s.nbands
    other = random_bands(s.pw, nb, seed=11)
    occ = np.linspace(2.0, 1.0, nb)
    ctx, ref = KSContext(s.pw, nb, prec), KSContext(s.pw, nb, prec)
    for x in (ctx, ref):
        x.set_species(s.tables)
        x.set_positions(s.sp, s.tau)
    ctx.wfn_load(ref.ortho(random_bands(s.pw, nb, seed=12)), s.occ)
    ctx.profile(True)

    def check(what, rho):
        print(f"case=later_hpsi {what} n={s.pw.n} prec={prec}", flush=True)
        v, _ = ref.vks(rho, s.xc)
        assert rel(ctx.vpsi(other, occ), O.vpsi(other, occ, v, s.pw.mill_pw, s.pw.n, s.pw.cell.g)) < tol
    for it in (1, 2):
        rho = ref.eval_density(ctx.wfn_store(), s.occ)
        ctx.scf_step(it, s.xc)
        check(f"step {it}", rho)
        check(f"step {it}, again", rho)
    assert "z_vpsi" in ctx.profile_names() and "yz_vpsi" in ctx.profile_names()
    rho2 = ref.eval_density(other, occ)
    ctx.vks(rho2, s.xc)
    check("V_KS", rho2)
    rho = ref.eval_density(ctx.wfn_store(), s.occ)
    ctx.scf_step(3, s.xc)
    check("step 3", rho)
    for x in (ctx, ref):
        x.close()


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("lacks", ["plane m3 = 0", "odd planes"])
def test_plane_wave_lists_with_empty_planes(lacks, prec, tol):
    """Lists whose planes are contiguous but not all there: without the plane
    m3 = 0, and so without the row (0, 0), at a row count (112) that fills its
    128-byte blocks, and with every second plane empty."""
    pw = PWSetup(Cell(np.diag([6.0, 9.0, 9.0])), 0.23 * (2 * np.pi / 0.5) ** 2, n=(24, 36, 36))
    m3 = pw.mill_pw[:, 2]
    pw.mill_pw = np.ascontiguousarray(pw.mill_pw[m3 != 0 if lacks == "plane m3 = 0" else m3 % 2 == 0])
    pw.ngpw = len(pw.mill_pw)
    nb = 5
    print(f"case=empty_planes {lacks} ngpw={pw.ngpw} prec={prec}", flush=True)
    c = random_bands(pw, nb, seed=8)
    occ = np.array([2.0, 1.0, 2.0, 0.0, 2.0])
    v = smooth_potential(pw)
    ctx = KSContext(pw, nb, prec)
    if lacks == "plane m3 = 0":
        assert ctx.sphere_geometry()["nrow"] == 112
    ctx.set_vks(v)
    assert rel(ctx.vpsi(c, occ), O.vpsi(c, occ, v, pw.mill_pw, pw.n, pw.cell.g)) < tol
    # (single precision scales the density by a norm that takes the first plane wave for G = 0)
    if prec == "fp64" or lacks == "odd planes":
        assert rel(ctx.eval_density(c, occ), O.eval_density(c, occ, pw.mill_pw, pw.n, pw.cell.omega)) < tol
    ctx.close()


@pytest.mark.parametrize("xc", ["PZ", "PBE"])
@pytest.mark.parametrize("n", [(20, 24, 30), (54, 64, 80), (90, 48, 100), (36, 108, 50), (120, 32, 72), (144, 40, 60), (160, 20, 96),
                               (30, 128, 150), (24, 162, 36), (48, 180, 32), (192, 20, 90)], ids=lambda n: "x".join(map(str, n)))
def test_potential_of_one_field(n, xc):
    """rho into G space and V_KS out of it as single real fields (the planes
    m3 >= 0 only), each length on some axis."""
    pw = sphere_to_the_edge(n)
    tab = psp.Tables(pw, [psp.gth("Si", "LDA")])
    tau = np.array([[1.0, 1.5, 2.0]])
    print(f"case=one_field n={n} ngrho={pw.ngrho} xc={xc}", flush=True)
    ctx = KSContext(pw, 2, "fp64")
    ctx.set_species(tab)
    ctx.set_positions([0], tau)
    orc = KSOracle(pw, tab, [0], tau, xc, workers=8)
    u = smooth_potential(pw)
    rho = 0.05 * np.exp(u / np.abs(u).max())
    v, e = ctx.vks(rho, xc)
    want, exc = orc.vks(rho, orc.rhor2g(rho))
    assert rel(v, want) < 1e-10
    assert abs(e["exc"] - exc) < 1e-10 * abs(exc)
    ctx.close()
