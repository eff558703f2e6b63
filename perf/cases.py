"""Performance cases: the work that a user of amdkiit_amd has the library do.

Each case is one call, or one short run, through KSContext (or, for the
density on device arrays, the C ABI under it):

  hpsi     H|psi>, local and kinetic part, on device-resident bands
  density  rho(r) of device-resident bands
  vks      V_KS(r) and the energies of a density held on the host
  ortho    Cholesky orthonormalisation of bands held on the host
  nonloc   fnl followed by fnonloc on bands held on the host
  scf      load bands, a run of SCF steps, store the bands (an SP run)
  md       as scf after new atomic positions, with the forces in the last
           step (one force evaluation of MD or of a geometry optimisation)

Systems are the seeded water boxes and displaced silicon of
amdkiit_amd.systems.  In the single-precision modes ("mixed", "bf16") H|psi>,
the density, the projections and all that follows from them are
single-precision numbers, and a program that chooses these modes keeps them in
that type, as these cases do; V_KS and the orthonormalisation are double in
every mode.
"""
import functools
import math

import numpy as np
import torch

from amdkiit_amd import lib, systems
from amdkiit_amd.context import KSContext

DEV = "cuda"
VOL_PER_MOLECULE = 202.06  # bohr^3 of a water molecule at 1 g/cm^3
RAGGIO = 1.2               # width of the Gaussian ion charges, bohr


def listed():
    water = dict(system="water", xc="PBE")
    return [
        # the smallest H|psi>: two molecules, a handful of bands; launches count
        dict(water, name="hpsi_2h2o_8b_fp64", kind="hpsi", m1=1, m2=1, m3=2, box=10.0, ecut=20.0, prec="fp64", nb=8),
        # the H|psi> whose bandwidth the benchmark reports
        dict(water, name="hpsi_32h2o_mixed", kind="hpsi", m1=4, m2=4, m3=2, box=18.63, ecut=70.0, prec="mixed", nb=128),
        # the largest box of the benchmark, one H|psi>
        dict(water, name="hpsi_128h2o_mixed", kind="hpsi", m1=8, m2=4, m3=4, box=29.57, ecut=80.0, prec="mixed", nb=512),
        # an odd band count on a box off the benchmark's sizes (90^3)
        dict(water, name="hpsi_27h2o_odd_fp64", kind="hpsi", m1=3, m2=3, m3=3, box=17.6, ecut=60.0, prec="fp64", nb=107),
        # density of a middling box (64^3)
        dict(water, name="density_8h2o_mixed", kind="density", m1=2, m2=2, m3=2, box=11.74, ecut=70.0, prec="mixed", nb=32),
        # potential of a host density, as a program that keeps the reference's arrays calls it
        dict(water, name="vks_32h2o_fp64", kind="vks", m1=4, m2=4, m3=2, box=18.63, ecut=70.0, prec="fp64", nb=128),
        # orthonormalisation of host bands after a geometry update
        dict(water, name="ortho_32h2o_fp64", kind="ortho", m1=4, m2=4, m3=2, box=18.63, ecut=70.0, prec="fp64", nb=128),
        # projections and the nonlocal part with BF16 products, silicon (s and p projectors)
        dict(name="nonloc_si64_bf16", kind="nonloc", system="si", xc="PZ", m1=2, m2=2, m3=2, box=0.0, ecut=30.0, prec="bf16",
             nb=128),
        # a whole small run: bound by latency
        dict(water, name="scf_2h2o_fp64", kind="scf", m1=1, m2=1, m3=2, box=10.0, ecut=20.0, prec="fp64", nb=8, steps=40,
             lowdin=False),
        # the benchmark's system, single-precision mode
        dict(water, name="scf_32h2o_mixed", kind="scf", m1=4, m2=4, m3=2, box=18.63, ecut=70.0, prec="mixed", nb=128, steps=40,
             lowdin=False),
        # the same in double precision, off the benchmark's box (odd bands, 108^3)
        dict(water, name="scf_32h2o_108_fp64", kind="scf", m1=4, m2=4, m3=2, box=19.4, ecut=73.0, prec="fp64", nb=127, steps=30,
             lowdin=False),
        # one force evaluation of 64 molecules
        dict(water, name="md_64h2o_mixed", kind="md", m1=4, m2=4, m3=4, box=23.47, ecut=80.0, prec="mixed", nb=256, steps=24,
             lowdin=False),
    ]


def draw(rng):
    kind = rng.choice(["hpsi", "hpsi", "density", "vks", "ortho", "nonloc", "scf", "scf", "md"])
    prec = rng.choice(["fp64", "mixed", "mixed", "bf16"]) if kind in ("nonloc", "scf", "md") else rng.choice(["fp64", "mixed"])
    while True:
        m = [rng.randint(1, 4) for _ in range(3)]
        nmol = m[0] * m[1] * m[2]
        box = round((nmol * VOL_PER_MOLECULE) ** (1.0 / 3.0) * rng.uniform(0.97, 1.15), 3)
        ecut = round(math.exp(rng.uniform(math.log(25.0), math.log(90.0))), 1)
        if nmol <= 48 and box >= 7.0 and 20 <= grid_of(box, ecut) <= 144:
            break
    # all the occupied bands, or a block of them (odd counts among them); a
    # whole run has all of them
    nb = 4 * nmol
    if kind not in ("scf", "md"):
        nb = max(2, int(nb * rng.uniform(0.5, 1.0)))
    c = dict(kind=kind, system="water", xc=rng.choice(["PBE", "PBE", "PZ"]), m1=m[0], m2=m[1], m3=m[2], box=box, ecut=ecut,
             prec=prec, nb=nb)
    if kind in ("scf", "md"):
        c.update(steps=rng.randint(8, 24), lowdin=rng.random() < 0.25)
    return c


def grid_of(box, ecut):
    return int(math.floor(box / math.pi * math.sqrt(4.0 * ecut) + 1.0))


# ---------------------------------------------------------------------------
# what a program has before the call

@functools.lru_cache(maxsize=None)
def _system(kind, m1, m2, m3, box, ecut, xc):
    """The basis and the species tables (made once per program)."""
    if kind == "si":
        return systems.si64_like(cells=m1, ecut=ecut, xc=xc)
    return systems.water_box((m1, m2, m3), box, ecut, xc)


def system_of(case):
    return _system(case["system"], case["m1"], case["m2"], case["m3"], case["box"], case["ecut"], case["xc"])


def generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def positions(s, seed):
    return s.tau + 0.05 * np.random.default_rng(seed).standard_normal(s.tau.shape)


def bands(s, nb, seed, orthonormal=True):
    """Seeded random bands damped by 1 / (1 + |G|^2), complex128 (nb, ngpw)."""
    u = torch.rand((nb, s.pw.ngpw, 2), dtype=torch.float64, device=DEV, generator=generator(seed)) - 0.5
    c = torch.view_as_complex(u) / (1.0 + torch.from_numpy(s.pw.g2_pw).to(DEV))
    c[:, 0] = c[:, 0].real.to(c.dtype)
    return cholesky_orthonormal(c) if orthonormal else c


def occupations(nb, seed):
    """Doubly occupied bands; the last one is at times half filled."""
    occ = np.full(nb, 2.0)
    occ[-1] = (2.0, 2.0, 1.0)[seed % 3]
    return occ


def internal_order(pw):
    """Where plane wave i of the caller's order sits in the library's arrays
    (amdk_pw_order: the half sphere m3 > 0, ..., sorted by m3, m2, m1), and
    whether it is held conjugated."""
    m = pw.mill_pw.astype(np.int64)
    conj = (m[:, 2] < 0) | ((m[:, 2] == 0) & ((m[:, 1] < 0) | ((m[:, 1] == 0) & (m[:, 0] < 0))))
    z = np.where(conj[:, None], -m, m)
    pos = np.empty(len(m), np.int64)
    pos[np.lexsort((z[:, 0], z[:, 1], z[:, 2]))] = np.arange(len(m))
    return torch.from_numpy(pos).to(DEV), torch.from_numpy(conj).to(DEV)


def to_internal(pw, c):
    """Bands as the device entry points take them: (nb, ldc), padded with 0."""
    pos, conj = internal_order(pw)
    out = torch.zeros((c.shape[0], (pw.ngpw + 63) // 64 * 64), dtype=c.dtype, device=DEV)
    out[:, pos] = torch.where(conj, c.conj().resolve_conj(), c)
    return out


def handed_on(case, t):
    """A result as its program keeps it: in the precision that made it."""
    t = torch.as_tensor(t)
    if case["prec"] == "fp64":
        return t
    return t.to(torch.complex64 if t.is_complex() else torch.float32)


def prepare(case, seed):
    s, kind, nb = system_of(case), case["kind"], case["nb"]
    st = dict(case=case, s=s, ctx=KSContext(s.pw, nb, case["prec"]), occ=occupations(nb, seed), tau=positions(s, seed))
    ctx = st["ctx"]
    if kind in ("hpsi", "density"):
        st["c0"] = to_internal(s.pw, bands(s, nb, seed))
        if kind == "hpsi":
            ctx.set_vks(local_potential(s, st["tau"]).cpu().numpy())
            st["c2"] = torch.zeros_like(st["c0"])
        else:
            st["rho"] = torch.zeros(s.pw.n[::-1], dtype=torch.float64, device=DEV)
        torch.cuda.synchronize()
        return st
    ctx.set_species(s.tables)
    if kind != "ortho":
        ctx.set_positions(s.sp, st["tau"])
    if kind == "vks":
        st["rho"] = ion_density(s, st["tau"]).cpu().numpy()
    elif kind == "ortho":
        st["c0"] = moved_bands(s, nb, seed).cpu().numpy()
    else:
        st["c0"] = bands(s, nb, seed).cpu().numpy()
    if kind == "nonloc":
        st["c2"] = bands(s, nb, seed + 1, False).cpu().numpy()
    if kind in ("scf", "md") and case["lowdin"]:
        ctx.set_ortho_method("lowdin")
    return st


def moved_bands(s, nb, seed):
    """Orthonormal bands after an update that spoils their orthonormality."""
    return bands(s, nb, seed) + 0.1 / math.sqrt(nb) * bands(s, nb, seed + 1)


def run(st):
    case, ctx, s = st["case"], st["ctx"], st["s"]
    kind, nb, occ = case["kind"], case["nb"], st["occ"]
    if kind == "hpsi":
        ctx.vpsi_dev(st["c0"].data_ptr(), st["c2"].data_ptr(), occ, nb)
        return handed_on(case, st["c2"])
    if kind == "density":
        ctx._chk(ctx.lib.amdk_density_dev(ctx.h, st["c0"].data_ptr(), lib.dptr(occ), nb,
                                          lib.C.cast(st["rho"].data_ptr(), lib._dp)))
        return handed_on(case, st["rho"])
    if kind == "vks":
        v, e = ctx.vks(st["rho"], case["xc"])
        return {"v": v, **{k: e[k] for k in ("eh", "eloc", "exc", "nelec")}}
    if kind == "ortho":
        return ctx.ortho(st["c0"])
    if kind == "nonloc":
        nl = ctx.fnl(st["c0"])
        return {"nl": handed_on(case, nl), "c2": handed_on(case, ctx.fnonloc(nl, st["c2"], occ))}
    forces = None
    if kind == "md":
        ctx.set_positions(s.sp, st["tau"])
    ctx.wfn_load(st["c0"], occ)
    energies = []
    for it in range(1, case["steps"] + 1):
        if kind == "md" and it == case["steps"]:
            e, forces = ctx.scf_step_tfor(it, case["xc"], True)
        else:
            e = ctx.scf_step(it, case["xc"])
        energies.append([e[k] for k in ENERGIES])
    out = {"c": handed_on(case, ctx.wfn_store()), "energies": handed_on(case, np.array(energies))}
    if forces is not None:
        out["forces"] = handed_on(case, forces)
    return out


ENERGIES = ("etot", "ekin", "estat", "eself", "esr", "eloc", "enl", "exc", "eh", "gemax", "cnorm", "nelec")


def work(case):
    """Bytes and operations that one pass cannot do without."""
    s = system_of(case)
    nb, kind, npw, nr = case["nb"], case["kind"], s.pw.ngpw, s.pw.nr
    n1, n2, n3 = s.pw.n
    band = 16.0 * nb * npw
    # 1D transforms of one band pair: rows of the sphere, columns of its
    # planes, full z columns
    r = np.abs(s.pw.mill_pw).max(axis=0)

    def fft(n):
        return 5.0 * n * math.log2(n)
    pair = math.pi * r[1] * r[2] * fft(n1) + (2 * r[2] + 1) * n1 * fft(n2) + n1 * n2 * fft(n3)
    grid_fft = 2.5 * nr * math.log2(nr)
    pairs = (nb + 1) // 2
    nproj = int(sum(s.tables.nproj[a] for a in s.sp))
    gemm = 4.0 * npw  # of one element of a band product
    if kind == "hpsi":
        return {"bytes": 2 * band + 8.0 * nr, "flops": pairs * (2 * pair + 8.0 * nr)}
    if kind == "density":
        return {"bytes": band + 8.0 * nr, "flops": pairs * (pair + 4.0 * nr)}
    vks = (7 if case["xc"] == "PBE" else 3) * grid_fft + 100.0 * nr
    if kind == "vks":
        return {"bytes": 16.0 * nr, "flops": vks}
    ortho = gemm * nb * nb + nb ** 3
    if kind == "ortho":
        return {"bytes": 2 * band, "flops": ortho}
    if kind == "nonloc":
        return {"bytes": 3 * band + 16.0 * npw * nproj, "flops": 2 * gemm * nproj * nb}
    step = pairs * (3 * pair + 12.0 * nr) + vks + ortho + gemm * nb * (2 * nb + 2 * nproj)
    return {"bytes": case["steps"] * (4 * band + 8.0 * nr) + 2 * band, "flops": case["steps"] * step}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch

def cholesky_orthonormal(c):
    """C U^-1 for S = U^T U, Im c(0) = 0."""
    low = torch.linalg.cholesky(overlap(c, c))
    inv = torch.linalg.solve_triangular(low, torch.eye(len(c), dtype=torch.float64, device=DEV), upper=False)
    c = torch.view_as_complex((inv @ torch.view_as_real(c).flatten(1)).view(*c.shape, 2))
    c[:, 0] = c[:, 0].real.to(c.dtype)
    return c


def overlap(a, b):
    """2 Re <a_i|b_j> - a_i(0) b_j(0) over the half sphere, G = 0 first."""
    ar, br = torch.view_as_real(a).flatten(1), torch.view_as_real(b).flatten(1)
    return 2.0 * (ar @ br.T) - torch.outer(a[:, 0].real, b[:, 0].real)


@functools.lru_cache(maxsize=2)
def _basis(pw):
    n = pw.n

    def index(m):
        m = np.mod(m, n)
        return torch.from_numpy(((m[:, 2] * n[1] + m[:, 1]) * n[0] + m[:, 0]).astype(np.int64)).to(DEV)
    b = {k: (index(m), index(-m), torch.from_numpy(pw.cell.gvec(m)).to(DEV)) for k, m in
         (("pw", pw.mill_pw), ("rho", pw.mill_rho))}
    return b


def to_grid(pw, which, a, b):
    """Real fields given on a half sphere -> a(r) + i b(r), batched, flat."""
    ip, im, _ = _basis(pw)[which]
    g = torch.zeros((a.shape[0], pw.nr), dtype=torch.complex128, device=DEV)
    g[:, im] = a.conj() + 1j * b.conj()
    g[:, ip] = a + 1j * b
    n = pw.n
    return torch.fft.ifftn(g.view(-1, n[2], n[1], n[0]), dim=(1, 2, 3), norm="forward").view(-1, pw.nr)


def from_grid(pw, which, f):
    """a(r) + i b(r) -> the two fields on the half sphere."""
    ip, im, _ = _basis(pw)[which]
    n = pw.n
    g = torch.fft.fftn(f.view(-1, n[2], n[1], n[0]), dim=(1, 2, 3), norm="forward").view(-1, pw.nr)
    p, m = g[:, ip], g[:, im].conj()
    return 0.5 * (p + m), -0.5j * (p - m)


def pair_blocks(pw, c):
    """Blocks of (first band, bands a, bands b) of about 2 GB of grids."""
    step = 2 * max(1, int(2e9 / (16.0 * pw.nr)) // 2)
    for i in range(0, len(c), step):
        a, b = c[i:i + step:2], c[i + 1:i + step:2]
        if len(b) < len(a):
            b = torch.cat([b, torch.zeros_like(a[:1])])
        yield i, a, b


def structure(s, tau, table):
    """sum over atoms of table_s(G) e^{-iG.R} on the density sphere."""
    G = _basis(s.pw)["rho"][2]
    out = torch.zeros(len(G), dtype=torch.complex128, device=DEV)
    t = torch.from_numpy(table).to(DEV)
    tau = torch.as_tensor(tau, dtype=torch.float64, device=DEV)
    for i in range(0, len(tau), 16):
        ph = G @ tau[i:i + 16].T
        out = out + (torch.polar(torch.ones_like(ph), -ph) * t[s.sp[i:i + 16]].T).sum(1)
    return out


def local_potential(s, tau):
    """A self-consistent run's kind of V(r): the ions' wells, screened."""
    v = structure(s, tau, s.tables.vps)
    v = v * 0.5
    v[0] = 0.0
    return to_grid(s.pw, "rho", v[None], torch.zeros_like(v)[None])[0].real.view(s.pw.n[::-1])


def ion_density(s, tau):
    """Valence charge around the ions, and a little everywhere."""
    q = -structure(s, tau, s.tables.rhos)
    rho = to_grid(s.pw, "rho", q[None], torch.zeros_like(q)[None])[0].real.view(s.pw.n[::-1])
    return 0.9 * rho + 0.1 * q[0].real


def plain_density(s, c, occ):
    rho = torch.zeros(s.pw.nr, dtype=torch.float64, device=DEV)
    w = torch.zeros(len(c) + 1, dtype=torch.float64, device=DEV)
    w[:len(c)] = torch.from_numpy(occ).to(DEV) / s.pw.cell.omega
    for i, a, b in pair_blocks(s.pw, c):
        p = to_grid(s.pw, "pw", a, b)
        k = 2 * len(a)
        rho += w[i:i + k:2] @ p.real ** 2 + w[i + 1:i + k:2] @ p.imag ** 2
    return rho


def plain_hpsi(s, c, occ, v):
    """-(f/2) (|G|^2 c + 2 (V psi)(G)), f = 0 counting as 2."""
    G = _basis(s.pw)["pw"][2]
    g2 = (G * G).sum(1)
    f = torch.from_numpy(np.where(occ == 0.0, 2.0, occ)).to(DEV)
    out = torch.empty_like(c)
    for i, a, b in pair_blocks(s.pw, c):
        fa, fb = from_grid(s.pw, "pw", to_grid(s.pw, "pw", a, b) * v.reshape(-1))
        k = min(2 * len(a), len(c) - i)
        out[i:i + k:2] = fa
        out[i + 1:i + k:2] = fb[:k // 2]
    return -0.5 * f[:, None] * (g2 * c + 2.0 * out)


def xc_energy_density(xc, rho, sigma):
    """rho eps_xc: Perdew-Zunger 1981, or PBE 1996 on Perdew-Wang 1992."""
    ex = -0.75 * (3.0 / math.pi) ** (1.0 / 3.0) * rho ** (1.0 / 3.0)
    rs = (3.0 / (4.0 * math.pi * rho)) ** (1.0 / 3.0)
    if xc == "PZ":
        low = -0.1423 / (1.0 + 1.0529 * rs.sqrt() + 0.3334 * rs)
        high = 0.0311 * rs.log() - 0.048 + 0.0020 * rs * rs.log() - 0.0116 * rs
        return rho * (ex + torch.where(rs >= 1.0, low, high))
    beta, gamma, kappa, mu = 0.06672455060314922, (1.0 - math.log(2.0)) / math.pi ** 2, 0.804, 0.2195149727645171
    kf = (3.0 * math.pi ** 2 * rho) ** (1.0 / 3.0)
    s2 = sigma / (4.0 * kf * kf * rho * rho)
    fx = 1.0 + kappa - kappa / (1.0 + mu * s2 / kappa)
    den = 2.0 * 0.0310907 * (7.5957 * rs.sqrt() + 3.5876 * rs + 1.6382 * rs ** 1.5 + 0.49294 * rs * rs)
    ec = -2.0 * 0.0310907 * (1.0 + 0.21370 * rs) * torch.log1p(1.0 / den)
    t2 = sigma / (16.0 * kf / math.pi * rho * rho)
    at2 = (beta / gamma) / torch.expm1(-ec / gamma) * t2
    h = gamma * torch.log1p((beta / gamma) * t2 * (1.0 + at2) / (1.0 + at2 + at2 * at2))
    return rho * (ex * fx + ec + h)


def plain_vks(s, tau, rho, xc):
    """V_KS(r) and eh, eloc, exc, nelec of a density, with its rho(G)."""
    pw = s.pw
    G = _basis(pw)["rho"][2]
    g2 = (G * G).sum(1)
    rho_g = from_grid(pw, "rho", rho.view(1, -1).to(torch.complex128))[0][0]
    eigv, eigr = structure(s, tau, s.tables.vps), structure(s, tau, s.tables.rhos)
    coul = torch.where(g2 > 1e-12, 4.0 * math.pi / g2.clamp_min(1e-12), 0.0)
    vg = coul * (rho_g + eigr) + eigv
    vg[0] = 0.0
    zero = torch.zeros_like(rho_g)
    grad = to_grid(pw, "rho", torch.stack([1j * G[:, 0] * rho_g, 1j * G[:, 2] * rho_g]),
                   torch.stack([1j * G[:, 1] * rho_g, zero]))
    grad = torch.stack([grad[0].real, grad[0].imag, grad[1].real])
    with torch.enable_grad():
        r = rho.reshape(-1).clamp_min(1e-12).requires_grad_()
        sigma = (grad * grad).sum(0).requires_grad_()
        f = xc_energy_density(xc, r, sigma)
        # the reference's smooth cut of the lowest densities (1e-8)
        cut = torch.where(r > 4e-8, 1.0, 1.0 / (1.0 + torch.exp(3.0 * (1.0 - r / 1e-8).clamp_min(-20.0))))
        exc = (torch.where(r > 1e-9, cut, 0.0) * f).sum()
        vr, vs = torch.autograd.grad(exc, (r, sigma), allow_unused=True)
    v2 = 2.0 * vs * grad if vs is not None else 0.0 * grad
    a, b = from_grid(pw, "rho", torch.stack([torch.complex(vr, v2[0]), torch.complex(v2[1], v2[2])]))
    vg = vg + a[0] - 1j * (G[:, 0] * b[0] + G[:, 1] * a[1] + G[:, 2] * b[1])
    v = to_grid(pw, "rho", vg[None], zero[None])[0].real
    rt = rho_g + eigr
    e = dict(eh=(coul * rt.abs() ** 2).sum(), exc=exc.detach() * pw.cell.omega / pw.nr,
             eloc=pw.cell.omega * (2.0 * (eigv * rho_g.conj()).real.sum() - (eigv[0] * rho_g[0].conj()).real),
             nelec=rho.sum() * pw.cell.omega / pw.nr)
    return v.view(pw.n[::-1]), {k: float(x) for k, x in e.items()}, rho_g


def projectors(s, tau):
    """beta (nproj, ngpw), real row coupling D, and the rows' atoms."""
    G, T = _basis(s.pw)["pw"][2], s.tables
    tau = torch.as_tensor(tau, dtype=torch.float64, device=DEV)
    rows, atoms = [], [(a, k) for a in range(len(tau)) for k in range(T.nproj[s.sp[a]])]
    twnl = torch.from_numpy(T.twnl).to(DEV)
    for a, k in atoms:
        ph = G @ tau[a]
        rows.append((-1j) ** int(T.proj_l[s.sp[a], k]) * twnl[s.sp[a], k] * torch.polar(torch.ones_like(ph), -ph))
    d = np.array([[T.dmat[s.sp[a], k, q] if a == b else 0.0 for b, q in atoms] for a, k in atoms])
    return torch.stack(rows), torch.from_numpy(d).to(DEV)


def ion_pairs(s, tau):
    """Short-range ion-ion energy, nearest images in a cubic box."""
    z = torch.from_numpy(s.tables.zv[s.sp]).to(DEV)
    i, j = torch.triu_indices(len(z), len(z), 1, device=DEV)
    box = float(s.pw.cell.a[0, 0])
    d = tau[i] - tau[j]
    d = d - box * torch.round(d.detach() / box)
    r = d.norm(dim=1)
    x = r / (math.sqrt(2.0) * RAGGIO)
    return torch.where(x <= 20.0, z[i] * z[j] * torch.erfc(x) / r, 0.0).sum()


def plain_forces(s, tau, c, occ, rho_g):
    """-dE/dR at fixed bands: local, Hartree with the ions, nonlocal, ion-ion."""
    pw, om = s.pw, s.pw.cell.omega
    G = _basis(pw)["rho"][2]
    g2 = (G * G).sum(1)
    coul = torch.where(g2 > 1e-12, 4.0 * math.pi / g2.clamp_min(1e-12), 0.0)
    f = torch.zeros((len(tau), 3), dtype=torch.float64, device=DEV)
    vh = coul * (rho_g + structure(s, tau, s.tables.rhos)).conj()
    vps, rhos = torch.from_numpy(s.tables.vps).to(DEV), torch.from_numpy(s.tables.rhos).to(DEV)
    t = torch.as_tensor(tau, dtype=torch.float64, device=DEV)
    for a in range(len(tau)):
        ph = G @ t[a]
        x = (rhos[s.sp[a]] * vh + vps[s.sp[a]] * rho_g.conj()) * torch.polar(torch.ones_like(ph), -ph)
        f[a] = -2.0 * om * (G * x.imag[:, None]).sum(0)
    beta, d = projectors(s, tau)
    rows = [a for a in range(len(tau)) for _ in range(s.tables.nproj[s.sp[a]])]
    w = torch.from_numpy(occ).to(DEV)
    dn = d @ overlap(beta, c)
    for k in range(3):
        part = -2.0 * (overlap(-1j * _basis(pw)["pw"][2][:, k] * beta, c) * dn * w).sum(1)
        f[:, k].index_add_(0, torch.tensor(rows, device=DEV), part)
    with torch.enable_grad():
        t = t.requires_grad_()
        g, = torch.autograd.grad(ion_pairs(s, t), t)
    return f - g


def plain_run(case, s, tau, occ, c):
    """The SCF steps of a run: bands, energies and the last step's forces."""
    pw, T = s.pw, s.tables
    G = _basis(pw)["pw"][2]
    g2 = (G * G).sum(1)
    f = torch.from_numpy(occ).to(DEV)
    beta, d = projectors(s, tau)
    zv = T.zv[s.sp]
    eself = float((zv * zv).sum()) / RAGGIO / math.sqrt(2.0 * math.pi)
    esr = float(ion_pairs(s, torch.from_numpy(tau).to(DEV)))
    count = np.bincount(s.sp, minlength=T.nsp)
    k = 0.5 * g2 + float(sum(count[i] * T.vps[i][0] for i in range(T.nsp)))
    for i in range(T.nsp):
        for q in range(T.nproj[i]):
            k = k + count[i] * float(T.wsg[i, q]) * torch.from_numpy(T.twnl[i, q]).to(DEV) ** 2
    precon = 1.0 / k.clamp_min(0.5)
    energies, direction, last, forces = [], 0.0, 1.0, None
    for it in range(1, case["steps"] + 1):
        v, e, rho_g = plain_vks(s, tau, plain_density(s, c, occ), case["xc"])
        nl = overlap(beta, c)
        c2 = plain_hpsi(s, c, occ, v) - ((d @ nl) * f).T.to(c.dtype) @ beta
        c2 = c2 - overlap(c2, c).T.to(c.dtype) @ c
        c2[:, 0] = c2[:, 0].real.to(c.dtype)
        if case["kind"] == "md" and it == case["steps"]:
            forces = plain_forces(s, tau, c, occ, rho_g)
        e.update(ekin=float((f[:, None] * g2 * c.abs() ** 2).sum()), enl=float(((nl * (d @ nl)) * f).sum()), esr=esr, eself=eself)
        e["estat"] = e["eh"] * pw.cell.omega + esr - eself
        e["etot"] = e["enl"] + e["eloc"] + e["ekin"] + e["exc"] + e["estat"]
        norm = 2.0 * c2.abs() ** 2
        norm[:, 0] *= 0.5
        e.update(gemax=float(c2.abs().max()), cnorm=math.sqrt(float(norm.sum()) / norm.numel()))
        energies.append([e[key] for key in ENERGIES])
        p = c2 * precon / f[:, None]
        norm = 2.0 * p.abs() ** 2
        norm[:, 0] *= 0.5
        gg = float(norm.sum())
        forget = 0.0 if it == 1 else 0.60 if it <= 10 else 0.91 if it <= 20 else 0.95
        direction = p + forget * gg / last * direction
        last = gg
        c = c + 25.0 / 400.0 * direction
        if case["lowdin"] and it > 1:
            w, u = torch.linalg.eigh(overlap(c, c))
            c = ((u / w.sqrt()) @ u.T).to(c.dtype) @ c
            c[:, 0] = c[:, 0].real.to(c.dtype)
        else:
            c = cholesky_orthonormal(c)
    return c, np.array(energies), forces


@torch.no_grad()
def exact(case, seed):
    s, kind, nb = system_of(case), case["kind"], case["nb"]
    occ, tau = occupations(nb, seed), positions(s, seed)
    if kind == "hpsi":
        return to_internal(s.pw, plain_hpsi(s, bands(s, nb, seed), occ, local_potential(s, tau)))
    if kind == "density":
        return plain_density(s, bands(s, nb, seed), occ).view(s.pw.n[::-1])
    if kind == "vks":
        v, e, _ = plain_vks(s, tau, ion_density(s, tau), case["xc"])
        return {"v": v, **e}
    if kind == "ortho":
        return cholesky_orthonormal(moved_bands(s, nb, seed))
    if kind == "nonloc":
        c0, c2 = bands(s, nb, seed), bands(s, nb, seed + 1, False)
        beta, d = projectors(s, tau)
        nl = overlap(beta, c0)
        return {"nl": nl, "c2": c2 - ((d @ nl) * torch.from_numpy(occ).to(DEV)).T.to(c2.dtype) @ beta}
    c, e, f = plain_run(case, s, tau, occ, bands(s, nb, seed))
    return {"c": c, "energies": e, **({} if f is None else {"forces": f})}
