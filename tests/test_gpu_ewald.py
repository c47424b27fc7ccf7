"""The Ewald blocks and pair sums of the device against the lattice sums written out in numpy:
every radius, both methods, cutoffs, unequal radii, and system sizes on either side of the 64-bead
tiles and of the number of workgroups a tile pair is split into."""
import math

import numpy as np
import pytest
from scipy.special import erfc

from bd_box_amd import workloads as wl

pytestmark = pytest.mark.gpu
KB8, KB6, SP = 0.00007903031804378703, 0.00010537375739171604, 1.77245385090551602729
PIF = float(np.float32(math.pi))


@pytest.fixture(scope="module")
def api():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from bd_box_amd import system
    return system


def _spheres(N, phi, seed, method, R=2, hydro="geyer"):
    rng = np.random.default_rng(seed)
    L = float(np.float32((N * 4.0 / 3.0 * math.pi * 25.0 ** 3 / phi) ** (1 / 3)))
    m = math.ceil(N ** (1 / 3) - 1e-9)
    site = rng.choice(m ** 3, N, replace=False)
    xyz = (np.stack([site // (m * m), site // m % m, site % m], 1) + 0.5) * (L / m) - L / 2
    xyz += rng.uniform(-0.3, 0.3, (N, 3)) * max(0.0, L / m - 50.0)
    a = rng.choice([20.0, 25.0], N)
    s = wl.System(np.concatenate([xyz, a[:, None]], 1), np.zeros(N), np.tile([25.0, 1.0], (N, 1)),
                  np.zeros((0, 2), np.int32), np.zeros((0, 3)))
    P = wl.parse_params(wl.chain_params(bc="periodic", xbox=L, ybox=L, zbox=L, hydro=hydro, ewald_method=method,
                                        ewald_real=R, ewald_recip=R, elec="no", cutoff_lj=-1, dt=1.0,
                                        rand_seed=seed))
    return s, P


def _sphere(R):
    return [(h, f, g) for h in range(-R, R + 1) for f in range(-R, R + 1) for g in range(-R, R + 1)
            if h * h + f * f + g * g <= R * R]


def _plain(s, P, ext=None):
    """D of non-overlapping beads; ext = (alpha scale, R_real, R_recip, r_cut)."""
    N, L = s.N, P.box
    pii = KB6 * P.T / (P.visc * P.vfactor)
    d = s.coord[None, :, :3] - s.coord[:, None, :3]
    a = s.coord[:, 3]
    sg = 0.5 * (a[:, None] ** 2 + a[None, :] ** 2)
    eye = np.eye(3)
    B = np.zeros((N, N, 3, 3))
    beenakker = P.ewald_method == 1
    scale, Rr, Rk, cut = ext or (1.0, P.ewald_real, P.ewald_real, 0.0)
    if ext:
        d = d - L * np.rint(d / L)
    al = scale * SP / L if beenakker else P.ewald_alpha
    u = 1.0 if beenakker else 1.0 / L
    for h, f, g in _sphere(Rr):
        x = d * u + (L * u) * np.array([h, f, g], float)
        r2 = (x * x).sum(-1)
        ok = (r2 != 0) & ((r2 <= cut * cut) if cut else True)
        r2 = np.where(ok, r2, 1.0)
        r, eg = np.sqrt(r2), np.exp(-al * al * r2)
        ec = erfc(al * r)
        if beenakker:
            c1 = eg / SP * (al * sg / r2 + 14 * al ** 3 * sg - 4.5 * al - 20 * al ** 5 * sg * r2 + 3 * al ** 3 * r2 +
                            4 * al ** 7 * sg * r2 * r2) + ec * (0.75 / r + 0.5 * sg / r ** 3)
            c2 = eg / SP * (-3 * al * sg / r2 - 2 * al ** 3 * sg + 1.5 * al + 16 * al ** 5 * sg * r2 -
                            3 * al ** 3 * r2 - 4 * al ** 7 * sg * r2 * r2) + ec * (0.75 / r - 1.5 * sg / r ** 3)
        else:
            m1 = 0.5641895835
            so, sq = ec / r, (ec + 2 * al * r * m1 * eg) / r ** 3
            pO, pQ = 0.75 / L, 0.5 * sg / L ** 3
            c1 = pO * so + pQ * sq
            c2 = pO * (so + 2 * al * m1 * eg) + pQ * (-3 * sq - 4 * al ** 3 * m1 * eg)
        B += np.where(ok, c1, 0)[..., None, None] * eye
        B += np.where(ok, c2 / r2, 0)[..., None, None] * x[..., :, None] * x[..., None, :]
    for h, f, g in _sphere(Rk):
        s2 = float(h * h + f * f + g * g)
        if s2 == 0:
            continue
        e = np.array([h, f, g]) / math.sqrt(s2)
        c = np.cos(2 * PIF * (d / L) @ np.array([h, f, g], float))
        if beenakker:
            k2 = s2 * 4 * math.pi ** 2 / L ** 2 if ext else s2 * 4 * PIF ** 2
            q = k2 / (al * al)
            G = (1 + q / 4 * (1 + q / 2)) * 6 * math.pi * math.exp(-q / 4) / k2
            B += ((1 - sg * k2 / 3) * G * c / L ** 3)[..., None, None] * (eye - np.outer(e, e))
        else:
            mp = float(-np.float32(math.pi) * np.float32(math.pi)) / (al * al)
            g1, g2 = 2 * math.exp(mp * s2) / (PIF * s2), 4 * PIF * math.exp(mp * s2)
            B += (0.75 / L * g1 * c)[..., None, None] * eye
            B += ((0.75 / L * g1 * (-1 + mp * s2) + 0.5 * sg / L ** 3 * g2) * c)[..., None, None] * np.outer(e, e)
    B *= pii
    if beenakker:
        self_ = pii / a + pii * (-6 * al / SP + 40 * al ** 3 * a * a / (3 * SP))
    else:
        m1, x = 0.5641895835, al * a / L
        self_ = pii / a - pii * (0.75 / L * 1.5 * al * a * m1 / L + 0.5 * a * a / L ** 3 * (x ** 3 * m1 / 3))
    for i in range(N):
        B[i, i] = np.diag(np.diag(B[i, i])) + self_[i] * eye
    return B.transpose(0, 2, 1, 3).reshape(3 * N, 3 * N)


@pytest.mark.parametrize("method,R,ext", [
    ("beenakker", 0, None), ("beenakker", 2, None), ("beenakker", 5, None), ("smith", 0, None), ("smith", 1, None),
    ("smith", 2, None), ("smith", 5, None), ("beenakker", 2, (1.25, 3, 3, 2.0)), ("beenakker", 2, (0.8, 5, 1, 0.0)),
    ("beenakker", 2, (1.7, 2, 5, 1.3)), ("beenakker", 2, (1.0, 4, 0, 0.0)), ("beenakker", 2, (3.0, 0, 4, 0.4))])
def test_ewald_tensor_vs_numpy(api, method, R, ext):
    """FP64 within 2e-13 of the largest entry: the sums hold up to 515 images of entries below it,
    each within a few 2^-53.  Mixed: the entries and the image terms are rounded to 2^-24, a few
    images of size 1 and many small ones: 1e-6."""
    s, P = _spheres(50, 0.15, 3, method, R)
    if ext:
        ext = ext[:3] + (ext[3] * P.box,)
    ref = _plain(s, P, ext)
    print("ewald tensor", method, R, ext, flush=True)
    for prec, tol in ((api.FP64, 2e-13), (api.MIXED, 1e-6)):
        b = api.BDSystem(s, P, precision=prec)
        if ext:
            b.set_ewald_split(ext[0], ext[1], ext[2], r_cut=ext[3])
        err = np.abs(b.compute_D() - ref).max() / np.abs(ref).max()
        assert err <= tol, (prec, err)
        b.close()


@pytest.mark.parametrize("N", [1, 2, 63, 64, 65, 130, 343, 700, 1100])
@pytest.mark.parametrize("method", ["beenakker", "smith"])
def test_pair_sums_vs_tensor(api, N, method):
    """D.F summed over blocks on the fly equals the assembled tensor times the forces for every
    split of the tile pairs: FP64 to 1e-12; mixed, whose assembled entries are the same blocks
    rounded to 2^-24, to 1e-6 (2-norm)."""
    s, P = _spheres(N, 0.1, 11, method)
    F = np.random.default_rng(N).normal(size=3 * N)
    print("pair sums", method, N, flush=True)
    for prec, tol in ((api.FP64, 1e-12), (api.MIXED, 1e-6)):
        b = api.BDSystem(s, P, precision=prec)
        b.set_forces(F)
        ref = P.dt / (0.001986248532617 * P.T) * (b.compute_D() @ F)
        err = np.linalg.norm(b.compute_Rf() - ref) / np.linalg.norm(ref)
        assert err <= tol, (prec, err)
        b.close()


@pytest.mark.parametrize("box", [1000.1, 999.9, 850.3, 640.0])
@pytest.mark.parametrize("R,ext", [(2, None), (3, None), (4, None), (5, None), (2, (1.25, 3, 3, 0.0)),
                                   (2, (0.8, 4, 2, 0.0)), (2, (1.0, 5, 1, 2.1))])
def test_ewald_tensor_any_box(api, box, R, ext):
    """Box edges with no short binary form (a .prm file's are rounded to 24 bits, a caller's own are
    not), where R L is inexact: a bead's own central image is left out all the same.  The bounds
    of test_ewald_tensor_vs_numpy."""
    s, P = _spheres(40, 0.05, 5, "beenakker", R)
    s.coord[:, :3] *= box / P.box
    P.box = box
    if ext:
        ext = ext[:3] + (ext[3] * box,)
    ref = _plain(s, P, ext)
    print("ewald tensor", box, R, ext, flush=True)
    for prec, tol in ((api.FP64, 2e-13), (api.MIXED, 1e-6)):
        b = api.BDSystem(s, P, precision=prec)
        if ext:
            b.set_ewald_split(ext[0], ext[1], ext[2], r_cut=ext[3])
        err = np.abs(b.compute_D() - ref).max() / np.abs(ref).max()
        assert err <= tol, (prec, err)
        b.close()


def _beenakker_long(s, P, R):
    """Off-diagonal blocks of the reference's split (no reciprocal terms) in extended precision."""
    LD = np.longdouble
    sp, kt = LD("1.77245385090551602729816748334114518"), LD(KB6 * P.T / (P.visc * P.vfactor))
    al, sg = LD(SP / P.box), (s.coord[:, None, 3] ** 2 + s.coord[None, :, 3] ** 2).astype(LD) / 2
    d = s.coord[None, :, :3].astype(LD) - s.coord[:, None, :3]
    B = np.zeros((s.N, s.N, 3, 3), LD)
    off = ~np.eye(s.N, dtype=bool)
    for hfg in _sphere(R):
        x = d + LD(P.box) * np.array(hfg, LD)
        r2 = np.where(off, (x * x).sum(-1), 1)
        r = np.sqrt(r2)
        y = al * r
        eg = np.exp(-y * y) / sp
        term, erf = y, y   # erf y = 2 exp(-y^2) / sqrt(pi) sum (2 y^2)^n y / (2 n + 1)!!
        for n in range(1, 260):
            term = term * (2 * y * y) / (2 * n + 1)
            erf = erf + term
        ec = 1 - 2 * eg * erf
        c1 = eg * (al * sg / r2 + 14 * al ** 3 * sg - LD(4.5) * al - 20 * al ** 5 * sg * r2 + 3 * al ** 3 * r2 +
                   4 * al ** 7 * sg * r2 * r2) + ec * (LD(0.75) / r + LD(0.5) * sg / (r * r2))
        c2 = eg * (-3 * al * sg / r2 - 2 * al ** 3 * sg + LD(1.5) * al + 16 * al ** 5 * sg * r2 - 3 * al ** 3 * r2 -
                   4 * al ** 7 * sg * r2 * r2) + ec * (LD(0.75) / r - LD(1.5) * sg / (r * r2))
        B += c1[..., None, None] * np.eye(3, dtype=LD) + (c2 / r2)[..., None, None] * x[..., :, None] * x[..., None, :]
    return kt * B, off


@pytest.mark.parametrize("seed", [3, 4])
def test_ewald_rounding(api, seed):
    """515 images in FP64 against extended precision: an entry's own rounding and as much again from
    the sum, each uniform in half the largest entry's unit 2^-52: rms 2^-53 sqrt(2 / 3)."""
    s, P = _spheres(50, 0.15, seed, "beenakker", 5)
    ref, off = _beenakker_long(s, P, 5)
    print("ewald rounding", seed, flush=True)
    b = api.BDSystem(s, P, precision=api.FP64)
    D = b.compute_D()
    b.close()
    err = np.abs(D.reshape(50, 3, 50, 3).transpose(0, 2, 1, 3) - ref)[off].max((1, 2)) / np.abs(D).max()
    assert np.sqrt((err ** 2).mean()) <= 2.0 ** -53 * np.sqrt(2 / 3), float(np.sqrt((err ** 2).mean()))


@pytest.mark.parametrize("R", [0, 2])
def test_smith_tensor_shows_nan(api, R):
    """A coordinate that is not a number is one in every Smith block of its bead, also where no
    reciprocal vector carries it; the other beads' blocks are as without it."""
    s, P = _spheres(20, 0.05, 7, "smith", R)
    print("smith nan", R, flush=True)
    for prec in (api.FP64, api.MIXED):
        b = api.BDSystem(s, P, precision=prec)
        ref = b.compute_D()
        c = s.coord.copy()
        c[4, 1] = np.nan
        b.set_coords(c)
        D = b.compute_D().reshape(20, 3, 20, 3)
        b.close()
        rest = [k for k in range(20) if k != 4]
        assert np.isnan(D[4][:, rest]).all() and np.isnan(D[rest][:, :, 4]).all()
        assert np.array_equal(D[np.ix_(rest, range(3), rest, range(3))], ref.reshape(20, 3, 20, 3)[np.ix_(rest, range(3), rest, range(3))])
