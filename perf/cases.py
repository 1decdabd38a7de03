"""Timed cases of the surface Green's function path, through ``SurfaceGF``.

Each case is one call that a surface-state calculation makes, host arrays in
and host arrays out, on a context that already holds the model (a calculation
sets its model once and then runs its path, plane or batch on it).  The
models are the seeded synthetic recipes of ``wannier_tools_amd.model``; the
orders follow the workloads of ``bench.py`` and the reference's examples.

Kinds:
  green  one ``surfgreen_1985`` instance (full G_LL, G_RR, G_B)
  ham    ``ham_qlayer2qlayer`` along a k path
  grid   ``spectral_grid``: k path x energies, optionally with spin traces
  batch  ``spectral_batch``: instances with their own k, omega and eta
  plane  ``spectral_grid`` on a k plane at omega = 0 (divisor pi)
  qpi    ``kplane_autocorrelation`` of a plane's spectral fields
  jdos   ``kpath_jdos`` of a path's spectral fields
"""
import math

import numpy as np
import torch

from wannier_tools_amd import model as M
from wannier_tools_amd.surface import SurfaceGF

# Iterations a decimation takes at eta of 1e-3 eV or so (the mean over the
# Ndim 72 benchmark grid is 16.8); only for the operation counts.
ITERATIONS = 17
ITERMAX = M.DECIMATION_ITERMAX


def listed():
    return [
        # a Fortran program calling the drop-in surfgreen_1985 per (k, omega)
        {"name": "green_72", "kind": "green", "nw": 36, "np": 2, "rmax": 3, "spin": 0},
        # H00(k), H01(k) of a path for a caller's own post-processing
        {"name": "ham_72", "kind": "ham", "nw": 36, "np": 2, "rmax": 3, "spin": 0, "nk": 257},
        # a four-band spinful model (BHZ-like), surface states with spin texture
        {"name": "grid_8_spin", "kind": "grid", "nw": 4, "np": 2, "rmax": 2, "spin": 1,
         "nk": 101, "nomega": 400, "eta_ev": 1e-3},
        # the 8-orbital model's full path x energy window
        {"name": "grid_16", "kind": "grid", "nw": 8, "np": 2, "rmax": 1, "spin": 0,
         "nk": 201, "nomega": 401, "eta_ev": 1e-3},
        # scattered (k, omega, eta) points of a 16-orbital model
        {"name": "batch_32", "kind": "batch", "nw": 16, "np": 2, "rmax": 2, "spin": 0,
         "nk": 500, "ninst": 5000},
        # a real material's size (30 spinful orbitals, two layers), a quick-look grid
        {"name": "grid_60_spin", "kind": "grid", "nw": 30, "np": 2, "rmax": 3, "spin": 1,
         "nk": 22, "nomega": 51, "eta_ev": 1e-3},
        # the headline model, a publication-sized part of its grid
        {"name": "grid_72", "kind": "grid", "nw": 36, "np": 2, "rmax": 3, "spin": 0,
         "nk": 64, "nomega": 128, "eta_ev": 1e-3},
        # three layers of the same orbitals, scattered points
        {"name": "batch_108", "kind": "batch", "nw": 36, "np": 3, "rmax": 2, "spin": 0,
         "nk": 100, "ninst": 1500},
        # the largest member of the mixed set, a small scattered batch
        {"name": "batch_216", "kind": "batch", "nw": 72, "np": 3, "rmax": 2, "spin": 0,
         "nk": 60, "ninst": 300},
        # a spinful 144-orbital constant-energy map on a coarse plane
        {"name": "plane_288", "kind": "plane", "nw": 144, "np": 2, "rmax": 3, "spin": 1,
         "nk1": 21, "nk2": 21, "eta_ev": 5e-4},
        # QPI (jsdos: spectral weight and three spin fields) of a k plane
        {"name": "qpi_257", "kind": "qpi", "nkx": 257, "nky": 257, "m1": 256, "m2": 256,
         "nfield": 4},
        # k-path joint density of states (left, right, bulk and one more field)
        {"name": "jdos_512", "kind": "jdos", "nk": 512, "nomega": 512, "nfield": 4},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["green", "ham", "grid", "grid", "grid", "batch", "batch", "plane", "qpi",
                       "jdos"])
    if kind == "qpi":
        nkx, nky = _log_int(rng, 9, 257), _log_int(rng, 9, 257)
        nfield = rng.choice([1, 4])
        cut = 1 if nfield == 1 else rng.choice([1, 2])
        return {"kind": kind, "nkx": nkx, "nky": nky, "m1": nkx - cut, "m2": nky - cut,
                "nfield": nfield}
    if kind == "jdos":
        return {"kind": kind, "nk": _log_int(rng, 21, 512), "nomega": _log_int(rng, 21, 512),
                "nfield": rng.randint(1, 4)}
    np_ = rng.randint(1, 3)
    spin = rng.choice([0, 1])
    top = {"green": 288, "ham": 144}.get(kind, 300)
    nw = max(2, _log_int(rng, 4, top) // np_)
    if spin and nw % 2:
        nw += 1
    n = nw * np_
    base = {"kind": kind, "nw": nw, "np": np_, "rmax": rng.choice([1, 2, 3]) if nw <= 72 else 2,
            "spin": spin}
    if kind == "green":
        return base
    if kind == "ham":
        return dict(base, nk=_log_int(rng, 1, 513))
    # at most the work of 350 instances of order 288; small orders are bound
    # by their count
    most = int(min(80000, 350 * (288.0 / n) ** 3))
    ninst = _log_int(rng, max(1, most // 64), most)
    if kind == "batch":
        return dict(base, nk=max(1, min(500, ninst // 3)), ninst=ninst)
    if kind == "plane":
        nk1 = max(3, int(math.sqrt(ninst * rng.uniform(0.5, 1.0))))
        return dict(base, nk1=nk1 | 1, nk2=max(3, ninst // nk1) | 1 if nk1 * nk1 > 9 else 3,
                    eta_ev=10.0 ** rng.uniform(-3.3, -2.0))
    nk = max(2, min(513, int(ninst ** rng.uniform(0.3, 0.7))))
    return dict(base, nk=nk, nomega=max(1, ninst // nk), eta_ev=10.0 ** rng.uniform(-3.3, -2.0))


def _model(case, seed):
    """(irvec, hr) of the case's synthetic model, in Hartree."""
    if case["nw"] <= 8 and case["rmax"] == 1:
        sigma, decay = 0.3, M.decay_l1
    else:
        sigma, decay = 0.5, M.decay_l2(1.5)
    return M.synthetic_model(case["nw"], case["rmax"], sigma, decay, seed=seed,
                             soc_sigma=0.05 if case["spin"] else 0.0).surface_cell()


def _points(case, seed):
    """k points, and the energies and broadenings (Hartree) of the case."""
    rng = np.random.default_rng([seed, 1])
    kind = case["kind"]
    if kind == "green":
        return (rng.uniform(-0.5, 0.5, (1, 2)), np.array([rng.uniform(-1.0, 1.0)]) * M.EV2HARTREE,
                1e-3 * M.EV2HARTREE)
    if kind == "batch":
        return (rng.uniform(-0.5, 0.5, (case["nk"], 2)),
                rng.uniform(-1.0, 1.0, case["ninst"]) * M.EV2HARTREE,
                10.0 ** rng.uniform(-3.0, -2.0, case["ninst"]) * M.EV2HARTREE)
    if kind == "plane":
        k, _, _ = M.kplane_slab((-0.5, -0.5), (1.0, 0.0), (0.0, 1.0), case["nk1"], case["nk2"])
        return k, np.array([0.0]), case["eta_ev"] * M.EV2HARTREE
    k = M.kpath_slab([((-0.5, 0.0), (0.5, 0.0))], max(2, case["nk"]))[:case["nk"]]
    # a path off the time-reversal invariant line, another one for every seed
    k = k + rng.uniform(-0.05, 0.05, (1, 2))
    if kind == "ham":
        return k, None, None
    return k, M.omega_grid(-1.0, 1.0, case["nomega"]) * M.EV2HARTREE, case["eta_ev"] * M.EV2HARTREE


def _fields(case, seed):
    """Spectral-weight-like fields: positive peaks on a smooth background, and
    signed spin fields where there are four on a plane."""
    rng = np.random.default_rng([seed, 2])
    if case["kind"] == "qpi":
        shape = (case["nfield"], case["nkx"], case["nky"])
    else:
        shape = (case["nfield"], case["nk"], case["nomega"])
    a = rng.uniform(0.0, 1.0, shape) ** 4
    if case["kind"] == "qpi" and case["nfield"] > 1:
        a[1:] *= rng.uniform(-1.0, 1.0, (case["nfield"] - 1,) + shape[1:])
    return a


def _k_index(case, seed):
    return np.random.default_rng([seed, 3]).integers(0, case["nk"], case["ninst"]).astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "gf": SurfaceGF(0)}
    gf = state["gf"]
    if kind in ("qpi", "jdos"):
        state["fields"] = _fields(case, seed)
        return state
    irvec, hr = _model(case, seed)
    gf.set_model_arrays(case["nw"], case["np"], irvec, hr)
    if kind == "grid" and case["spin"]:
        gf.set_spin_traces("surfstat")
    state["k"], state["w"], state["eta"] = _points(case, seed)
    if kind == "batch":
        state["k_index"] = _k_index(case, seed)
    if kind == "green":
        # H00, H01 as the caller's own arrays
        h00, h01 = gf.ham_qlayer2qlayer(state["k"][0])
        state["h00"], state["h01"] = np.asfortranarray(h00), np.asfortranarray(h01)
    return state


def run(state):
    case, gf = state["case"], state["gf"]
    kind = case["kind"]
    if kind == "green":
        return gf.surfgreen_1985(float(state["w"][0]), state["h00"], state["h01"], state["eta"])
    if kind == "ham":
        return gf.ham_qlayer2qlayer(state["k"])
    if kind == "batch":
        return gf.spectral_batch(state["k"], state["k_index"], state["w"], state["eta"])
    if kind == "plane":
        return gf.spectral_grid(state["k"], state["w"], state["eta"], divisor=M.REF_PI)
    if kind == "grid":
        out = gf.spectral_grid(state["k"], state["w"], state["eta"])
        return out + gf.spin_download() if case["spin"] else out
    if kind == "qpi":
        return gf.kplane_autocorrelation(state["fields"], case["m1"], case["m2"])
    return gf.kpath_jdos(state["fields"])


def _instances(case):
    kind = case["kind"]
    if kind == "green":
        return 1
    if kind == "batch":
        return case["ninst"]
    if kind == "plane":
        # kplane_slab rounds up to odd
        return (case["nk1"] | 1) * (case["nk2"] | 1)
    return case["nk"] * case["nomega"]


def work(case):
    kind = case["kind"]
    if kind == "qpi":
        plane = case["nkx"] * case["nky"]
        # one forward transform per field, one back: the sum is a cyclic correlation
        m = case["m1"] * case["m2"]
        return {"bytes": 8 * (case["nfield"] + 1) * plane,
                "flops": (case["nfield"] + 1) * 5 * m * max(1.0, math.log2(m))}
    if kind == "jdos":
        rows = case["nfield"] * case["nomega"]
        return {"bytes": 16 * rows * case["nk"], "flops": 1.5 * rows * case["nk"] ** 2}
    nw, np_ = case["nw"], case["np"]
    n = nw * np_
    model = 16 * (2 * case["rmax"] + 1) ** 3 * nw * nw
    if kind == "green":
        return {"bytes": 5 * 16 * n * n, "flops": (56 * ITERATIONS + 24) * n ** 3}
    # the Fourier sum over the R3 slots that H00 and H01 use
    slots = sum(1 for d in range(-(np_ - 1), 2 * np_) if abs(d) <= case["rmax"])
    nk = (case["nk1"] | 1) * (case["nk2"] | 1) if kind == "plane" else case["nk"]
    fourier = 8 * nk * slots * (2 * case["rmax"] + 1) ** 2 * nw * nw
    if kind == "ham":
        return {"bytes": model + nk * 2 * 16 * n * n, "flops": fourier}
    ninst = _instances(case)
    outs = 3 * 8 + 2 * 4 + (6 * 8 if kind == "grid" and case["spin"] else 0)
    return {"bytes": model + nk * 16 + ninst * (outs + (20 if kind == "batch" else 0)),
            "flops": fourier + ninst * (56 * ITERATIONS + 24) * n ** 3}


def tolerance(case):
    kind = case["kind"]
    if kind in ("qpi", "jdos", "ham"):
        # plain double sums
        return {"rel": 1e-13, "max": 1e-11}
    # The decimation squares its couplings every iteration and amplifies
    # rounding by up to 1e9 near band edges at small eta: single instances of
    # two correct FP64 implementations differ by up to 1e-7 of their value.
    # An iteration count changes by one where the sum meets the threshold.
    # Against torch's inverses and products the path
    # shows 1e-12 to 2e-8 in the 2-norm, the Ndim 288 plane the most.
    return {"rel": 8e-8, "max": 1e-5, "differ": 1e-3}


# ---- the same numbers in plain torch / numpy ---------------------------------
def _hamiltonians(case, irvec, hr, kpts):
    """H00, H01 of every k point, (nk, n, n) complex128."""
    nw, np_ = case["nw"], case["np"]
    n, nk = nw * np_, kpts.shape[0]
    h00 = np.zeros((nk, n, n), dtype=np.complex128)
    h01 = np.zeros((nk, n, n), dtype=np.complex128)
    for d in range(-(np_ - 1), 2 * np_):
        sel = np.nonzero(irvec[:, 2] == d)[0]
        if sel.size == 0:
            continue
        phase = np.exp(1j * (2.0 * M.REF_PI) * (kpts @ irvec[sel, :2].T.astype(np.float64)))
        hij = (phase @ hr[sel].reshape(sel.size, -1)).reshape(nk, nw, nw)
        for i in range(np_):
            j = i + d
            if 0 <= j < np_:
                h00[:, i * nw:(i + 1) * nw, j * nw:(j + 1) * nw] = hij
            elif np_ <= j < 2 * np_:
                j -= np_
                h01[:, i * nw:(i + 1) * nw, j * nw:(j + 1) * nw] = hij
    return h00, h01


def _decimate(h00, h01, z):
    """G_LL, G_RR, G_B and iteration counts of a batch (torch complex128)."""
    n = h00.shape[-1]
    eye = torch.eye(n, dtype=h00.dtype, device=h00.device)
    zi = z[:, None, None] * eye
    es, et, ei = h00.clone(), h00.clone(), h00.clone()
    al, be = h01.clone(), h01.mH.contiguous()
    iters = torch.full((h00.shape[0],), ITERMAX, dtype=torch.int32, device=h00.device)
    live = torch.arange(h00.shape[0], device=h00.device)
    for it in range(1, ITERMAX + 1):
        g = torch.linalg.inv(zi[live] - ei[live])
        a, b = al[live], be[live]
        m1, m2 = a @ g, b @ g
        d1, d2 = m1 @ b, m2 @ a
        es[live] += d1
        et[live] += d2
        ei[live] += d1 + d2
        a, b = m1 @ a, m2 @ b
        al[live], be[live] = a, b
        done = a.abs().sum(dim=(1, 2)) <= M.DECIMATION_ACCURACY
        iters[live[done]] = it
        live = live[~done]
        if live.numel() == 0:
            break
    inv = torch.linalg.inv
    return inv(zi - es), inv(zi - et), inv(zi - ei), iters


def _spin(g, nw, n):
    """-sum over the top orbitals 1..nw of Im (G sigma_c)(io, io), c = x, y, z."""
    h = nw // 2
    up = torch.arange(h, device=g.device)
    dn = up + h
    gud, gdu = g[:, up, dn], g[:, dn, up]
    sx = -(gud.imag + gdu.imag).sum(dim=1)
    sy = -(gud.real - gdu.real).sum(dim=1)
    d = torch.diagonal(g, dim1=1, dim2=2).imag
    sz = -(d[:, up] - d[:, dn]).sum(dim=1)
    return torch.stack([sx, sy, sz])


def exact(case, seed):
    kind = case["kind"]
    if kind == "jdos":
        a = _fields(case, seed)
        nk = case["nk"]
        h = (nk - 1) // 2
        odd = 2 * h + 1
        size = 2 * odd
        f = np.fft.rfft(a[:, :odd], size, axis=1)
        full = np.fft.irfft(np.conj(f) * f, size, axis=1)
        out = np.empty_like(a)
        out[:] = full[:, (np.arange(nk) + 1 - h) % size]
        return out
    if kind == "qpi":
        a, m1, m2 = _fields(case, seed), case["m1"], case["m2"]
        i1, i2 = np.arange(case["nkx"]) % m1, np.arange(case["nky"]) % m2
        e = np.zeros((case["nfield"], m1, m2))
        for j1, c1 in enumerate(i1):
            for f in range(case["nfield"]):
                np.add.at(e[f, c1], i2, a[f, j1])
        c = np.fft.ifft2((np.conj(np.fft.fft2(e)) * np.fft.fft2(a[:, :m1, :m2])).sum(axis=0)).real
        return c[np.ix_(i1, i2)]
    irvec, hr = _model(case, seed)
    kpts, w, eta = _points(case, seed)
    h00, h01 = _hamiltonians(case, irvec, hr, kpts)
    if kind == "ham":
        return h00, h01
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    n, nw, ninst = case["nw"] * case["np"], case["nw"], _instances(case)
    # about 20 seconds of library inverses and products (on the GPU: 2 s for
    # 441 instances of order 288, under a second for 8192 of order 72)
    if ninst * (2e-5 + 2e-10 * n ** 3) * (1 if dev == "cuda" else 20) > 20.0:
        return None
    if kind == "green":
        ik, om, et = np.zeros(1, dtype=np.int64), w, np.array([eta])
    elif kind == "batch":
        ik, om, et = _k_index(case, seed), w, eta
    else:
        ik = np.repeat(np.arange(kpts.shape[0]), w.size)
        om = np.tile(w, kpts.shape[0])
        et = np.full(om.size, eta)
    h00, h01 = torch.from_numpy(h00).to(dev), torch.from_numpy(h01).to(dev)
    top = torch.arange(nw, device=dev)
    dl, dr, db, its, sl, sr = [], [], [], [], [], []
    step = max(1, min(2048, int(4e6 / (n * n))))
    for t0 in range(0, om.size, step):
        k = torch.from_numpy(np.asarray(ik[t0:t0 + step], dtype=np.int64)).to(dev)
        z = torch.from_numpy(om[t0:t0 + step] + 1j * et[t0:t0 + step]).to(dev)
        gll, grr, gb, it = _decimate(h00[k], h01[k], z)
        if kind == "green":
            return gll[0].cpu().numpy(), grr[0].cpu().numpy(), gb[0].cpu().numpy(), int(it[0])
        diag = [torch.diagonal(g, dim1=1, dim2=2).imag for g in (gll, grr, gb)]
        dl.append(-diag[0][:, top].sum(dim=1))
        dr.append(-diag[1][:, n - nw + top].sum(dim=1))
        db.append(-diag[2].sum(dim=1))
        its.append(it)
        if kind == "grid" and case["spin"]:
            sl.append(_spin(gll, nw, n))
            sr.append(_spin(grr, nw, n))
    div = M.REF_PI if kind == "plane" else 1.0
    shape = (om.size,) if kind == "batch" else (kpts.shape[0], w.size)
    out = [(torch.cat(x) / div).cpu().numpy().reshape(shape) for x in (dl, dr, db)]
    out += [torch.cat(its).cpu().numpy().reshape(shape), np.zeros(shape, dtype=np.int32)]
    if kind == "grid" and case["spin"]:
        out += [torch.cat(x, dim=1).cpu().numpy().reshape((3,) + shape) for x in (sl, sr)]
    return tuple(out)
