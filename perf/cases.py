"""What a program does with this package, as cases that can be timed.

The sizes are those of the repository's own tests, bench workloads and
configurations, or lie between them: block-tridiagonal devices of 16 to 768
orbitals per slab, lead decimations, block inversions, the energy-axis
correlations and the GW stages, through the public entry points (the Python
layer, or the C ABI with device pointers where a program keeps its results
resident).  Device Hamiltonians are random Hermitian blocks of nearest
bonds of about -1 eV with sparse couplings, energies lie inside the bands.

Sweeps that return whole spectra take a contact broadening of 10 meV: at the
default 1e-5 eV single points next to a band edge are so ill conditioned that
two correct double-precision operation orders differ by 1e-7 and more; the
transmission case runs at the default, where the contact currents are not.
"""
import ctypes as C
import math

import numpy as np
import torch

from quantum_transport_amd import rgf

DEV = "cuda"
CPU = "cpu"
BOLTZ = 8.61734e-05  # eV/K, as in the reference
PI = 3.14159265359   # the reference's constant
C128 = torch.complex128


def listed():
    return [
        # the reference's CPU-size ballistic run: one small device, an energy grid
        dict(name="sweep 64x32 e256", kind="sweep", nb=64, slabs=32, points=256, kz=1, variant="forward",
             precision="fp64", spectra=True, barrier=False),
        # the production block size: 4 kz points, identical slabs, whole spectra
        dict(name="sweep 512x20 e64 kz4", kind="sweep", nb=512, slabs=20, points=64, kz=4, variant="forward",
             precision="fp64", spectra=True, barrier=False),
        # the precision mode that meets the 1e-8 bar, at an odd block size
        dict(name="sweep 250x12 e48 3m", kind="sweep", nb=250, slabs=12, points=48, kz=2, variant="forward",
             precision="fp64_3m", spectra=True, barrier=False),
        # T(E) only, backward ordering, a potential barrier, the default contact broadening
        dict(name="transmission 160x16 e100", kind="sweep", nb=160, slabs=16, points=100, kz=1, variant="backward",
             precision="fp64", spectra=False, barrier=True),
        # slabs of unequal size, as a sliced device has them
        dict(name="uneven 128-768 e16", kind="uneven", small=128, large=768, slabs=9, points=16),
        # one energy point through the per-point interface, full block lists
        dict(name="point 32x6", kind="point", nb=32, slabs=6, variant="forward"),
        # the lead stage by itself: surface Green's functions of many energies
        dict(name="leads 192 e60", kind="leads", nb=192, points=60),
        # Schur complements inverted by a program that holds its blocks on the device
        dict(name="invert 300 x48", kind="invert", n=300, batch=48),
        # correlation of long energy series
        dict(name="corr 2048 x8192", kind="series", mode="corr", n=2048, count=8192),
        # GW polarisation, one k point, every element of the blocks
        dict(name="pol nm80 x2 e2048", kind="pol", nm=80, slabs=2, energies=2048, nky=1, nkz=1, ndiag=79),
        # GW self-energy with a k sum, a band of elements and a ragged energy axis
        dict(name="sigma nm40 x2 e1000 k4", kind="sigma", nm=40, slabs=2, energies=1000, nky=2, nkz=2, ndiag=20),
        # one GW-SCBA iteration with everything resident
        dict(name="scba nm96 x4 e256", kind="scba", nm=96, slabs=4, energies=256, ndiag=95),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    top = work(listed()[1])["flops"]
    while True:
        kind = rng.choice(["sweep", "sweep", "sweep", "uneven", "point", "leads", "invert", "series", "pol", "sigma",
                           "scba"])
        if kind == "sweep":
            spectra = rng.random() < 0.7
            c = dict(kind=kind, nb=_log(rng, 16, 512), slabs=rng.randint(4, 40), points=_log(rng, 4, 300),
                     kz=rng.choice([1, 1, 2, 4]), variant=rng.choice(["forward", "forward", "backward"]),
                     precision=rng.choice(["fp64", "fp64", "fp64_3m"]), spectra=spectra,
                     barrier=rng.random() < 0.5)
        elif kind == "uneven":
            c = dict(kind=kind, small=_log(rng, 32, 200), large=_log(rng, 240, 768), slabs=rng.randint(4, 12),
                     points=rng.randint(4, 24))
        elif kind == "point":
            c = dict(kind=kind, nb=_log(rng, 8, 64), slabs=rng.randint(3, 12),
                     variant=rng.choice(["forward", "backward"]))
        elif kind == "leads":
            c = dict(kind=kind, nb=_log(rng, 32, 256), points=_log(rng, 6, 60))
        elif kind == "invert":
            n = _log(rng, 24, 900)
            c = dict(kind=kind, n=n, batch=min(_log(rng, 4, 256), (60 << 20) // (520 * n)))
        elif kind == "series":
            c = dict(kind=kind, mode=rng.choice(["corr", "conv"]), n=_log(rng, 100, 2048), count=_log(rng, 500, 8192))
        elif kind in ("pol", "sigma"):
            nky, nkz = rng.choice([(1, 1), (1, 1), (1, 3), (2, 2)])
            nm = _log(rng, 24, 80)
            c = dict(kind=kind, nm=nm, slabs=rng.randint(1, 3), energies=_log(rng, 200, 2048), nky=nky, nkz=nkz,
                     ndiag=rng.choice([nm - 1, nm // 3]))
        else:
            nm = _log(rng, 16, 96)
            c = dict(kind=kind, nm=nm, slabs=rng.randint(3, 6), energies=rng.randint(48, 256),
                     ndiag=rng.choice([nm - 1, nm // 3]))
        if work(c)["flops"] <= top:
            return c


# ------------------------------------------------------------------ inputs


def _block(rng, n, bonds=4):
    """Hermitian on-site block: energies in [-1, 1] eV, a few bonds per orbital."""
    h = np.zeros((n, n), np.complex128)
    for i in range(n):
        for j in rng.integers(0, n, bonds):
            h[i, j] = -1.0 - 0.1 * rng.standard_normal()
            h[j, i] = h[i, j]
    h[np.arange(n), np.arange(n)] = rng.uniform(-1.0, 1.0, n)
    return np.asfortranarray(h)


def _coupling(rng, nr, nc, hermitian=False):
    p = min(0.5, max(0.05, 6.0 / nc))
    u = np.where(rng.random((nr, nc)) < p, -1.0 - 0.1 * rng.standard_normal((nr, nc)), 0.0).astype(np.complex128)
    if hermitian:
        u = np.tril(u) + np.tril(u, -1).conj().T
    return np.asfortranarray(u)


def _energies(rng, points, lo=-2.0, hi=2.0):
    """A grid over the window, its origin shifted from input to input."""
    d = (hi - lo) / points
    return lo + d * (np.arange(points) + rng.random())


def _device(c, seed):
    """(Hii, H1i, En, kidx) of a sweep: host blocks [k][slab], [k][coupling]."""
    rng = np.random.default_rng([seed, 11])
    if c["kind"] == "uneven":
        lo, hi, nx = c["small"], c["large"], c["slabs"]
        # slab sizes spread over the range (the golden ratio's multiples), part of the case
        sizes = [int(round(lo * (hi / lo) ** ((0.618034 * s) % 1.0))) for s in range(nx)]
        Hii = [[_block(rng, n) for n in sizes]]
        edge = [sizes[0]] + sizes + [sizes[-1]]
        H1i = [[_coupling(rng, edge[s + 1], edge[s]) for s in range(nx + 1)]]
        return Hii, H1i, _energies(rng, c["points"]), np.zeros(c["points"], np.int32)
    n, nx, nk = c["nb"], c["slabs"], c.get("kz", 1)
    h0 = _block(rng, n)
    u = _coupling(rng, n, n, hermitian=c["variant"] == "backward")
    tz = _coupling(rng, n, n) * 0.5 if nk > 1 else None
    Hii, H1i = [], []
    for k in range(nk):
        h = h0
        if tz is not None:
            ph = np.exp(1j * math.pi * k / nk)
            h = np.asfortranarray(h0 + tz * ph + (tz * ph).conj().T)
        blocks = [h] * nx
        if c.get("barrier"):  # a smooth on-site potential inside the device, zero at both contacts
            blocks = []
            for s in range(nx):
                b = h.copy()
                b[np.arange(n), np.arange(n)] += 0.3 * math.sin(math.pi * s / (nx - 1)) ** 2
                blocks.append(b)
            blocks[-1] = blocks[0]
        Hii.append(blocks)
        H1i.append([u] * (nx + 1))
    pts = c.get("points", 1)
    if c["kind"] == "point":  # between the two chemical potentials, 0 and -0.1 eV
        return Hii, H1i, _energies(rng, 1, -0.1, 0.0), np.zeros(1, np.int32)
    return Hii, H1i, _energies(rng, pts), (np.arange(pts) % nk).astype(np.int32)


def _gen(seed, tag):
    return torch.Generator(device=DEV).manual_seed(seed * 16 + tag)


def _green(shape, seed, tag, lo=0.2):
    """Complex samples with a smooth energy dependence along the last axis, as
    Green's functions have it, and a little noise."""
    g = _gen(seed, tag)
    a = torch.randn(shape[:-1] + (4,), dtype=C128, device=DEV, generator=g)
    x = torch.linspace(-1.0, 1.0, shape[-1], dtype=torch.float64, device=DEV)
    out = torch.randn(shape, dtype=C128, device=DEV, generator=g).mul_(0.02)
    for i in range(4):
        pole = -0.9 + 0.6 * i
        out.addcmul_(a[..., i, None], (1.0 / (x - pole + lo * 1j)).expand(shape))
    return out


def _params(c):
    prec = {"fp64": rgf.QT_PREC_FP64, "fp64_3m": rgf.QT_PREC_FP64_3M}[c.get("precision", "fp64")]
    return rgf.make_params(c.get("variant", "forward"), mul=0.0, mur=-0.1, lead_eta=_eta(c),
                           coupling_fix=c["kind"] == "uneven", device_outputs=True, precision=prec)


def _eta(c):
    return 1e-2 if c.get("spectra", True) else 1e-5


def prepare(case, seed):
    c, kind = case, case["kind"]
    rgf.init(0)
    if kind in ("sweep", "uneven"):
        Hii, H1i, En, k = _device(c, seed)
        H = rgf.Hamiltonian(Hii, H1i)
        pts, nd = len(En), sum(H.nm)
        out = {"tr": torch.zeros(pts, dtype=torch.float64, device=DEV),
               "tre": torch.zeros(pts, dtype=torch.float64, device=DEV)}
        if c.get("spectra", True):
            for key in ("gr_diag", "gl_diag", "gg_diag"):
                out[key] = torch.zeros(pts, nd, dtype=C128, device=DEV)
        return dict(case=c, H=H, En=En, k=k, p=_params(c), out=out)
    if kind == "point":
        Hii, H1i, En, _ = _device(dict(c, points=1), seed)
        return dict(case=c, Hii=Hii[0], H1i=H1i[0], En=float(En[0]))
    if kind == "leads":
        h, u, En = _leads(c, seed)
        return dict(case=c, h=[h] * len(En), u=[u] * len(En), En=En)
    if kind == "invert":
        A = _schur(c, seed)
        return dict(case=c, A=A, W=torch.empty_like(A), X=torch.empty_like(A),
                    info=torch.zeros(c["batch"], dtype=torch.int32, device=DEV))
    if kind == "series":
        shape = (c["count"], c["n"])
        return dict(case=c, X=_green(shape, seed, 1), Y=_green(shape, seed, 2),
                    Z=torch.empty(shape, dtype=C128, device=DEV))
    if kind in ("pol", "sigma"):
        shape = _gw_shape(c)
        G = [_green(shape, seed, 1 + i) for i in range(3)]
        W = [_green(shape, seed, 4 + i) for i in range(3)] if kind == "sigma" else []
        return dict(case=c, inputs=G + W, out=[torch.empty(shape, dtype=C128, device=DEV) for _ in range(3)])
    return _prepare_scba(c, seed)


def _leads(c, seed):
    rng = np.random.default_rng([seed, 12])
    n = c["nb"]
    return _block(rng, n), _coupling(rng, n, n), _energies(rng, c["points"])


def _schur(c, seed):
    """E - H - Sigma with a broad self-energy, column-major blocks (batch, col, row)."""
    n, b = c["n"], c["batch"]
    rng = np.random.default_rng([seed, 13])
    h = torch.from_numpy(_block(rng, n)).to(DEV)
    e = torch.from_numpy(_energies(rng, b)).to(DEV)
    g = torch.randn(b, n, n, dtype=C128, device=DEV, generator=_gen(seed, 3)) / math.sqrt(n)
    s = 0.2 * (g - 1j * (g @ g.mH))
    return (e[:, None, None] * torch.eye(n, dtype=C128, device=DEV) - h - s).mT.contiguous()


def _gw_shape(c):
    return (c["nm"] ** 2, c["slabs"], c["nky"] * c["nkz"], c["energies"])


def _scba_inputs(c, seed):
    nm, nx, nen = c["nm"], c["slabs"], c["energies"]
    rng = np.random.default_rng([seed, 14])
    h, u = _block(rng, nm), _coupling(rng, nm, nm)
    cr = lambda s: s * (rng.standard_normal((nm, nm, nx)) + 1j * rng.standard_normal((nm, nm, nx)))
    V = cr(0.05 / math.sqrt(nm))
    V = V + V.conj().transpose(1, 0, 2)
    for s in range(nx):
        V[:, :, s] += np.diag(rng.uniform(0.5, 1.0, nm))
    V1 = cr(0.02 / math.sqrt(nm))
    En = np.linspace(-2.0, 2.0, nen) + 1e-3 * rng.random()
    # a previous iteration's scattering: Sigma^R = -i Gamma/2 with a broadening of some 0.1 eV
    g = torch.randn(nx, nm, nm, dtype=C128, device=DEV, generator=_gen(seed, 5)) / math.sqrt(nm)
    gam = 0.1 * (g @ g.mH + 0.3 * torch.eye(nm, dtype=C128, device=DEV))
    f = torch.from_numpy(1.0 / (1.0 + np.exp(En / 0.2))).to(DEV)
    prof = torch.from_numpy(1.0 + 0.5 * np.cos(En)).to(DEV)
    base = gam.permute(2, 1, 0).reshape(nm * nm, nx)  # element row + col*nm, slab
    S = [base[:, :, None] * (prof * w)[None, None, :] for w in (-0.5j * torch.ones_like(f), 1j * f, -1j * (1.0 - f))]
    return h, u, V, V1, En, [s.contiguous() for s in S]


def _prepare_scba(c, seed):
    nm, nx, nen = c["nm"], c["slabs"], c["energies"]
    h, u, V, V1, En, S0 = _scba_inputs(c, seed)
    H = rgf.Hamiltonian([[h] * nx], [[u] * (nx + 1)])
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v.transpose(2, 1, 0))).to(DEV)  # column-major blocks
    new = lambda: [torch.zeros(nm * nm, nx, 1, nen, dtype=C128, device=DEV) for _ in range(3)]
    return dict(case=c, H=H, V=dev(V), V1=dev(V1), En=En, S0=[s.view(nm * nm, nx, 1, nen) for s in S0], S=new(),
                G=new(), P=new(), tr=np.zeros(nen), tre=np.zeros(nen),
                p=rgf.make_params("gw", 0.1, -0.1, 300.0, 300.0, lead_eta=1e-3, lead_nmax=100, lead_reset=True))


# ------------------------------------------------------------------ one pass


def run(state):
    c, kind, L = state["case"], state["case"]["kind"], rgf.lib()
    if kind in ("sweep", "uneven"):
        o, out = rgf.Outputs(), state["out"]
        o.tr = C.cast(out["tr"].data_ptr(), C.POINTER(C.c_double))
        o.tre = C.cast(out["tre"].data_ptr(), C.POINTER(C.c_double))
        if "gr_diag" in out:
            o.gr_diag, o.gl_diag, o.gg_diag = (out[k].data_ptr() for k in ("gr_diag", "gl_diag", "gg_diag"))
        En, k = state["En"], state["k"]
        rgf.check(L.qt_rgf_solve(state["H"].handle, C.byref(state["p"]), C.c_int32(len(En)),
                                 En.ctypes.data_as(C.c_void_p), k.ctypes.data_as(C.c_void_p), None, None, C.byref(o)))
        return out
    if kind == "point":
        f = rgf.rgf_variableblock_forward if c["variant"] == "forward" else rgf.rgf_variableblock_backward
        r = f(state["Hii"], state["H1i"], state["En"], 0.0, -0.1)
        return {k: r[k] for k in ("G_r", "G_lesser", "G_greater", "Jdens", "tr", "tre")}
    if kind == "leads":
        G00, _, _, conv = rgf.sancho(state["h"], state["u"], state["En"], eta=1e-2, nmax=100, want_gbb=False)
        return {"G00": G00, "converged": conv}
    if kind == "invert":
        state["W"].copy_(state["A"])  # the call destroys its input
        torch.cuda.current_stream().synchronize()  # the library works on a stream of its own
        st = L.qt_invert_batched_noalloc(c["n"], c["batch"], state["W"].data_ptr(), state["X"].data_ptr(),
                                         state["info"].data_ptr())
        rgf.check(st)
        return {"X": state["X"], "info": state["info"]}
    if kind == "series":
        f = L.qt_corr1d2_batched if c["mode"] == "corr" else L.qt_conv1d2_batched
        rgf.check(f(c["n"], c["count"], state["X"].data_ptr(), state["Y"].data_ptr(), state["Z"].data_ptr(),
                    rgf.QT_F_DEVICE_OUTPUTS))
        return state["Z"]
    ptr = lambda v: [t.data_ptr() for t in v]
    if kind == "pol":
        rgf.check(L.qt_gw_polarization(c["energies"], c["nky"], c["nkz"], c["slabs"], c["nm"], c["ndiag"], _dE(c), 2.0,
                                       *ptr(state["inputs"]), *ptr(state["out"]), rgf.QT_F_DEVICE_OUTPUTS))
        return state["out"]
    if kind == "sigma":
        rgf.check(L.qt_gw_selfenergy(c["energies"], c["nky"], c["nkz"], c["slabs"], c["nm"], c["ndiag"], _dE(c),
                                     *ptr(state["inputs"]), *ptr(state["out"]), rgf.QT_F_DEVICE_OUTPUTS))
        return state["out"]
    for s, s0 in zip(state["S"], state["S0"]):
        s.copy_(s0)
    torch.cuda.current_stream().synchronize()
    p3 = lambda v: (C.c_void_p * 3)(*ptr(v))
    st = L.qt_gw_scba_step(state["H"].handle, C.byref(state["p"]), c["energies"],
                           state["En"].ctypes.data_as(C.c_void_p), c["ndiag"], 2.0, 0.5, state["V"].data_ptr(),
                           state["V1"].data_ptr(), p3(state["S"]), p3(state["G"]), p3(state["P"]),
                           state["tr"].ctypes.data_as(C.c_void_p), state["tre"].ctypes.data_as(C.c_void_p), None)
    rgf.check(st)
    return {"S": state["S"], "G": state["G"], "P": state["P"], "tr": state["tr"], "tre": state["tre"]}


def _dE(c):
    return 4.0 / (c["energies"] - 1)


# ------------------------------------------------------------------ work


def _lead_steps(c):
    return 20 if _eta(c) > 1e-3 else 26


def work(case):
    """Products and inversions count 8 n^3 each (complex128).  A slab of a
    sweep takes ten products and one inversion, a decimation step six and
    one; transforms of the energy axis count 5 L log2 L."""
    c, kind = case, case["kind"]
    if kind in ("sweep", "uneven", "point"):
        if kind == "uneven":
            sizes = [c["small"] * (c["large"] / c["small"]) ** ((0.618034 * s) % 1.0) for s in range(c["slabs"])]
            ends = [sizes[0], sizes[-1]]
        else:
            sizes, ends = [c["nb"]] * c["slabs"], [c["nb"]]
        pts, nk = c.get("points", 1), c.get("kz", 1)
        flops = pts * (sum(88.0 * n ** 3 for n in sizes) + sum(56.0 * n ** 3 * _lead_steps(c) for n in ends))
        if kind == "point":
            byts = 16.0 * c["nb"] ** 2 * c["slabs"] * 8
        else:
            byts = 32.0 * nk * sum(n * n for n in sizes) + 16.0 * pts * (1 + 3 * sum(sizes) * c.get("spectra", True))
        return {"bytes": byts, "flops": flops}
    if kind == "leads":
        n = c["nb"]
        return {"bytes": 16.0 * n * n * (2 + c["points"]), "flops": 56.0 * n ** 3 * 20 * c["points"]}
    if kind == "invert":
        return {"bytes": 32.0 * c["n"] ** 2 * c["batch"], "flops": 8.0 * c["n"] ** 3 * c["batch"]}
    if kind == "series":
        return {"bytes": 48.0 * c["n"] * c["count"], "flops": 3.0 * _fft(c["n"]) * c["count"]}
    nm, nd = c["nm"], c["ndiag"]
    el = sum(min(nm, i + nd + 1) - max(0, i - nd) for i in range(nm)) * c["slabs"] * float(c.get("nky", 1) * c.get("nkz", 1))
    every = float(nm * nm * c["slabs"] * c.get("nky", 1) * c.get("nkz", 1))
    n = c["energies"]
    if kind == "pol":
        return {"bytes": 48.0 * n * (el + every), "flops": 3.5 * _fft(n) * el}
    if kind == "sigma":
        return {"bytes": 48.0 * n * (2 * el + every), "flops": 6.0 * _fft(n) * el}
    blocks = c["slabs"] * float(n)
    flops = blocks * 8.0 * nm ** 3 * (20 + 60) + n * 56.0 * nm ** 3 * 2 * 16 + 9.5 * _fft(n) * el
    return {"bytes": 16.0 * every * n * 12, "flops": flops}


def _fft(n):
    return 5.0 * 2 * n * math.log2(2 * n)


# ------------------------------------------------------------------ the same in plain torch


def exact(case, seed):
    """On the host, in 64 bits; None where that would take too long."""
    c, kind = case, case["kind"]
    if work(c)["flops"] > 8e11 or c.get("points", 1) * c.get("slabs", 1) > 2000 or kind == "uneven":
        return None
    if kind in ("sweep", "uneven"):
        r = _sweep(c, *_device(c, seed))
        return {k: r[k] for k in (("tr", "tre", "gr_diag", "gl_diag", "gg_diag") if c.get("spectra", True)
                                  else ("tr", "tre"))}
    if kind == "point":
        r = _sweep(dict(c, points=1, spectra=False), *_device(dict(c, points=1), seed))
        return {"G_r": r["G_r"], "G_lesser": r["G_lesser"], "G_greater": r["G_greater"], "Jdens": None,
                "tr": float(r["tr"][0]), "tre": float(r["tre"][0])}
    if kind == "leads":
        h, u, En = _leads(c, seed)
        up = lambda a: torch.from_numpy(a).expand(len(En), -1, -1)
        G = _sancho(torch.from_numpy(En) + 1e-2j, up(h), up(u), 100)
        return {"G00": list(G.numpy()), "converged": None}
    if kind == "invert":
        return {"X": torch.linalg.inv(_schur(c, seed).cpu().mT).mT.contiguous(), "info": None}
    if kind == "series":
        X, Y = (_green((c["count"], c["n"]), seed, i).cpu() for i in (1, 2))
        return _corr(X, Y) if c["mode"] == "corr" else _conv(X, Y)
    if kind == "pol":
        return _pol(c, seed)
    if kind == "sigma":
        return _sigma(c, seed)
    return None


def _inv(a):
    return torch.linalg.inv(a)


def _sancho(z, H00, H10, nmax):
    eye = torch.eye(H00.shape[-1], dtype=C128, device=H00.device)
    zs = z[:, None, None] * eye
    hs, hb, h10, h01 = H00.clone(), H00.clone(), H10.clone(), H10.mH.clone()
    act = torch.ones(len(z), dtype=torch.bool, device=H00.device)
    for _ in range(nmax):
        a = _inv(zs - hb)
        c, ap = h01 @ (a @ h10), h10 @ (a @ h01)
        n10, n01 = h10 @ (a @ h10), h01 @ (a @ h01)
        m = act[:, None, None]
        hs, hb = torch.where(m, hs + c, hs), torch.where(m, hb + c + ap, hb)
        h10, h01 = torch.where(m, n10, h10), torch.where(m, n01, h01)
        act = act & ~(n01.abs().sum((-1, -2)) < 1e-100)
        if not bool(act.any()):
            break
    return _inv(zs - hs)


def _sweep(c, Hii, H1i, En, kidx):
    """The recursive Green's function sweep of one batch of points: left (or,
    backward, right) connected blocks, then the full ones."""
    fwd, fix = c.get("variant", "forward") == "forward", c["kind"] == "uneven"
    up = lambda blocks, s: torch.from_numpy(np.stack([np.asarray(b[s]) for b in blocks]))[k]
    k = torch.from_numpy(kidx.astype(np.int64))
    nx = len(Hii[0])
    E = torch.from_numpy(En)
    ferm = lambda mu: (1.0 / (1.0 + torch.exp((E - mu) / (BOLTZ * 300.0))))[:, None, None]
    fF, fL = ferm(-0.1), ferm(0.0)
    order = list(range(nx)) if fwd else list(range(nx - 1, -1, -1))
    sf, sl = order[0], order[-1]
    cF, cL = (0, nx) if fwd else (nx, 0)
    z = E + 1j * _eta(c)
    uF, uL = up(H1i, cF), up(H1i, cL)
    sigF = uF @ _sancho(z, up(Hii, sf), uF.mH if fwd else uF, 50) @ uF.mH
    sigL = uL.mH @ _sancho(z, up(Hii, sl), uL if fwd else uL.mH, 50) @ uL
    gl, gln, prev = {}, {}, None
    for s in order:
        h = up(Hii, s)
        sig, inj = torch.zeros_like(h), torch.zeros_like(h)
        if prev is None:
            sig, inj = sigF, -(sigF - sigF.mH) * fF
        else:
            u = up(H1i, s if fwd else s + 1)
            sig, inj = u @ gl[prev] @ u.mH, u @ gln[prev] @ u.mH
        if s == sl:
            sig, inj = sig + sigL, inj - (sigL - sigL.mH) * fL
        gl[s] = _inv(E[:, None, None] * torch.eye(h.shape[-1], dtype=C128, device=CPU) - h - sig)
        gln[s] = gl[s] @ inj @ gl[s].mH
        prev = s
    G, L = {sl: gl[sl]}, {sl: gln[sl]}
    for q, s in zip(order[:0:-1], order[-2::-1]):
        w = up(H1i, s + 1 if fwd and fix else s)
        x = gl[s] @ w.mH
        g0 = x @ G[q]
        G[s] = gl[s] + g0 @ (w @ gl[s])
        t = g0 @ (w @ gln[s])
        L[s] = gln[s] + x @ L[q] @ x.mH + t - t.mH

    def current(sig, s, f):
        om, w = -(sig - sig.mH), L[s] + f * (G[s] - G[s].mH)
        return (om * w.mT).sum((-1, -2)).real

    diag = lambda A: torch.cat([A[s].diagonal(dim1=-2, dim2=-1) for s in range(nx)], -1)
    last, first = current(sigL, sl, fL), current(sigF, sf, fF)
    gr, gle = diag(G), diag(L)
    host = lambda A: [A[s][0].numpy() for s in range(nx)]
    out = {"tr": last if fwd else first, "tre": first if fwd else last, "gr_diag": gr, "gl_diag": gle,
           "gg_diag": gle + gr - gr.conj()}
    if c["kind"] == "point":
        out.update(G_r=host(G), G_lesser=host(L), G_greater=host({s: L[s] + G[s] - G[s].mH for s in L}))
    return out


def _fwd(x):
    return torch.fft.fft(x, 2 * x.shape[-1])


def _lags(f):  # of a product with the spectrum of a flipped operand
    n = f.shape[-1] // 2
    return torch.fft.ifft(f)[..., n - 1 - n // 2:2 * n - 1 - n // 2].contiguous()


def _samples(f):
    n = f.shape[-1] // 2
    return torch.fft.ifft(f)[..., n // 2:n // 2 + n].contiguous()


def _corr(x, y):
    return _lags(_fwd(x) * _fwd(y.flip(-1)))


def _conv(x, y):
    return _samples(_fwd(x) * _fwd(y))


def _paired(iq, ik, nky, nkz):
    """k' of (k, q), folded into the grid (the reference's 1-based rule)."""
    a = ik % nkz - iq % nkz + nkz // 2
    b = ik // nkz - iq // nkz + nky // 2

    def fold(v, m):  # the 1-based difference: the two ones cancel
        v = v + m if v < 1 else v
        v = v - m if v > m else v
        return 1 if m == 1 else v

    return fold(a, nkz) - 1 + (fold(b, nky) - 1) * nkz


def _gw(c, seed, count):
    nm = c["nm"]
    ij = torch.arange(nm * nm, device=CPU)
    row, col = ij % nm, ij // nm
    band = ((row - col).abs() <= c["ndiag"]).to(torch.float64)[:, None, None, None]
    A = [_green(_gw_shape(c), seed, 1 + i).cpu() for i in range(count)]
    A[:3] = [1j * a.imag for a in A[:3]]
    return A, col + row * nm, band


def _pol(c, seed):
    A, t, band = _gw(c, seed, 3)
    nk = c["nky"] * c["nkz"]
    R, L, G = (_fwd(a) for a in A)
    cR, Lt, Gt = _fwd(A[0].conj().flip(-1)), _fwd(A[1].flip(-1))[t], _fwd(A[2].flip(-1))[t]
    out = [torch.zeros_like(R) for _ in range(3)]
    # element by element: the transpose of element ij is element t[ij]
    for iq in range(nk):
        for ik in range(nk):
            kd = _paired(iq, ik, c["nky"], c["nkz"])
            out[0][:, :, iq] += L[:, :, ik] * cR[:, :, kd] + R[:, :, ik] * Lt[:, :, kd]
            out[1][:, :, iq] += L[:, :, ik] * Gt[:, :, kd]
            out[2][:, :, iq] += G[:, :, ik] * Lt[:, :, kd]
    f = -1j * _dE(c) / 2.0 / PI * 2.0 / nk
    return [f * band * _lags(p) for p in out]


def _sigma(c, seed):
    A, t, band = _gw(c, seed, 6)
    nk = c["nky"] * c["nkz"]
    R, L, G, WR, WL, WG = (_fwd(a) for a in A)
    out = [torch.zeros_like(R) for _ in range(3)]
    for ik in range(nk):
        for iq in range(nk):
            kd = _paired(iq, ik, c["nky"], c["nkz"])
            out[0][:, :, ik] += R[:, :, kd] * (WL[:, :, iq] + WR[:, :, iq]) + L[:, :, kd] * WR[:, :, iq]
            out[1][:, :, ik] += L[:, :, kd] * WL[:, :, iq]
            out[2][:, :, ik] += G[:, :, kd] * WG[:, :, iq]
    f = 1j * _dE(c) / 2.0 / PI / nk
    R, L, G = (f * band * _samples(s) for s in out)
    R = torch.complex(R.real, 0.5 * (G - L).imag)
    return [0.5 * (s + s[t]) for s in (R, L, G)]
