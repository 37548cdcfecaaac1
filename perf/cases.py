"""Performance cases: what a simulation run asks of libmgpu, through its public calls.

kind "run"     a stretch of a COLA run between two outputs: particles from the LPT
               fields, then `steps` force evaluations with Kick and Drift, then the
               particles back to the caller.  "call" says how the program steps:
                 separate  GetDisplacements, Kick, Drift as separate calls, the means on
                           the host (how a C program with the reference's loop calls it)
                 device    mgpu_step, the means on the device
                 graph     mgpu_step with one hipGraph launch per step
                 batch     mgpu_batch_step over `members` realizations at once
kind "ic"      2LPT initial conditions
kind "output"  what an output adds: P(k) and the redshift-space multipoles of both lines
               of sight

Boxes have 2 Mpc/h per particle, the spacing of the workloads here; the steps cover the
late times (a = 0.65 on, 0.035 per step), where the particles are clustered.  P(k) is
returned as float32: it is binned from a float32 mesh.  A run returns the velocities, and
the positions too while few particles are there to sit at the box's edge, where the same
trajectory, rounded otherwise, comes back at either end of the box (every step's forces,
and so the velocities, follow from all positions).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "mg-picola-public_amd"))
import mgpicola as M  # noqa: E402

OMEGA, HUBBLE, NS, SIGMA8 = 0.3, 0.7, 0.96, 0.8
FOFR0, RC_H0, C_H0 = 1e-5, 1.0, 2997.92458
A0, DA = 0.65, 0.035
MODELS = {"lcdm": M.LCDM, "fofr": M.FOFR, "dgp": M.DGP, "jbd": M.BRANSDICKE}
MESHES = (32, 48, 64, 96, 128, 192, 256, 384)


def _case(name, kind, model, ns, nmesh, steps=1, call="separate", members=1, pofk=False, sd=False, screening=True,
          spacing=2.0):
    return dict(name=name, kind=kind, model=model, nsample=ns, nmesh=nmesh, box=spacing * ns, steps=steps, call=call,
                members=members, pofk=pofk, sd=sd, screening=screening)


def listed():
    return [
        # the smallest calls: a test-sized run of the model whose force is a plain rescaling (no fused path)
        _case("jbd_16_32", "run", "jbd", 16, 32, steps=4, pofk=True),
        # the small LCDM run of the parity workloads, 10 steps
        _case("lcdm_64_128", "run", "lcdm", 64, 128, steps=10),
        # ensemble members: one after the other, and as one batch
        _case("dgp_96_192_graph", "run", "dgp", 96, 192, steps=10, call="graph"),
        _case("dgp_96_192_batch8", "run", "dgp", 96, 192, steps=5, call="batch", members=8),
        _case("dgp_192_384", "run", "dgp", 192, 384, steps=8, call="device"),
        # a lattice that does not divide the mesh, P(k) every step
        _case("fofr_100_256", "run", "fofr", 100, 256, steps=5, pofk=True),
        # scale-dependent growth: the LPT fields are remade every step
        _case("fofr_sd_128_256", "run", "fofr", 128, 256, steps=5, pofk=True, sd=True),
        # coarse (Nmesh = Nsample) and fine (Nmesh = 3 Nsample) meshes of a training pair
        _case("lcdm_256_256", "run", "lcdm", 256, 256, steps=8),
        _case("fofr_256_768", "run", "fofr", 256, 768, steps=4),
        # the production run: scale-dependent f(R) with screening, P(k) every step
        _case("fofr_sd_512_1024", "run", "fofr", 512, 1024, steps=6, pofk=True, sd=True),
        _case("ic_192_384", "ic", "lcdm", 192, 384),
        _case("output_192_384", "output", "lcdm", 192, 384, pofk=True),
    ]


def draw(rng):
    n = rng.choice(MESHES)
    kind = rng.choice(("run", "run", "run", "run", "ic", "output"))
    ratio = rng.choice((1, 2, 2, 3, 0))
    ns = n // ratio if ratio else rng.randint(n // 3, n - 1)  # 0: a lattice of any size
    ns = max(8, min(ns, 256))
    model = rng.choice(("lcdm", "fofr", "dgp", "jbd")) if kind == "run" else "lcdm"
    sd = kind == "run" and model == "fofr" and n <= 256 and n % ns == 0 and ns % 8 == 0 and rng.random() < 0.5
    call = "separate" if sd or model == "jbd" else rng.choice(("separate", "device", "graph", "batch"))
    batch = rng.randint(2, 6) if call == "batch" and kind == "run" else 1
    pofk = kind == "output" or (kind == "run" and call == "separate" and rng.random() < 0.5)
    case = _case("", kind, model, ns, n, steps=rng.randint(2, 6) if kind == "run" else 1,
                 call=call if kind == "run" else "separate", members=batch, pofk=pofk, sd=sd,
                 screening=call != "separate" or sd or rng.random() < 0.7, spacing=rng.uniform(1.5, 2.5))
    del case["name"]
    return case


# ---------------------------------------------------------------- cosmology of the calls' scalars
def _E(a):
    return math.sqrt(OMEGA / a**3 + 1.0 - OMEGA)


def _growth(a):
    """Linear growth, normalised at a = 1 (the fit of Carroll, Press & Turner 1992)."""
    def g(x):
        om = OMEGA / (OMEGA + (1 - OMEGA) * x**3)
        ol = 1 - om
        return 2.5 * om * x / (om ** (4 / 7) - ol + (1 + om / 2) * (1 + ol / 70))
    return g(a) / g(1.0)


def _rates(a):
    """D, D2 and their first and second derivatives in y (dy = da / (a^3 E))."""
    q, h = a**3 * _E(a), 1e-4
    d, dd = _growth(a), (_growth(a + h) - _growth(a - h)) / (2 * h)
    return {"D": (d, d * d), "dD": (q * dd, 2 * q * d * dd),
            "ddD": (1.5 * OMEGA * a * d, 1.5 * OMEGA * a * (10 / 3) * d * d)}


def _step_scalars(i):
    """(a, dda, dyyy, kick growth terms, drift growth terms) of step i."""
    a = A0 + i * DA
    ai, af, aff = (a if i == 0 else a - DA / 2), a + DA / 2, a + DA
    dda = (af**-2.5 - ai**-2.5) * a / (a**3 * _E(a)) / (-2.5 * a**-3.5)
    t = np.linspace(a, aff, 65)
    f = np.array([x**-2.5 / (x**3 * _E(x)) for x in t])
    w = np.ones(65)
    w[1:-1:2], w[2:-1:2] = 4, 2
    dyyy = float((w * f).sum() * (t[1] - t[0]) / 3) / af**-2.5
    r0, r1 = _rates(a), _rates(aff)
    return a, dda, dyyy, r0["ddD"], tuple(y - x for x, y in zip(r0["D"], r1["D"]))


def _mg(model, a):
    """The model hooks at a: Hu-Sawicki f(R) n = 1, nDGP, or a constant rescaling."""
    fl = 4 * (1 - OMEGA)
    mass2 = (OMEGA + fl) * ((OMEGA / a**3 + fl) / (OMEGA + fl)) ** 3 / (2 * FOFR0)
    phi = 1.5 * FOFR0 * ((OMEGA + fl) / (OMEGA / a**3 + fl)) ** 2
    h = 1e-4
    beta = 1 + 2 * RC_H0 * (_E(a) + a * (_E(a + h) - _E(a - h)) / (2 * h) / 3)
    return dict(a=a, coupling=1 / (3 * beta) if model == "dgp" else 1 / 3, mass2=mass2, phi_crit=phi,
                dgp_fac=8 / 9 * OMEGA * (RC_H0 / beta) ** 2, rsmooth=1.0, geff=1.05)


def _power(k):
    """P(k) today: n_s and the cold dark matter transfer function of Bardeen et al. 1986, sigma_8 normalised."""
    def shape(x):
        q = np.maximum(x, 1e-12) / (OMEGA * HUBBLE)
        t = np.log(1 + 2.34 * q) / (2.34 * q) * (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3
                                                 + (6.71 * q) ** 4) ** -0.25
        return np.where(x > 0, x**NS * t * t, 0.0)
    lk = np.linspace(math.log(1e-4), math.log(1e2), 8001)
    x = np.exp(lk) * 8.0
    w = 3 * (np.sin(x) - x * np.cos(x)) / x**3
    s2 = (shape(x / 8) * w * w * (x / 8) ** 3).sum() * (lk[1] - lk[0]) / (2 * math.pi**2)
    return shape(np.asarray(k, np.float64)) * SIGMA8**2 / s2


# ---------------------------------------------------------------- inputs
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _freq(n, half=False, nyquist=1):
    """Integer wavenumbers of an axis; nyquist = +1 or -1: the sign of n/2."""
    i = torch.arange(n // 2 + 1 if half else n, device=_dev(), dtype=torch.float64)
    return i if half else torch.where((i > n // 2) | ((i == n / 2) & (nyquist < 0)), i - n, i)


def _grid(n, nyquist=1):
    k = _freq(n, nyquist=nyquist)
    kz = _freq(n, True)
    if nyquist < 0 and n % 2 == 0:
        kz = torch.where(kz == n // 2, -kz, kz)
    return k[:, None, None], k[None, :, None], kz[None, None, :]


def _c2r(x, n):
    """Unnormalised c2r: complex transforms over x and y, then the z rows with Im of their ends dropped."""
    y = torch.fft.ifft2(x, dim=(0, 1), norm="forward")
    y[..., 0].imag.zero_()
    if n % 2 == 0:
        y[..., -1].imag.zero_()
    return torch.fft.irfft(y, n=n, dim=2, norm="forward")


def _spectra(ns, box, seed):
    """delta(k) and the 2LPT source S(k) on the ns^3 lattice (normalised so that c2r gives the field)."""
    g = torch.Generator(device=_dev()).manual_seed(int(seed))
    k = _grid(ns)
    n2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    white = torch.randn(ns, ns, ns, generator=g, device=_dev(), dtype=torch.float64)
    table = torch.from_numpy(np.sqrt(_power(2 * math.pi / box * np.sqrt(np.arange(3 * (ns // 2) ** 2 + 1)))))
    dk = torch.fft.rfftn(white, norm="forward") * table.to(_dev())[n2.long()] * math.sqrt(ns**3 / box**3)
    if ns % 2 == 0:
        dk[ns // 2], dk[:, ns // 2], dk[:, :, ns // 2] = 0, 0, 0
    inv = torch.where(n2 > 0, 1 / n2.clamp(min=1), torch.zeros_like(n2))
    d = [_c2r(-k[a] * k[a] * inv * dk, ns) for a in range(3)]
    src = d[0] * (d[1] + d[2]) + d[1] * d[2]
    for a, b in ((0, 1), (0, 2), (1, 2)):
        src -= _c2r(-k[a] * k[b] * inv * dk, ns) ** 2
    sk = torch.fft.rfftn(src, norm="forward")
    sk[0, 0, 0] = 0
    if ns % 2 == 0:
        sk[ns // 2], sk[:, ns // 2], sk[:, :, ns // 2] = 0, 0, 0
    return dk, sk


def _lattice_fields(ns, box, seed):
    """The ZA and 2LPT displacements of the lattice, float32 [2][3][ns^3], as a program holds them."""
    dk, sk = _spectra(ns, box, seed)
    k = _grid(ns)
    n2 = (k[0] ** 2 + k[1] ** 2 + k[2] ** 2).clamp(min=1)
    f = box / (2 * math.pi)
    return [torch.stack([_c2r(1j * k[a] / n2 * f * c * s, ns).reshape(-1) for a in range(3)]).float()
            for s, c in ((dk, 1.0), (sk, 3 / 7))]


def _embed(s, ns, n):
    """A lattice spectrum on the n^3 mesh's half spectrum."""
    out = torch.zeros(n, n, n // 2 + 1, dtype=torch.complex128, device=_dev())
    h = (ns + 1) // 2
    for a in (slice(0, h), slice(-h + 1, None) if h > 1 else slice(0, 0)):
        for b in (slice(0, h), slice(-h + 1, None) if h > 1 else slice(0, 0)):
            out[a, b, :h] = s[a, b, :h]
    return out


def _sd_factor(a, lnk):
    """Scale dependence of the growth, 1 + e(k, a), and its d/dln k."""
    x2 = np.exp(2 * (lnk - math.log(0.5)))
    e = 0.15 * a**3
    return 1 + e * x2 / (1 + x2), 2 * e * x2 / (1 + x2) ** 2


def _sd_growth(which, i, order, lnk):
    """(value, d/dln k) of the scale-dependent growth of one field: D, dD, ddD at step i or D(next) - D."""
    a = A0 + i * DA
    if which == "delta":
        v1, d1 = _sd_growth("D", i + 1, order, lnk)
        v0, d0 = _sd_growth("D", i, order, lnk)
        return v1 - v0, d1 - d0
    f, df = _sd_factor(a, lnk)
    r = _rates(a)[which][order]
    return (r * f, r * df) if order == 0 else (r * f * f, 2 * r * f * df)


def _sd_slice(case, which, i, order, keep):
    nk = 1000
    lnk0 = math.log(2 * math.pi / case["box"] / 2)
    dlnk = (math.log(2 * math.pi / case["box"] * case["nmesh"]) - lnk0) / (nk - 1)
    lnk = lnk0 + dlnk * np.arange(nk)
    den = _sd_factor(1.0, lnk)
    if order == 1:
        den = (den[0] ** 2, 2 * den[0] * den[1])
    arr = [np.ascontiguousarray(x) for x in _sd_growth(which, i, order, lnk) + den]
    keep.append(arr)
    p = [x.ctypes.data_as(M.C.POINTER(M.C.c_double)) for x in arr]
    return M.KSlice(lnk0, dlnk, nk, p[0], p[1], p[2], p[3], 1.0 if order == 0 else -3 / 7 / case["nmesh"] ** 3)


def _with_positions(case):
    return case["members"] * case["nsample"] ** 3 <= 1 << 18


def _pinned(np_, count):
    return [torch.empty(3, np_, dtype=torch.float32, pin_memory=torch.cuda.is_available()) for _ in range(count)]


def _ic_power(nmesh, box):
    return _power(2 * math.pi / box * np.sqrt(np.arange(M.n2_table_len(nmesh), dtype=np.float64)))


def prepare(case, seed):
    n, ns, box, kind = case["nmesh"], case["nsample"], case["box"], case["kind"]
    mgon = case["model"] != "lcdm"
    args = dict(model=MODELS[case["model"]], mg_active=int(mgon), include_screening=int(mgon and case["screening"]),
                filter=M.FILTER_GAUSSIAN if case["model"] == "dgp" else M.FILTER_NONE, scale_dependent=int(case["sd"]))
    if case["call"] == "batch":
        gs = M.MGPU.batch(case["members"], n, ns, box, OMEGA, **args)
    else:
        gs = [M.MGPU(n, ns, box, OMEGA, **args)]
    gs[0].autotune_fft()
    for g in gs[1:]:
        g.set_fft_tile(0, gs[0].fft_tile(0))
    state = dict(case=case, gs=gs, seed=seed, keep=[],
                 out=[_pinned(ns**3, 2 if kind == "ic" or _with_positions(case) else 1) for _ in gs])
    state["steps"] = [(_step_scalars(i), M.MG(**_mg(case["model"], A0 + i * DA)) if mgon else None)
                      for i in range(case["steps"])]
    if kind == "ic":
        state["pk"] = _ic_power(n, box)
    elif case["sd"]:
        if n <= 256:
            d, s = _spectra(ns, box, seed)
            gs[0].set_mesh(M.MESH_CDELTA1, _embed(d, ns, n).cpu().numpy())
            gs[0].set_mesh(M.MESH_CDELTA2, (-n**3 * _embed(s, ns, n)).cpu().numpy())
        else:
            gs[0].ic_displacement_fields(seed, _ic_power(n, box))

        def pair(which, i):
            return tuple(_sd_slice(case, which, i, o, state["keep"]) for o in (0, 1))
        state["start"] = (pair("D", 0), pair("dD", 0))
        state["slices"] = [(pair("ddD", i), pair("delta", i)) for i in range(case["steps"])]
    else:
        for r, g in enumerate(gs):
            for slot, f in enumerate(_lattice_fields(ns, box, seed + 1000003 * r)):
                g.set_lpt(slot, f.cpu().numpy())
        if kind == "output":
            g = gs[0]
            g.init_particles(*_rates(A0)["D"])
            vel = _output_velocities(ns, seed)
            M.lib().mgpu_set_particles(g.ctx, None, vel.data_ptr())
    return state


def _output_velocities(ns, seed):
    """Residual velocities of the particles at an output (a = 0.65)."""
    g = torch.Generator().manual_seed(int(seed) + 77)
    return (0.2 * torch.randn(3, ns**3, generator=g)).contiguous()


def _rsd_scalars(case):
    """vnorm and the LPT velocity terms at a = 0.65: mesh units per velocity unit."""
    r = _rates(A0)["dD"]
    return 1.0 / (A0 * A0 * _E(A0)) * case["nmesh"] / case["box"], r[0], r[1]


# ---------------------------------------------------------------- one pass
def run(state):
    case, gs = state["case"], state["gs"]
    g = gs[0]
    if case["kind"] == "ic":
        g.ic_displacement_fields(state["seed"], state["pk"])
        for slot, o in enumerate(state["out"][0]):
            M.lib().mgpu_get_lpt(g.ctx, slot, o.data_ptr())
        return {"lpt": state["out"][0]}
    if case["kind"] == "output":
        pk = g.pm_density(pofk=True)
        rsd = [g.rsd_power_spectrum(axis, *_rsd_scalars(case)) for axis in (1, 2)]
        return {"pofk": np.float32(pk), "rsd": np.float32(rsd)}
    if case["sd"]:
        M.lpt_fields_slices2(g, *state["start"])
    for m in gs:
        m.init_particles(*_rates(A0)["D"])
    spectra, sum_v = [], None
    for i, ((a, dda, dyyy, (k1, k2), (d1, d2)), mg) in enumerate(state["steps"]):
        if i > 0 and case["call"] != "separate":
            if case["call"] == "batch":
                M.MGPU.batch_step(gs, dda, a, k1, k2, dyyy, d1, d2, mg=mg)
            else:
                g.step(dda, a, k1, k2, dyyy, d1, d2, mg=mg, graph=case["call"] == "graph")
            continue
        for m in gs:
            sum_d, pk = m.get_displacements(mg, pofk=case["pofk"])
            if pk is not None:
                spectra.append(np.float32(pk))
            if case["sd"]:
                M.lpt_fields_slices2(m, *state["slices"][i])
            if i == 0:
                sum_v = m.kick(dda, a, k1, k2, sum_d)
                m.drift(dyyy, d1, d2, sum_v)
            else:
                sum_v = m.kick_drift(dda, a, k1, k2, sum_d, dyyy, d1, d2, sum_v)
    out = {}
    for r, (m, (vel, *pos)) in enumerate(zip(gs, state["out"])):
        M.lib().mgpu_get_particles(m.ctx, pos[0].data_ptr() if pos else None, vel.data_ptr())
        out["vel%d" % r] = vel
        if pos:
            out["pos%d" % r] = pos[0]
    if spectra:
        out["pofk"] = np.stack(spectra)
    return out


def work(case):
    """Per step each particle's position, velocity and LPT terms once and its new state; the transforms' operations."""
    n, np_ = case["nmesh"], case["nsample"] ** 3
    fft = 2.5 * n**3 * 3 * math.log2(n)
    if case["kind"] == "ic":
        return {"bytes": 24.0 * np_, "flops": 13 * fft}
    if case["kind"] == "output":
        return {"bytes": 72.0 * np_, "flops": 3 * fft}
    transforms = 6 if case["model"] in ("fofr", "dgp") and case["screening"] else 4
    per = transforms * fft + 300.0 * np_
    if case["sd"]:
        per += 6 * 2.5 * np_ * math.log2(np_)
    return {"bytes": case["members"] * (72.0 * np_ * case["steps"] + 12.0 * np_),
            "flops": case["members"] * per * case["steps"]}


# ---------------------------------------------------------------- the same in 64 bits
def _corners(x, n):
    i = torch.floor(x).long()
    d = x - i
    i = i % n
    j = (i + 1) % n
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                w = (d[0] if a else 1 - d[0]) * (d[1] if b else 1 - d[1]) * (d[2] if c else 1 - d[2])
                yield ((j[0] if a else i[0]) * n + (j[1] if b else i[1])) * n + (j[2] if c else i[2]), w


def _deposit(x, n, ns):
    rho = torch.zeros(n**3, dtype=torch.float64, device=x.device)
    for idx, w in _corners(x, n):
        rho.index_add_(0, idx, w)
    return (rho * (n / ns) ** 3 - 1).reshape(n, n, n)


def _gather(mesh, x, n):
    m = mesh.reshape(-1)
    return sum(m[idx] * w for idx, w in _corners(x, n))


def _bins(dk, n, box, ns, moments):
    """Sums over the linear |n| bins (width 1, n of them): P, mu^2 and mu^4 moments, |n|, count."""
    k = _grid(n)
    n2 = (k[0] ** 2 + k[1] ** 2 + k[2] ** 2)
    kmag = n2.sqrt()
    b = (kmag + 0.5).long()
    w = torch.full_like(k[2], 2.0)
    w[..., 0] = w[..., -1] = 1.0
    w = (w + 0 * kmag)
    p = dk.real**2 + dk.imag**2
    for q in k:
        t = math.pi * q.abs() / n
        p = p * torch.where(t > 0, (t / torch.sin(t.clamp(min=1e-30))) ** 4, torch.ones_like(t))
    mu2 = torch.where(n2 > 0, k[2] ** 2 / n2.clamp(min=1), torch.zeros_like(n2))
    b, w, p, mu2, kmag = (v[..., :].reshape(-1) for v in (b, w, p * w / float(n) ** 6, mu2, kmag))
    ok = b < n

    def s(v):
        return torch.bincount(b[ok], weights=v[ok], minlength=n)[:n]
    cnt = s(w)
    sums = [s(p), s(p * mu2), s(p * mu2**2)] if moments else [s(p)]
    safe = cnt.clamp(min=1)
    full = cnt > 0
    return [torch.where(full, v / safe * box**3, v) for v in sums], torch.where(
        full, s(kmag * w) / safe * 2 * math.pi / box, torch.zeros_like(cnt)), cnt, full, (box / ns) ** 3


def _pofk(dk, n, box, ns):
    (p,), k, cnt, full, shot = _bins(dk, n, box, ns, False)
    return torch.stack([torch.where(full, p - shot, p), k, cnt]).cpu().numpy()


def _rsd(pos, vel, fields, case, axis):
    n, ns, box = case["nmesh"], case["nsample"], case["box"]
    vnorm, s1, s2 = _rsd_scalars(case)
    x = pos * (n / box)
    z = (x[axis] + vnorm * (vel[axis] + fields[0][axis] * s1 + fields[1][axis] * s2)) % n
    dk = torch.fft.rfftn(_deposit(torch.stack([x[0], x[3 - axis], z]), n, ns))
    (p0, p2, p4), _, cnt, full, shot = _bins(dk, n, box, ns, True)
    p4 = 9 * (35 * p4 - 30 * p2 + 3 * p0) / 8
    p2 = 5 * (3 * p2 - p0) / 2
    k = torch.arange(n, device=cnt.device, dtype=torch.float64) * 2 * math.pi / box
    return torch.stack([torch.where(full, v, torch.zeros_like(v)) for v in (p0 - shot, p2 - shot, p4 - shot, k)]
                       + [cnt]).cpu().numpy()


def _force(delta, dk, case, mg):
    """The three force meshes of delta(x), with the model's fifth force."""
    n, box = case["nmesh"], case["box"]
    k = _grid(n)
    n2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    inv = torch.where(n2 > 0, 1 / n2.clamp(min=1), torch.zeros_like(n2))
    p, model = dk, case["model"]
    if model == "jbd":
        p = dk * mg["geff"]
    elif model == "fofr":
        m2 = mg["a"] ** 2 * mg["mass2"] / (2 * math.pi * C_H0 / box) ** 2
        eff = dk
        if case["screening"]:
            phi = _c2r(-dk * inv, n) * (1.5 * OMEGA / mg["a"] * (box / C_H0 / (2 * math.pi)) ** 2 / float(n) ** 3)
            s = torch.where(phi < 0, (mg["phi_crit"] / phi.clamp(max=-1e-300)).abs().clamp(max=1.0),
                            torch.ones_like(phi))
            eff = torch.fft.rfftn(delta * s)
        p = dk + mg["coupling"] * n2 / (n2 + m2) * eff * (n2 > 0)
    elif model == "dgp":
        if case["screening"]:
            kr = n2.sqrt() * (2 * math.pi / box * mg["rsmooth"])
            f = mg["dgp_fac"] * (1 + _c2r(dk * torch.exp(-0.5 * kr * kr), n) / float(n) ** 3)
            s = torch.where(f < 1e-5, torch.ones_like(f), 2 * ((1 + f.clamp(min=-1)).sqrt() - 1) / f)
            p = dk + torch.fft.rfftn(delta * s * mg["coupling"])
        else:
            p = dk * (1 + mg["coupling"])
    for a in range(3):
        yield _c2r(-1j * k[a] * inv * p, n) / (float(n) ** 3 * 2 * math.pi / box)


def _exact_run(case, fields, sd_fields):
    n, ns, box = case["nmesh"], case["nsample"], case["box"]
    g = torch.arange(ns, device=_dev(), dtype=torch.float64) * (box / ns)
    q = torch.stack([t.reshape(-1) for t in torch.meshgrid(g, g, g, indexing="ij")])
    r = _rates(A0)["D"]
    pos = (q + (sd_fields("D", 0) if case["sd"] else fields[0].double() * r[0] + fields[1].double() * r[1])) % box
    vel, spectra, sum_v = torch.zeros_like(pos), [], 0.0
    for i in range(case["steps"]):
        a, dda, dyyy, (k1, k2), (d1, d2) = _step_scalars(i)
        x = pos * (n / box)
        delta = _deposit(x, n, ns)
        dk = torch.fft.rfftn(delta)
        if case["pofk"]:
            spectra.append(_pofk(dk, n, box, ns))
        disp = torch.stack([_gather(f, x, n) for f in _force(delta, dk, case, _mg(case["model"], a))])
        if case["sd"]:
            lk, ld = sd_fields("ddD", i), sd_fields("delta", i)
        else:
            lk, ld = (fields[0].double() * u + fields[1].double() * v for u, v in ((k1, k2), (d1, d2)))
        new = vel + dda * (-1.5 * OMEGA * (disp - disp.mean(1, keepdim=True)) - lk / a)
        sum_v = new.mean(1, keepdim=True) if i == 0 else sum_v
        vel, pos = new, (pos + (new - sum_v) * dyyy + ld) % box
        sum_v = vel.mean(1, keepdim=True)
    return pos, vel, spectra


def _ranlux(seeds, draws):
    """`draws` uniforms of each seed's stream: the 48-bit RANLUX of Luescher (1994), luxury 202 of 12."""
    s = seeds.to(torch.int64)
    bits = [(torch.where(s == 0, torch.ones_like(s), s) >> k) & 1 for k in range(31)]
    one, y, i, j = 2.0**-48, [], 0, 18
    for _ in range(12):
        x = torch.zeros(s.shape, dtype=torch.float64, device=s.device)
        for _ in range(48):
            x = 2 * x + (bits[i] ^ 1)
            bits[i] = bits[i] ^ bits[j]
            i, j = (i + 1) % 31, (j + 1) % 31
        y.append(x * one)
    c = torch.zeros_like(y[0])
    while draws > 0:
        for t in range(202):
            v = y[(t + 7) % 12] - y[t % 12] - c
            low = v < 0
            y[t % 12] = torch.where(low, v + 1, v)
            c = low * one
        y = y[10:] + y[:10]
        for t in y[:draws]:
            yield t
        draws -= 12


def _seed_table(n, seed):
    """The n^2 column seeds, drawn shell by shell so that small wavenumbers keep theirs on any mesh."""
    r = _ranlux(torch.tensor([seed % 2**32]), n * n)
    t = np.zeros((n, n), np.int64)
    for i in range(n // 2):
        for flip_i, flip_j in ((0, 0), (1, 0), (0, 1), (1, 1)):
            for swap in (0, 1):
                for j in range(i + swap):
                    a, b = (j, i) if swap else (i, j)
                    t[n - 1 - a if flip_i else a, n - 1 - b if flip_j else b] = int(0x7FFFFFFF * float(next(r)))
    return torch.from_numpy(t).to(_dev())


def _exact_ic(case, seed):
    n, ns, box = case["nmesh"], case["nsample"], case["box"]
    h = n // 2
    k = _grid(n, -1)
    pk = torch.from_numpy(_ic_power(n, box)).to(_dev())
    seeds = _seed_table(n, seed)
    cd = torch.zeros(n, n, h + 1, dtype=torch.complex128, device=_dev())
    ki, kj = k[0][:, :, 0], k[1][:, :, 0]
    stream = _ranlux(seeds, n)
    for z in range(h):
        phase, ampl = next(stream) * 2 * math.pi, next(stream)
        n2 = (ki**2 + kj**2 + z * z).long().clamp(max=pk.numel() - 1)
        d = torch.sqrt(-torch.log(ampl) * pk[n2]) * box**-1.5
        use = (ki.abs() <= ns // 2) & (kj.abs() <= ns // 2) & (z <= ns // 2) & (ki != -h) & (kj != -h)
        v = torch.where(use & (n2 > 0), torch.polar(d, phase), torch.zeros_like(cd[:, :, 0]))
        if z == 0:  # the kz = 0 plane: half of it drawn, the other half conjugate
            half = torch.zeros_like(v)
            half[1:h], half[0, :h] = v[1:h], v[0, :h]
            v = half + torch.roll(half.flip(0, 1), (1, 1), (0, 1)).conj()
        cd[:, :, z] = v
    n2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    inv = torch.where(n2 > 0, 1 / n2.clamp(min=1), torch.zeros_like(n2))
    d = [_c2r(-k[a] * k[a] * inv * cd, n) for a in range(3)]
    src = d[0] * (d[1] + d[2]) + d[1] * d[2]
    for a, b in ((0, 1), (0, 2), (1, 2)):
        src -= _c2r(-k[a] * k[b] * inv * cd, n) ** 2
    sk = torch.fft.rfftn(src, norm="forward")
    g = torch.arange(ns, device=_dev(), dtype=torch.float64)
    q = torch.stack([t.reshape(-1) for t in torch.meshgrid(g, g, g, indexing="ij")])
    lpt = []
    for s, c in ((cd, 1.0), (sk, 3 / 7)):
        f = torch.stack([_gather(_c2r(1j * k[a] * inv * s, n), q * n / ns, n) for a in range(3)])
        f = f * (c * box / (2 * math.pi))
        lpt.append(f - f.mean(1, keepdim=True))
    return {"lpt": [t.cpu().numpy() for t in lpt]}


def exact(case, seed):
    n, ns, box = case["nmesh"], case["nsample"], case["box"]
    if case["kind"] == "ic":
        return _exact_ic(case, seed)
    if n > 768:
        return None  # the spectra of a 1024^3 mesh's initial conditions alone take longer than this may
    if case["kind"] == "output":
        f = _lattice_fields(ns, box, seed)
        one = dict(case, steps=0)
        pos, _, _ = _exact_run(one, f, None)
        vel = _output_velocities(ns, seed).to(_dev()).double()
        fd = [t.double() for t in f]
        return {"pofk": _pofk(torch.fft.rfftn(_deposit(pos * (n / box), n, ns)), n, box, ns),
                "rsd": np.stack([_rsd(pos, vel, fd, case, axis) for axis in (1, 2)])}
    out = {}
    for r in range(case["members"]):
        fields = sd_fields = None
        if case["sd"]:
            dk, sk = (s.to(torch.complex64).to(torch.complex128) for s in _spectra(ns, box, seed))
            k = _grid(ns)
            n2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2

            def sd_fields(which, i):
                lnk = np.log(2 * math.pi / box) + 0.5 * np.log(np.maximum(n2.cpu().numpy(), 1))
                fac = _sd_factor(1.0, lnk)[0]
                g1 = torch.from_numpy(_sd_growth(which, i, 0, lnk)[0] / fac).to(_dev())
                g2 = torch.from_numpy(_sd_growth(which, i, 1, lnk)[0] / fac**2).to(_dev())
                s = (g1 * dk + 3 / 7 * g2 * sk) / n2.clamp(min=1) * (box / (2 * math.pi))
                return torch.stack([_c2r(1j * k[a] * s, ns).reshape(-1) for a in range(3)])
        else:
            fields = _lattice_fields(ns, box, seed + 1000003 * r)
        pos, vel, spectra = _exact_run(case, fields, sd_fields)
        out["vel%d" % r] = vel.cpu().numpy()
        if _with_positions(case):
            out["pos%d" % r] = pos.cpu().numpy()
    if spectra:
        out["pofk"] = np.stack(spectra)
    return out
