"""Work that users of this framework have it do, measured through its public entry points.

Four kinds of case:

- ``run``: one simulation stepped on and its results read back (``fields.step`` for the
  shortest, ``fields.step_n`` for the others).  Options are those simulations differ in: 2D
  TM, 2D TE and 3D; FP64 (the reference's default) and FP32; uPML on every face, or a periodic
  cell with real fields (k = 0), or with a Bloch vector and so complex fields; no dispersive
  material, a Drude metal, or a Lorentz-Drude medium in half of the cell; a point dipole or a
  current sheet; flux spectra or DFT field maps.
- ``batch``: many uneven 2D simulations stepped together.
- ``gradient``: one iteration of a topology optimisation, the objective and its gradient by
  the reverse mode through ``meep_amd.autograd``.
- ``far``: the near-to-far transformation of a finished run, on a far plane or at the points of
  a radiation pattern one by one.

``exact`` is the same physics in plain torch, FP64, written from the published scheme (Yee's
leapfrog with uPML, auxiliary-equation poles, discrete Fourier sums, the homogeneous-medium
Green's functions).
"""

import math

import numpy as np
import torch

import meep_amd
from meep_amd import autograd, capi

RES = 10.0        # pixels per unit length
COURANT = 0.5
EPS_LO, EPS_HI = 1.0, 5.0
BLOCK = 8         # cells per side of the random dielectric blocks
# (resonance, damping, Drude?, sigma) of the poles, in the order they are added
POLES = {"none": (), "drude": ((1.0, 0.1, True, 3.0),),
         "lorentz-drude": ((1.0, 0.05, False, 1.5), (1.0, 0.1, True, 3.0))}
GRAD_RES = 50.0
FAR_RES = 10.0


def listed():
    return [
        # an interactive script or a step function called every step: one step of a small cell,
        # then the field map; latency and launches are all of it
        dict(name="step_tm_96x64_f64", kind="run", dim="tm", nx=96, ny=64, nz=0, pml=10, bloch="none", poles="none",
             prec="f64", steps=1, source="point", out="map", nfreq=0),
        # the straight waveguide of the tests (320 x 160, uPML, 100 flux frequencies), FP64
        dict(name="flux_tm_320x160_f64", kind="run", dim="tm", nx=320, ny=160, nz=0, pml=10, bloch="none", poles="none",
             prec="f64", steps=400, source="point", out="flux", nfreq=100),
        # a plasmonic 2D cell of odd size: TE fields, half of it a Drude metal
        dict(name="metal_te_401x263_f32", kind="run", dim="te", nx=401, ny=263, nz=0, pml=12, bloch="none",
             poles="drude", prec="f32", steps=400, source="point", out="dft", nfreq=4),
        # a parameter sweep: 64 small 2D simulations of uneven size, together
        dict(name="batch_64_tm_f32", kind="batch", count=64, lo=128, hi=512, pml=10, prec="f32", steps=400, nfreq=16),
        # a topology-optimisation iteration: forward run, objective, reverse sweep
        dict(name="gradient_400x300_f32", kind="gradient", nx=400, ny=300, pml=40, design=140, steps=1200, nfreq=10,
             prec="f32"),
        # scattering in 3D: a dipole among dielectric blocks inside uPML, a closed flux box;
        # an odd size, launch-bound
        dict(name="flux_3d_131x118x125_f32", kind="run", dim="3d", nx=131, ny=118, nz=125, pml=12, bloch="none",
             poles="none", prec="f32", steps=400, source="point", out="fluxbox", nfreq=20),
        # a periodic cell, real fields: the bandwidth case
        dict(name="periodic_3d_256_f32", kind="run", dim="3d", nx=256, ny=256, nz=256, pml=0, bloch="real",
             poles="none", prec="f32", steps=200, source="point", out="dft", nfreq=2),
        # the same at an odd, uneven size in FP64
        dict(name="periodic_3d_187x203x190_f64", kind="run", dim="3d", nx=187, ny=203, nz=190, pml=0, bloch="real",
             poles="none", prec="f64", steps=100, source="point", out="dft", nfreq=2),
        # a band-structure cell: a Bloch vector, so complex fields and phase-shifted halos
        dict(name="bloch_3d_96x72x80_f64", kind="run", dim="3d", nx=96, ny=72, nz=80, pml=0, bloch="complex",
             poles="none", prec="f64", steps=100, source="point", out="dft", nfreq=2),
        # the largest: the benchmark's cell with uPML, a Lorentz-Drude medium in the lower half, a current
        # sheet and a DFT map with compensated FP32 accumulators
        dict(name="medium_3d_384x384x192_f32", kind="run", dim="3d", nx=384, ny=384, nz=192, pml=16, bloch="none",
             poles="lorentz-drude", prec="f32", steps=200, source="sheet", out="dft", nfreq=8),
        # the fields on a far plane above a six-face box
        dict(name="far_3d_plane", kind="far", dim=3, cells=64, half=20, nfreq=10, points=64, one_by_one=False),
        # a 2D radiation pattern, one call per angle
        dict(name="far_2d_pattern", kind="far", dim=2, cells=120, half=40, nfreq=8, points=60, one_by_one=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run2d", "run2d", "run3d", "run3d", "run3d", "batch", "gradient", "far"])
    if kind == "run2d":
        nx, ny = _log(rng, 60, 640), _log(rng, 60, 480)
        return dict(kind="run", dim=rng.choice(["tm", "te"]), nx=nx, ny=ny, nz=0, pml=rng.randint(8, 14), bloch="none",
                    poles=rng.choice(["none", "none", "drude", "lorentz-drude"]), prec=rng.choice(["f64", "f32"]),
                    steps=_log(rng, 120, 400), source=rng.choice(["point", "sheet"]),
                    out=rng.choice(["flux", "dft", "map"]), nfreq=rng.randint(1, 40))
    if kind == "run3d":
        edge = rng.choice(["pml", "pml", "real", "complex"])
        cap = 5.0e6 if edge != "complex" else 8.0e5
        while True:
            n = [_log(rng, 50, 300) for _ in range(3)]
            if 1.5e5 <= n[0] * n[1] * n[2] <= cap:
                break
        poles = rng.choice(["none", "none", "drude", "lorentz-drude"]) if edge == "pml" else "none"
        source = rng.choice(["point", "sheet"]) if edge == "pml" else "point"
        return dict(kind="run", dim="3d", nx=n[0], ny=n[1], nz=n[2], pml=rng.randint(6, 11) if edge == "pml" else 0,
                    bloch="none" if edge == "pml" else edge, poles=poles, prec=rng.choice(["f64", "f32"]),
                    steps=rng.randint(100, 200), source=source,
                    out=rng.choice(["flux", "fluxbox" if source == "point" else "dft", "dft"]) if edge == "pml" else "dft",
                    nfreq=rng.randint(1, 8))
    if kind == "batch":
        lo = rng.randint(60, 160)
        return dict(kind="batch", count=_log(rng, 4, 64), lo=lo, hi=lo + rng.randint(20, 300), pml=rng.randint(8, 12),
                    prec=rng.choice(["f32", "f64"]), steps=rng.randint(100, 300), nfreq=rng.randint(4, 20))
    if kind == "gradient":
        nx, ny = rng.randint(200, 400), rng.randint(160, 300)
        return dict(kind="gradient", nx=nx, ny=ny, pml=rng.randint(20, 40),
                    design=min(nx, ny) // 3 + rng.randint(0, 10), steps=rng.randint(600, 1000),
                    nfreq=rng.randint(2, 12), prec=rng.choice(["f32", "f64"]))
    if rng.random() < 0.5:
        return dict(kind="far", dim=3, cells=rng.randint(44, 64), half=rng.randint(8, 18), nfreq=rng.randint(1, 11),
                    points=rng.randint(12, 56), one_by_one=False)
    return dict(kind="far", dim=2, cells=rng.randint(70, 140), half=rng.randint(12, 24), nfreq=rng.randint(1, 12),
                points=rng.randint(20, 80), one_by_one=rng.random() < 0.5)


# ---- the simulation a case describes, as plain data ---------------------------------------
# (used by prepare to set the framework up and by exact to compute the same)

def _dims(case):
    """Cells per direction X, Y, Z (0: no such direction)."""
    return case["nx"], case["ny"], case["nz"] if case["dim"] == "3d" else 0


def _components(case):
    return {"tm": ("Ez", "Hx", "Hy"), "te": ("Hz", "Ex", "Ey"),
            "3d": ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")}[case["dim"]]


def _plan(case, seed):
    """Everything random or derived about a ``run`` case."""
    rng = np.random.default_rng([seed, 11])
    n = _dims(case)
    dirs = [d for d in range(3) if n[d]]
    nb = [-(-(n[d] + 1) // BLOCK) for d in dirs]
    inv_eps = 1.0 / rng.uniform(EPS_LO, EPS_HI, size=nb)
    dt = COURANT / RES
    span = max(case["steps"], 60) * dt  # the pulse peaks within the first pass
    fcen = rng.uniform(0.35, 0.45) if case["dim"] != "3d" else rng.uniform(0.5, 0.7)
    fwidth = 1.2 * fcen
    size = [n[d] / RES for d in range(3)]
    comp = {"tm": "Ez", "te": "Hz", "3d": "Ex"}[case["dim"]]
    if case["source"] == "point":
        at = [0.5 * size[d] + 0.3 * rng.uniform(-1, 1) if n[d] else 0.0 for d in range(3)]
        where = (tuple(at), tuple(at))
    else:  # a sheet (2D: a line) across the whole cell, normal to its last direction
        last = dirs[-1]
        at = round(n[last] * 5 / 6) / RES
        where = (tuple(at if d == last else 0.0 for d in range(3)), tuple(at if d == last else size[d] for d in range(3)))
    k = tuple(rng.uniform(0.1, 0.4, size=3) * RES / np.maximum(n, 1)) if case["bloch"] == "complex" else None
    freqs = np.linspace(0.8 * fcen, 1.2 * fcen, case["nfreq"]) if case["nfreq"] > 1 else np.array([fcen] * case["nfreq"])
    return dict(n=n, dirs=dirs, inv_eps=inv_eps, dt=dt, size=size, comp=comp, where=where, k=k, freqs=freqs,
                fcen=fcen, fwidth=fwidth, peak=min(0.4 * span, 3.0))


def _eps_map(p):
    """1/eps at every point of a component's array: random blocks of 8 cells a side."""
    at = np.ix_(*[np.arange(p["n"][d] + 1) // BLOCK for d in p["dirs"]])
    return np.ascontiguousarray(p["inv_eps"][at])


def _medium_lines(case, p, value):
    """A pole's sigma as a product of one factor per direction: ``value`` over the lower half
    along the last direction, clear of the uPML, in which a metal's waves grow without bound
    over the thousands of steps that passes add up to."""
    m = case["pml"] + 2
    out = []
    for d in p["dirs"]:
        j = np.arange(p["n"][d] + 1)
        last = d == p["dirs"][-1]
        hi = p["n"][d] // 2 if last else p["n"][d] + 1 - m
        out.append(np.where((j >= m) & (j < hi), value if last else 1.0, 0.0))
    return out


def _medium_map(case, p, value):
    v = np.array(1.0)
    for q in _medium_lines(case, p, value):
        v = np.multiply.outer(v, q)
    return v


def _volumes(case, p):
    """The monitors of the case: (direction or None, low corner, high corner)."""
    n, size = p["n"], p["size"]
    if case["out"] == "flux":  # across the cell inside the uPML, a unit from the source
        m = (case["pml"] + 4) / RES
        across = 0 if case["source"] == "point" else p["dirs"][-1]
        x = p["where"][0][across] - 1.03
        lo = tuple(x if d == across else (m if n[d] else 0.0) for d in range(3))
        hi = tuple(x if d == across else (size[d] - m if n[d] else 0.0) for d in range(3))
        return [(across, lo, hi)]
    if case["out"] == "fluxbox":  # the faces of a closed box around the source
        h = min([2.53] + [0.5 * size[d] - (case["pml"] + 3) / RES for d in p["dirs"]])
        out = []
        for d in p["dirs"]:
            for x in (-h, h):
                lo = tuple(0.5 * size[q] + (x if q == d else -h) if n[q] else 0.0 for q in range(3))
                hi = tuple(0.5 * size[q] + (x if q == d else h) if n[q] else 0.0 for q in range(3))
                out.append((d, lo, hi))
        return out
    if case["out"] == "dft":  # the whole cross-section (2D: the whole cell), on the centred grid
        last = p["dirs"][-1]
        plane = (n[last] // 2 + 0.5) / RES
        flat = len(p["dirs"]) == 3
        lo = tuple(0.0 if not n[d] else plane if flat and d == last else 0.5 / RES for d in range(3))
        hi = tuple(0.0 if not n[d] else plane if flat and d == last else (n[d] - 0.5) / RES for d in range(3))
        return [(None, lo, hi)]
    return []


def _mapped(case):
    """The components whose DFT map is taken."""
    return {"tm": ["Ez"], "te": ["Hz"], "3d": ["Ex", "Ey", "Ez"]}[case["dim"]]


def _component(name):
    return getattr(capi, name)


def _source(fcen, fwidth, peak):
    """A Gaussian pulse that peaks at time ``peak``."""
    return capi.gaussian_src_time(fcen, fwidth, start_time=peak - 5.0 / fwidth)


def _real(case, v):
    """A result in the precision that the simulation runs in."""
    if case["prec"] == "f64":
        return v
    return v.astype(np.complex64 if np.iscomplexobj(v) else np.float32)


# ---- prepare and run ------------------------------------------------------------------------

def _prepare_run(case, seed):
    lib = meep_amd.load_library()
    p = _plan(case, seed)
    single = case["prec"] == "f32"
    s = capi.structure(lib, dim=len(p["dirs"]), size=p["size"][:len(p["dirs"])], a=RES, courant=COURANT, single=single,
                       pml=[t for d in p["dirs"] for t in capi.pml(case["pml"] / RES, d)] if case["pml"] else ())
    electric = [c for c in _components(case) if c[0] == "E"]
    chi = _eps_map(p)
    for c in electric:
        s.set_chi1inv(_component(c), chi)
    del chi
    for f0, gamma, drude, sigma in POLES[case["poles"]]:
        i = s.add_susceptibility(None, f0, gamma, drude=drude)
        sig = _medium_map(case, p, sigma)
        for c in electric:
            s.set_sigma(i, _component(c), sig)
        del sig
    f = capi.fields(s)
    if case["bloch"] == "complex":
        f.use_bloch(p["k"])
    else:
        if case["bloch"] == "real":
            f.use_bloch((0.0, 0.0, 0.0))
        f.use_real_fields()
    f.add_volume_source(_component(p["comp"]), _source(p["fcen"], p["fwidth"], p["peak"]), *p["where"])
    f.set_dft_accumulator(capi.DFT_KAHAN32 if single else capi.DFT_F64)
    mons = []
    for d, lo, hi in _volumes(case, p):
        if d is None:
            mons.append(f.add_dft_fields([_component(c) for c in _mapped(case)], lo, hi, p["freqs"], decimation_factor=1))
        else:
            mons.append(f.add_dft_flux(d, lo, hi, p["freqs"], decimation_factor=1))
    return dict(case=case, s=s, f=f, mons=mons)


def _run_run(st):
    case, f, mons = st["case"], st["f"], st["mons"]
    if case["steps"] == 1:
        f.step()
    else:
        f.step_n(case["steps"])
    out = []
    if case["out"] == "dft":
        out = [_real(case, mons[0].dft(i)) for i in range(mons[0].num_chunks())]
    elif case["out"] != "map":
        out = [_real(case, m.flux()) for m in mons]
    if case["dim"] != "3d":  # the field as it stands, as one plots it
        out.append(_real(case, f.get_array(_component(_components(case)[0]))[0]))
    return out


def _batch_layout(case, seed):
    rng = np.random.default_rng([seed, 12])
    sides = rng.integers(case["lo"], case["hi"] + 1, size=case["count"])
    sims = []
    for side in sides:
        nb = -(-(int(side) + 1) // 16)
        sims.append(dict(side=int(side), fcen=rng.uniform(0.2, 0.4), inv_eps=1.0 / rng.uniform(EPS_LO, EPS_HI, size=(nb, nb))))
    return sims


def _batch_line(case, side):
    """Source point and flux line of one simulation of a batch."""
    m = (case["pml"] + 4) / RES
    size = side / RES
    return (size - m - 1.2, size / 2, 0.0), (size - m, m, 0.0), (size - m, size - m, 0.0)


def _batch_pulse(case, fcen):
    span = case["steps"] * COURANT / RES
    return fcen, 1.5 * fcen, min(0.3 * span, 3.0)


def _prepare_batch(case, seed):
    lib = meep_amd.load_library()
    sims = []
    for q in _batch_layout(case, seed):
        size = q["side"] / RES
        s = capi.structure(lib, dim=2, size=(size, size), a=RES, courant=COURANT, pml=capi.pml(case["pml"] / RES)[:4],
                           single=case["prec"] == "f32")
        b = np.arange(q["side"] + 1) // 16
        s.set_chi1inv(capi.Ez, q["inv_eps"][np.ix_(b, b)])
        f = capi.fields(s)
        f.use_real_fields()
        f.set_dft_accumulator(capi.DFT_F64)
        at, lo, hi = _batch_line(case, q["side"])
        f.add_volume_source(capi.Ez, _source(*_batch_pulse(case, q["fcen"])), at, at)
        fl = f.add_dft_flux(capi.X, lo, hi, np.linspace(0.9 * q["fcen"], 1.1 * q["fcen"], case["nfreq"]), decimation_factor=1)
        sims.append((s, f, fl))
    return dict(case=case, sims=sims, batch=capi.batch([f for _, f, _ in sims]))


def _run_batch(st):
    st["batch"].step_n(st["case"]["steps"])
    return _real(st["case"], np.stack([fl.flux() for _, _, fl in st["sims"]]))


def _grad_layout(case):
    """Positions of the optimisation cell: the design square in the middle, a line source on its
    left, the objective's line on its right."""
    a = GRAD_RES
    nx, ny, nd, m = case["nx"], case["ny"], case["design"], case["pml"]
    x0, y0 = (nx - nd) // 2, (ny - nd) // 2
    left, right = (m + x0) // 2, nx - (m + x0) // 2
    return dict(x0=x0, y0=y0, src=((left / a, y0 / a, 0.0), (left / a, (y0 + nd) / a, 0.0)),
                mon=((right / a, (ny // 2 - 20) / a, 0.0), (right / a, (ny // 2 + 20) / a, 0.0)),
                design=((x0 / a, y0 / a, 0.0), ((x0 + nd - 1) / a, (y0 + nd - 1) / a, 0.0)),
                freqs=np.linspace(0.8, 1.2, case["nfreq"]))


def _grad_design(case, seed):
    """1/eps of a smooth random density between vacuum and eps = 6."""
    rng = np.random.default_rng([seed, 13])
    nd = case["design"]
    r = rng.uniform(0.0, 1.0, size=(nd, nd))
    k = np.fft.fftfreq(nd)
    g = np.exp(-2 * (np.pi * 5.0) ** 2 * (k[:, None] ** 2 + k[None, :] ** 2))
    r = np.real(np.fft.ifft2(np.fft.fft2(r) * g))
    r = (r - r.min()) / max(r.max() - r.min(), 1e-12)
    return 1.0 / (1.0 + 5.0 * r)


def _grad_build(lib, case, chi):
    g = _grad_layout(case)
    a = GRAD_RES
    s = capi.structure(lib, dim=2, size=(case["nx"] / a, case["ny"] / a), a=a, courant=COURANT,
                       pml=capi.pml(case["pml"] / a)[:4], single=case["prec"] == "f32")
    s.set_chi1inv(capi.Ez, np.full(s.shape, 0.9) if chi is None else chi)
    f = capi.fields(s)
    f.use_real_fields()
    f.add_volume_source(capi.Ez, _source(1.0, 0.5, 2.0), *g["src"])
    mon = f.add_dft_fields([capi.Ez], *g["mon"], g["freqs"], decimation_factor=1)
    return s, f, mon


def _prepare_gradient(case, seed):
    lib = meep_amd.load_library()
    g = _grad_layout(case)
    prob = autograd.Problem(lib, lambda L, chi: _grad_build(L, case, chi), (capi.Ez,) + g["design"], case["steps"])
    dtype = torch.float32 if case["prec"] == "f32" else torch.float64
    chi = torch.as_tensor(_grad_design(case, seed), dtype=dtype, device="cuda").requires_grad_(True)
    prob.base_chi()
    return dict(prob=prob, chi=chi)


def _run_gradient(st):
    J = autograd.fdtd_objective(st["chi"], st["prob"])
    (g,) = torch.autograd.grad(J, st["chi"])
    return dict(J=J.detach(), grad=g)


def _far_layout(case, seed):
    rng = np.random.default_rng([seed, 14])
    dim, size = case["dim"], case["cells"] / FAR_RES
    c, h = size / 2, (case["half"] + 0.3) / FAR_RES
    box = []
    for d in range(dim):
        for sgn in (1.0, -1.0):
            lo = [c - h if q < dim else 0.0 for q in range(3)]
            hi = [c + h if q < dim else 0.0 for q in range(3)]
            lo[d] = hi[d] = c + sgn * h
            box.append((tuple(lo), tuple(hi), sgn, d))
    fcen = rng.uniform(0.45, 0.55)
    freqs = np.linspace(0.85 * fcen, 1.15 * fcen, case["nfreq"]) if case["nfreq"] > 1 else np.array([fcen])
    at = [c + h * rng.uniform(-0.4, 0.4) if q < dim else 0.0 for q in range(3)]
    if dim == 3:
        lo, hi = (c - 20.0, c - 20.0, c + 28.0), (c + 20.0, c + 20.0, c + 28.0)
    else:
        lo, hi = (c - 40.0, c + 60.0, 0.0), (c + 40.0, c + 60.0, 0.0)
    n = case["points"]
    axis = [np.linspace(lo[q], hi[q], n) if hi[q] > lo[q] else np.array([lo[q]]) for q in range(3)]
    # a far grid has max(1, int(length * resolution)) points, spread from end to end
    res = (n + 0.5) / (hi[0] - lo[0])
    if case["one_by_one"]:
        ang = 2 * np.pi * np.arange(n) / n
        pts = np.stack([c + 1000.0 * np.cos(ang), c + 1000.0 * np.sin(ang), np.zeros(n)], axis=1)
    else:
        g = np.meshgrid(*axis, indexing="ij")
        pts = np.stack([q.ravel() for q in g], axis=1)
    return dict(size=size, box=box, freqs=freqs, fcen=fcen, at=tuple(at), lo=lo, hi=hi, res=res, pts=pts, steps=100)


def _prepare_far(case, seed):
    lib = meep_amd.load_library()
    p = _far_layout(case, seed)
    dim = case["dim"]
    s = capi.structure(lib, dim=dim, size=(p["size"],) * dim, a=FAR_RES, courant=COURANT,
                       pml=capi.pml(1.0)[:2 * dim])
    f = capi.fields(s)
    f.use_real_fields()
    f.add_volume_source(capi.Ez, _source(p["fcen"], p["fcen"], 2.0), p["at"], p["at"])
    n2f = f.add_dft_near2far(p["box"], p["freqs"], decimation_factor=1)
    f.step_n(p["steps"])
    return dict(case=case, s=s, f=f, n2f=n2f, p=p, pts=[tuple(float(x) for x in q) for q in p["pts"]])


def _run_far(st):
    n2f, p = st["n2f"], st["p"]
    if st["case"]["one_by_one"]:
        return np.stack([n2f.farfield(x) for x in st["pts"]])
    return n2f.get_farfields_array(p["lo"], p["hi"], p["res"])[0]


def prepare(case, seed):
    return {"run": _prepare_run, "batch": _prepare_batch, "gradient": _prepare_gradient, "far": _prepare_far}[case["kind"]](case, seed) | {"kind": case["kind"]}


def run(state):
    return {"run": _run_run, "batch": _run_batch, "gradient": _run_gradient, "far": _run_far}[state["kind"]](state)


# ---- what a pass cannot do without ----------------------------------------------------------

def _step_work(n, pml, npoles, word, cmps=1):
    """Bytes and operations of one step: every field of the state (D, E, B, and where uPML or a
    pole acts its auxiliaries and polarisations) read and written once, 1/eps read once."""
    dirs = [x for x in n if x]
    cells = float(np.prod(dirs))
    three = len(dirs) == 3
    inner = float(np.prod([max(x - 2 * pml, 0) for x in dirs]))
    words = (21 if three else 7) * cells + (12 if three else 4) * npoles * cells / 2 + (10 if three else 6) * (cells - inner)
    return words * word * cmps, (36 if three else 12) * cells * cmps + (30 if three else 10) * npoles * cells / 2


def work(case):
    word = 4 if case.get("prec") == "f32" else 8
    if case["kind"] == "run":
        n = _dims(case)
        b, fl = _step_work(n, case["pml"], len(POLES[case["poles"]]), word, 2 if case["bloch"] == "complex" else 1)
        p = _plan(case, 0)
        acc = 0.0
        for d, lo, hi in _volumes(case, p):
            pts = np.prod([max(1.0, (hi[q] - lo[q]) * RES) for q in p["dirs"]])
            acc += pts * case["nfreq"] * 16 * (4 if d is not None else len(_mapped(case)))
        return dict(bytes=b * case["steps"] + acc, flops=fl * case["steps"])
    if case["kind"] == "batch":
        b = fl = 0.0
        for q in _batch_layout(case, 0):
            x, y = _step_work((q["side"], q["side"], 0), case["pml"], 0, word)
            b, fl = b + x, fl + y
        return dict(bytes=b * case["steps"], flops=fl * case["steps"])
    if case["kind"] == "gradient":
        b, fl = _step_work((case["nx"], case["ny"], 0), case["pml"], 0, word)
        return dict(bytes=3 * b * case["steps"], flops=3 * fl * case["steps"])
    p = _far_layout(case, 0)
    side = 2.0 * case["half"]
    currents = 4 * 2 * case["dim"] * side ** (case["dim"] - 1)
    pairs = len(p["pts"]) * case["nfreq"]
    return dict(bytes=currents * (24 + 16 * case["nfreq"]) + pairs * 96, flops=pairs * currents * 30)


# ---- the same in plain torch, FP64 ----------------------------------------------------------

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_AXIS = {"x": 0, "y": 1, "z": 2}


class _Yee:
    """Yee's scheme with uPML, Lorentz and Drude poles on (n + 1) points per direction: integer
    points 0 .. n, half points 0 .. n - 1, perfect conductors outside a cell that is not
    periodic.  Every update makes new tensors, so autograd can run through it."""

    def __init__(self, n, res, pml, comps, chi=None, poles=(), sigma=None, bloch=None, k=None):
        self.n, self.res = n, res
        self.dt = COURANT / res
        self.dirs = [d for d in range(3) if n[d]]
        self.ax = {d: i for i, d in enumerate(self.dirs)}
        self.shape = [n[d] + 1 for d in self.dirs]
        self.comps = comps
        self.bloch, self.chi, self.sigma = bloch, chi, sigma
        self.dtype = torch.complex128 if bloch == "complex" else torch.float64
        self.phase = {d: complex(np.exp(2j * np.pi * k[d] * n[d] / res)) if k is not None else 1.0 for d in self.dirs}
        self.prof = {}
        for d in self.dirs:
            if pml:
                i = np.arange(2 * n[d] + 2)
                depth = np.maximum(pml * 2 - i, i - (2 * n[d] - pml * 2)).clip(0)  # half pixels into the layer
                thick = pml / res
                self.prof[d] = 0.5 * self.dt * (-math.log(1e-15)) / (4 * thick / 3.0) * (depth * 0.5 / res / thick) ** 2
        self.coef = []
        for f0, gamma, drude, _ in poles:
            w, g = 2 * math.pi * f0 * self.dt, math.pi * gamma * self.dt
            self.coef.append((1 / (1 + g), 1 - g, w * w, 0.0 if drude else w * w))
        zero = lambda: torch.zeros(self.shape, dtype=self.dtype, device=_DEV)  # noqa: E731
        self.flux_like = {c: zero() for c in comps}   # D and B
        self.f = {c: zero() for c in comps}           # E and H
        self.u = {c: zero() for c in comps}
        self.w = {c: zero() for c in comps}
        self.P = {c: [zero() for _ in poles] for c in comps if c[0] == "E"}
        self.Pp = {c: [zero() for _ in poles] for c in comps if c[0] == "E"}
        self.own = {}
        for c in comps:
            m = torch.ones(self.shape, dtype=torch.float64, device=_DEV)
            for d in self.dirs:
                edge = [0, n[d]] if not self.half(c, d) else [n[d]]
                if bloch != "none":
                    edge = [0] if not self.half(c, d) else [n[d]]
                m.index_fill_(self.ax[d], torch.tensor(edge, device=_DEV), 0.0)
            self.own[c] = m

    @staticmethod
    def half(c, d):
        """Whether component c sits on the half points along direction d."""
        own = _AXIS[c[1]]
        return (d == own) == (c[0] == "E")

    def along(self, v, d):
        shape = [1] * len(self.dirs)
        shape[self.ax[d]] = -1
        return torch.as_tensor(v, dtype=torch.float64, device=_DEV).reshape(shape)

    def sig(self, c, d):
        """uPML conductivity times dt/2 along d at the points of c, or None."""
        if d not in self.prof:
            return None
        j = np.arange(self.n[d] + 1)
        return self.along(self.prof[d][2 * j + (1 if self.half(c, d) else 0)], d)

    def halo(self, v, c):
        if self.bloch == "none":
            return v
        for d in self.dirs:
            a, n, ph = self.ax[d], self.n[d], self.phase[d]
            if self.half(c, d):
                v = torch.cat([v.narrow(a, 0, n), ph * v.narrow(a, 0, 1)], dim=a)
            else:
                back = ph.conjugate() if isinstance(ph, complex) else ph
                v = torch.cat([back * v.narrow(a, n, 1), v.narrow(a, 1, n)], dim=a)
        return v

    def diff(self, v, d, forward):
        a, n = self.ax[d], self.n[d]
        g = v.narrow(a, 1, n) - v.narrow(a, 0, n)
        z = torch.zeros_like(v.narrow(a, 0, 1))
        return torch.cat([g, z] if forward else [z, g], dim=a)

    def curl_update(self, c, src):
        kind = "E" if c[0] == "H" else "H"
        C = _AXIS[c[1]]
        d1, d2 = (C + 1) % 3, (C + 2) % 3
        name = {0: "x", 1: "y", 2: "z"}
        cu = torch.zeros(self.shape, dtype=self.dtype, device=_DEV)
        sgn = 1.0 if c[0] == "H" else -1.0
        for d, other, s in ((d1, d2, sgn), (d2, d1, -sgn)):
            g = kind + name[other]
            if d in self.ax and g in self.f:
                cu = cu + s * self.diff(self.f[g], d, c[0] == "H")
        cu = COURANT * cu
        f, s1, s2 = self.flux_like[c], self.sig(c, d1), self.sig(c, d2)
        plain = f - cu if s1 is None else ((1 - s1) * f - cu) / (1 + s1)
        if s2 is not None:
            u = self.u[c]
            un = u - cu if s1 is None else ((1 - s1) * u - cu) / (1 + s1)
            on = s2 > 0
            self.u[c] = torch.where(on, un, u)
            f = torch.where(on, ((1 - s2) * f + un - u) / (1 + s2), plain)
        else:
            f = plain
        for comp, at, amp, pulse in src:
            if comp == c:
                f = f.index_put(at, -amp * pulse, accumulate=True)
        self.flux_like[c] = self.halo(f * self.own[c], c)

    def field_update(self, c):
        g = self.flux_like[c]
        electric = c[0] == "E"
        if electric:
            for P in self.P[c]:
                g = g - P
        w = g * self.chi[c] if electric and self.chi is not None else g
        s = self.sig(c, _AXIS[c[1]])
        e = w if s is None else torch.where(s > 0, self.f[c] + (1 + s) * w - (1 - s) * self.w[c], w)
        self.w[c] = w
        if electric:
            for q, (g1i, g1, w2, w2d) in enumerate(self.coef):
                P, Pp = self.P[c][q], self.Pp[c][q]
                new = g1i * (P * (2 - w2d) - g1 * Pp + w2 * (self.sigma[q] * w))
                self.P[c][q], self.Pp[c][q] = new, P
        self.f[c] = self.halo(e * self.own[c], c)

    def points(self, c, lo, hi, centred=False):
        """Per direction the points of c's grid (or of the centred grid) around [lo, hi] and the
        integral of their linear hats over it (the hat's value where lo equals hi)."""
        idx, wts = [], []
        for d in self.dirs:
            off = 0.5 if centred or self.half(c, d) else 0.0
            a, b = lo[d] * self.res - off, hi[d] * self.res - off
            first, last = math.floor(a + 1e-9), math.ceil(b - 1e-9)
            if a == b:
                first, last = math.floor(a + 1e-9), math.ceil(a - 1e-9)
            j = np.arange(first, last + 1)
            if a == b:
                w = 1.0 - np.abs(j - a)
            else:
                t = lambda x: np.where(x < 0, 0.5 * (1 + x) ** 2, 1 - 0.5 * (1 - x) ** 2)  # noqa: E731
                w = t(np.clip(b - j, -1, 1)) - t(np.clip(a - j, -1, 1))
            if centred or self.half(c, d):
                keep = (j >= 0) & (j <= self.n[d] - 1)
            else:
                keep = (j >= 1) & (j <= self.n[d])
            idx.append(j[keep])
            wts.append(w[keep])
        return idx, wts

    def source(self, comp, lo, hi, fcen, fwidth, peak):
        idx, wts = self.points(comp, lo, hi)
        amp = np.array(1.0)
        for w in wts:
            amp = np.multiply.outer(amp, w)
        amp = amp * self.res ** sum(1 for d in self.dirs if lo[d] == hi[d])
        grid = np.meshgrid(*idx, indexing="ij")
        at = tuple(torch.as_tensor(g.ravel(), device=_DEV) for g in grid)
        return dict(comp=comp, at=at, amp=torch.as_tensor(amp.ravel(), dtype=self.dtype, device=_DEV), fcen=fcen, fwidth=fwidth, peak=peak)

    def pulse(self, s, time):
        """current times dt at time."""
        def dipole(t):
            t = t - s["peak"]
            if np.float32(abs(t)) > np.float32(5.0 / s["fwidth"]):
                return 0.0
            return np.exp(-0.5 * (t * s["fwidth"]) ** 2) * np.exp(-2j * np.pi * s["fcen"] * t) / (-2j * np.pi * s["fcen"])
        v = complex(dipole(time + self.dt) - dipole(time))
        return v if self.dtype == torch.complex128 else v.real

    def sheet(self, comp, lo, hi, freqs, centred=True):
        """A DFT monitor of comp on the centred grid, or on its own."""
        idx, wts = self.points(comp, lo, hi, centred)
        sel = [slice(int(j[0]), int(j[-1]) + 1) for j in idx]
        npts = int(np.prod([len(j) for j in idx]))
        om = torch.as_tensor(2 * np.pi * np.asarray(freqs), dtype=torch.float64, device=_DEV)
        return dict(comp=comp, idx=idx, wts=wts, sel=sel, om=om, centred=centred,
                    acc=torch.zeros((npts, len(freqs)), dtype=torch.complex128, device=_DEV))

    def accumulate(self, m, t):
        v = self.f[m["comp"]]
        for d, sl in zip(self.dirs, m["sel"]):
            a = self.ax[d]
            n = sl.stop - sl.start
            lower = v.narrow(a, sl.start, n)
            v = 0.5 * (lower + v.narrow(a, sl.start + 1, n)) if m["centred"] and not self.half(m["comp"], d) else lower
        time = t * self.dt - (0.5 * self.dt if m["comp"][0] == "H" else 0.0)
        ph = torch.polar(torch.ones_like(m["om"]), m["om"] * time) * (self.dt / math.sqrt(2 * math.pi))
        m["acc"] = m["acc"] + v.reshape(-1, 1) * ph

    def weights(self, m, lo, hi):
        w = np.array(1.0)
        for q in m["wts"]:
            w = np.multiply.outer(w, q)
        w = w / self.res ** sum(1 for d in self.dirs if lo[d] != hi[d])
        return torch.as_tensor(w.reshape(-1, 1), dtype=torch.float64, device=_DEV)

    def step_n(self, steps, sources, mons):
        mag = [c for c in self.comps if c[0] == "H"]
        ele = [c for c in self.comps if c[0] == "E"]
        for t in range(steps):
            for group, off in ((mag, 0.0), (ele, 0.5)):
                src = [(s["comp"], s["at"], s["amp"], self.pulse(s, (t + off) * self.dt)) for s in sources if s["comp"] in group]
                for c in group:
                    self.curl_update(c, src)
                for c in group:
                    self.field_update(c)
            for m in mons:
                self.accumulate(m, t + 1)


def _flux_pairs(d):
    return {0: (("Ey", "Hz"), ("Ez", "Hy")), 1: (("Ez", "Hx"), ("Ex", "Hz")), 2: (("Ex", "Hy"), ("Ey", "Hx"))}[d]


def _flux_monitors(y, d, lo, hi, freqs):
    return [(y.sheet(e, lo, hi, freqs), y.sheet(h, lo, hi, freqs), s) for (e, h), s in zip(_flux_pairs(d), (1.0, -1.0))
            if e in y.comps and h in y.comps]


def _flux_of(y, mons, lo, hi):
    out = 0.0
    for e, h, s in mons:
        out = out + s * (y.weights(e, lo, hi) * (e["acc"] * h["acc"].conj()).real).sum(dim=0)
    return out.cpu().numpy()


def _exact_run(case, seed):
    p = _plan(case, seed)
    chi = torch.as_tensor(_eps_map(p), device=_DEV)
    comps = _components(case)
    poles = POLES[case["poles"]]
    shape = [p["n"][d] + 1 for d in p["dirs"]]
    sigma = []
    for q in poles:
        v = 1.0
        for i, line in enumerate(_medium_lines(case, p, q[3])):
            v = v * torch.as_tensor(line, device=_DEV).reshape([-1 if j == i else 1 for j in range(len(shape))])
        sigma.append(v)
    y = _Yee(p["n"], RES, case["pml"], comps, {c: chi for c in comps if c[0] == "E"}, poles, sigma, case["bloch"], p["k"])
    src = y.source(p["comp"], p["where"][0], p["where"][1], p["fcen"], p["fwidth"], p["peak"])
    vols = _volumes(case, p)
    if case["out"] == "dft":
        mons = [y.sheet(c, vols[0][1], vols[0][2], p["freqs"]) for c in _mapped(case)]
        y.step_n(case["steps"], [src], mons)
        out = [m["acc"].cpu().numpy() for m in reversed(mons)]
        return out + ([y.f[comps[0]].cpu().numpy()] if case["dim"] != "3d" else [])
    flux = [_flux_monitors(y, d, lo, hi, p["freqs"]) for d, lo, hi in vols]
    y.step_n(case["steps"], [src], [m for q in flux for e, h, _ in q for m in (e, h)])
    out = [_flux_of(y, q, lo, hi) for q, (_, lo, hi) in zip(flux, vols)]
    return out + ([y.f[comps[0]].cpu().numpy()] if case["dim"] != "3d" else [])


def _exact_batch(case, seed):
    out = []
    for q in _batch_layout(case, seed):
        b = np.arange(q["side"] + 1) // 16
        comps = ("Ez", "Hx", "Hy")
        y = _Yee((q["side"], q["side"], 0), RES, case["pml"], comps,
                 {"Ez": torch.as_tensor(np.ascontiguousarray(q["inv_eps"][np.ix_(b, b)]), device=_DEV)}, bloch="none")
        at, lo, hi = _batch_line(case, q["side"])
        src = y.source("Ez", at, at, *_batch_pulse(case, q["fcen"]))
        m = _flux_monitors(y, 0, lo, hi, np.linspace(0.9 * q["fcen"], 1.1 * q["fcen"], case["nfreq"]))
        y.step_n(case["steps"], [src], [x for e, h, _ in m for x in (e, h)])
        out.append(_flux_of(y, m, lo, hi))
    return np.stack(out)


def _exact_gradient(case, seed):
    g = _grad_layout(case)
    dtype = torch.float32 if case["prec"] == "f32" else torch.float64
    design = torch.as_tensor(_grad_design(case, seed), dtype=dtype).to(torch.float64).to(_DEV).requires_grad_(True)
    nd, x0, y0 = case["design"], g["x0"], g["y0"]
    chi = torch.nn.functional.pad(design - 0.9, (y0, case["ny"] + 1 - y0 - nd, x0, case["nx"] + 1 - x0 - nd)) + 0.9
    y = _Yee((case["nx"], case["ny"], 0), GRAD_RES, case["pml"], ("Ez", "Hx", "Hy"), {"Ez": chi}, bloch="none")
    src = y.source("Ez", g["src"][0], g["src"][1], 1.0, 0.5, 2.0)
    m = y.sheet("Ez", g["mon"][0], g["mon"][1], g["freqs"])
    y.step_n(case["steps"], [src], [m])
    J = (m["acc"].real ** 2 + m["acc"].imag ** 2).sum()
    (gr,) = torch.autograd.grad(J, design)
    return dict(J=J.detach().cpu().numpy(), grad=gr.cpu().numpy())


def _bessel(x):
    """H0 and H1 of the first kind."""
    s = torch.special
    return torch.complex(s.bessel_j0(x), s.bessel_y0(x)), torch.complex(s.bessel_j1(x), s.bessel_y1(x))


def _exact_far(case, seed):
    p = _far_layout(case, seed)
    dim = case["dim"]
    n = tuple(case["cells"] if d < dim else 0 for d in range(3))
    comps = ("Ez", "Hx", "Hy") if dim == 2 else ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")
    y = _Yee(n, FAR_RES, int(FAR_RES), comps, bloch="none")
    src = y.source("Ez", p["at"], p["at"], p["fcen"], p["fcen"], 2.0)
    mons = []
    for lo, hi, sgn, nd in p["box"]:
        fd = [(nd + 1) % 3, (nd + 2) % 3]
        for j in range(2):
            # a tangential H makes an electric current along the other tangent, a tangential E a
            # magnetic one: J = n x H, M = -n x E
            for kind, s in (("E", -1.0), ("H", 1.0)):
                c = kind + "xyz"[fd[j]]
                if c in comps:
                    mons.append((y.sheet(c, lo, hi, p["freqs"], centred=False), lo, hi, sgn * s * (1.0 if j == 0 else -1.0), fd[1 - j], kind == "H"))
    y.step_n(p["steps"], [src], [m[0] for m in mons])
    X = torch.as_tensor(p["pts"], dtype=torch.float64, device=_DEV)
    nf = case["nfreq"]
    out = torch.zeros((len(p["pts"]), nf, 6), dtype=torch.complex128, device=_DEV)
    for m, lo, hi, sgn, pd, electric in mons:
        acc = m["acc"] * (sgn * y.weights(m, lo, hi))
        grid = np.meshgrid(*[(j + (0.5 if y.half(m["comp"], d) else 0.0)) / FAR_RES for d, j in zip(y.dirs, m["idx"])],
                           indexing="ij")
        at = torch.zeros((acc.shape[0], 3), dtype=torch.float64, device=_DEV)
        for d, q in zip(y.dirs, grid):
            at[:, d] = torch.as_tensor(q.ravel(), device=_DEV)
        chunk = max(1, 20_000_000 // max(1, at.shape[0]))
        for b in range(0, X.shape[0], chunk):
            r = X[b:b + chunk, None, :] - at[None, :, :]
            R = r.norm(dim=2)
            rh = r / R[..., None]
            for q, fr in enumerate(p["freqs"]):
                k = 2 * math.pi * float(fr)
                G, dG, ddG = _green(dim, k, R)
                # own kind: i w (G p + grad div (G p) / k^2); the other kind: +- grad G x p
                prh = rh[..., pd]
                a = G if dim == 2 and pd == 2 else G + dG / R / k ** 2  # nothing varies along z in 2D
                c2 = (ddG - dG / R) / k ** 2 * prh
                for d in range(3):
                    own = (1j * k) * (c2 * rh[..., d] + (a if d == pd else 0.0))
                    e1, e2 = (d + 1) % 3, (d + 2) % 3
                    if pd == e2:
                        cross = dG * rh[..., e1]
                    elif pd == e1:
                        cross = -dG * rh[..., e2]
                    else:
                        cross = None
                    out[b:b + chunk, q, d + (0 if electric else 3)] += own @ acc[:, q]
                    if cross is not None:
                        out[b:b + chunk, q, d + (3 if electric else 0)] += (cross if electric else -cross) @ acc[:, q]
    if case["one_by_one"]:
        return out.cpu().numpy()
    v = torch.view_as_real(out.permute(2, 0, 1).contiguous()).permute(0, 3, 1, 2)
    return v.contiguous().cpu().numpy()


def _green(dim, k, R):
    """The scalar Green's function of the plane or of space, and its first two derivatives."""
    if dim == 3:
        G = torch.polar(1 / (4 * math.pi * R), k * R)
        dG = G * torch.complex(-1 / R, torch.full_like(R, k))
        ddG = -k * k * G - 2 * dG / R
        return G, dG, ddG
    h0, h1 = _bessel(k * R)
    G = 0.25j * h0
    dG = -0.25j * k * h1
    return G, dG, -k * k * G - dG / R


def exact(case, seed):
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    with torch.no_grad():
        return {"run": _exact_run, "batch": _exact_batch, "far": _exact_far}[case["kind"]](case, seed)
