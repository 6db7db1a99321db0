"""Performance cases of the large step: what programs have this library do.

A case is a dict of plain values.  `kind` names the entry point:

* ``step``      - a run in progress (te_host.Run): one output interval, i.e. a
  number of large steps and then the prognostic fields read to the host;
* ``adaptive``  - the same with the clock choosing dt and nsound every step;
* ``ensemble``  - members of uneven grids stepped together, then read;
* ``gradient``  - a checkpointed window, the reverse sweep over it, and the
  gradients with respect to the window's first state;
* ``advect``    - a caller's own command tape (te_host.Replayer): the WENO
  advection tendency of one scalar, dispatch by dispatch.

Outputs are whole fields (halos included) in page-locked host buffers that the
program keeps, as one that writes history files does.  The state lives on the
GPU and goes on from pass to pass, as a run does.
"""
import ctypes
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "thunderengine-web_amd"))

import te_host  # noqa: E402

SPINUP = 20  # large steps before the first pass: winds, cloud and turbulence are under way


def listed():
    return [
        # the smallest run: a test grid, every launch far below a full chip
        dict(name="step_32x24x16_tke", kind="step", nx=32, ny=24, nz=16, tke=1, steps=10),
        # odd and ragged: no extent a multiple of anything, seven water species
        dict(name="step_37x29x17_species7", kind="step", nx=37, ny=29, nz=17, tke=1, species=7, dt=4.0, nsound=4,
             steps=10),
        # the library's default configuration (no turbulence closure)
        dict(name="step_64x64x40_default", kind="step", nx=64, ny=64, nz=40, steps=10),
        # the reference's supercell preset: open sides, TKE, heating, moving domain, dry-mass correction
        dict(name="step_120x120x40_open", kind="step", nx=120, ny=120, nz=40, tke=1, species=7, open_x=1, open_y=1,
             dissipative_heating=1, mass_conservation=1, umove=12.5, vmove=3.0, steps=10),
        # the reference's squall-line grid: open ends along x, periodic along y
        dict(name="step_300x60x40_squall", kind="step", nx=300, ny=60, nz=40, tke=1, species=7, open_x=1,
             dissipative_heating=1, steps=10),
        # the benchmark workload: one hour of a supercell is 600 such steps
        dict(name="step_192x192x80_hour", kind="step", nx=192, ny=192, nz=80, tke=1, steps=10),
        # the tornado-resolving column (tanh-stretched levels, 100 m grid, 15 substeps), the largest state
        dict(name="step_256x256x120_tornado", kind="step", nx=256, ny=256, nz=120, tke=1, stretched_z=1, dx=100.0,
             dt=0.5, nsound=8, steps=5),
        # adapt_dt = 1: the clock reads the stability maxima and re-encodes every step
        dict(name="adaptive_96x80x48", kind="adaptive", nx=96, ny=80, nz=48, tke=1, steps=10),
        # an uneven ensemble of perturbed soundings stepped together
        dict(name="ensemble_8", kind="ensemble", members=8, steps=10),
        # sensitivities: the benchmark's adjoint grid, and a small one
        dict(name="gradient_128x128x60", kind="gradient", nx=128, ny=128, nz=60, steps=10, every=5),
        dict(name="gradient_40x36x24", kind="gradient", nx=40, ny=36, nz=24, steps=10, every=5),
        # a caller's tape: positive-definite moisture advected by WENO5
        dict(name="advect_160x144x64_weno", kind="advect", nx=160, ny=144, nz=64, pdef=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def _grid(rng, most, nz_hi=128):
    """nx, ny, nz spread over the logarithm, at most `most` points."""
    while True:
        nx, ny, nz = _log_int(rng, 24, 320), _log_int(rng, 20, 320), _log_int(rng, 12, nz_hi)
        if 8000 <= nx * ny * nz <= most:
            return dict(nx=nx, ny=ny, nz=nz)


def draw(rng):
    kind = rng.choice(["step", "step", "step", "open", "adaptive", "ensemble", "gradient", "advect"])
    if kind == "step":
        c = dict(kind="step", steps=10, **_grid(rng, 3_000_000))
        c["tke"] = rng.choice([0, 1, 1])
        what = rng.choice(["", "", "dry", "species7", "weno_momentum", "explicit_vdiff"])
        if what == "dry":
            c["moist"] = 0
        elif what == "species7":
            c["species"] = 7
        elif what == "weno_momentum":
            c["weno_momentum"] = 1
        elif what == "explicit_vdiff" and c["tke"]:
            c["explicit_vdiff"] = 1
        return c
    if kind == "open":
        c = dict(kind="step", steps=10, tke=1, species=rng.choice([3, 7]), umove=12.5, vmove=3.0, **_grid(rng, 800_000, 80))
        c["open_x"], c["open_y"] = rng.choice([(1, 1), (1, 0), (0, 1)])
        c["dissipative_heating"] = rng.choice([0, 1])
        c["mass_conservation"] = rng.choice([0, 1])
        return c
    if kind == "adaptive":
        return dict(kind="adaptive", steps=10, tke=1, **_grid(rng, 1_000_000))
    if kind == "ensemble":
        while True:
            c = dict(kind="ensemble", members=rng.randint(2, 8), steps=10, layout=rng.randint(1, 1 << 20))
            if sum(m["nx"] * m["ny"] * m["nz"] for m in _member_cases(c)) <= 4_000_000:
                return c
    if kind == "gradient":
        return dict(kind="gradient", every=rng.choice([2, 5, 10]), steps=10, **_grid(rng, 600_000, 80))
    return dict(kind="advect", pdef=rng.choice([0, 1, 2]), **_grid(rng, 4_000_000))


# ------------------------------------------------------------------ inputs
def _config(case, seed):
    """te_config of a case; the seed draws the sounding's perturbation, the bubble, the shear and the noise."""
    rng = np.random.default_rng(seed)
    nz = case["nz"]
    kw = dict(nx=case["nx"], ny=case["ny"], nz=nz, dx=case.get("dx", 1000.0), dy=case.get("dx", 1000.0),
              dz=20000.0 / nz, dt=case.get("dt", 6.0), nsound=case.get("nsound", 6), rayleigh=1,
              rayleigh_zd=15000.0, seed=int(seed) + 1, sounding_seed=int(seed) + 1, th_pert_sigma=0.3,
              qv_pert_sigma=0.03, noise_sigma=0.1, bubble_amp=float(rng.uniform(1, 3)),
              shear_umax=float(rng.uniform(10, 35)))
    for k in ("moist", "species", "open_x", "open_y", "weno_momentum", "tke", "explicit_vdiff", "dissipative_heating",
              "mass_conservation", "umove", "vmove"):
        if k in case:
            kw[k] = case[k]
    if case.get("tke"):
        kw["initial_tke"] = 3
    if case.get("stretched_z"):
        kw.update(zf=te_host.tanh_faces(nz), dz=0.0, rayleigh_zd=18000.0, bubble_rh=2000.0, bubble_rv=1000.0,
                  bubble_zc=1000.0, hodo_radius=13.8, hodo_depth=1000.0)
    if case["kind"] == "adaptive":
        kw.update(adaptive_dt=1, tapfrq=60.0)
    return te_host.config(**kw)


def _prognostic(case):
    f = ["u", "v", "w", "th", "pp3d"]
    if case.get("moist", 1):
        f += ["qv", "qc"] + (["qr", "qi", "qs", "qg"] if case.get("species") == 7 else [])
    return f + (["tke"] if case.get("tke") else [])


class _Reader:
    """Page-locked host buffers for named fields of a context and their download."""

    def __init__(self, handle, offset_of, names, words, shape):
        self.h, self.words = handle, words
        self.offs = [offset_of(n) for n in names]
        self.host = {n: torch.empty(words, dtype=torch.float32, pin_memory=True) for n in names}
        self.views = {n: t.numpy().reshape(shape) for n, t in self.host.items()}
        self.ptrs = [ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_uint32)) for t in self.host.values()]

    def read(self):
        L = te_host.lib()
        for off, ptr in zip(self.offs, self.ptrs):
            if L.te_download_words(self.h, off, ptr, self.words) != te_host.TE_OK:
                raise te_host.TeError("te_download_words failed")
        return self.views


class _Stepped:
    def __init__(self, case, seed):
        self.n = case["steps"]
        self.run_ = te_host.Run(_config(case, seed))
        self.run_.init_state()
        self.adaptive = case["kind"] == "adaptive"
        if self.adaptive:
            self.run_.adaptive_start()
        self.forward(SPINUP)
        self.run_.sync()
        r = self.run_
        self.out = _Reader(r.h, r.field_offset, _prognostic(case), r.sJ * r.sK * (r.nz + 1),
                           (r.nz + 1, r.sK, r.sJ))

    def forward(self, n):
        if self.adaptive:
            self.run_.adaptive_step(n)
        else:
            self.run_.step(n)

    def go(self):
        self.forward(self.n)
        return self.out.read()


def _member_cases(case):
    """Uneven member grids of an ensemble (from the case alone)."""
    rng = np.random.default_rng(20260102 + case.get("layout", 0))
    out = []
    for _ in range(case["members"]):
        nx, ny = (int(v) for v in rng.choice([64, 96, 128, 160], 2))
        out.append(dict(kind="step", nx=nx, ny=ny, nz=int(rng.choice([40, 60, 80])), tke=1))
    return out


class _Ensemble:
    def __init__(self, case, seed):
        self.n = case["steps"]
        members = _member_cases(case)
        self.ens = te_host.Ensemble([_config(m, 1000 * seed + q) for q, m in enumerate(members)])
        self.ens.step(SPINUP)
        self.ens.sync()
        self.outs = []
        L = te_host.lib()
        for q, m in enumerate(members):
            h = L.te_ensemble_member(self.ens.h, q)
            g = (ctypes.c_int32 * 5)()
            if L.te_grid(h, g) != te_host.TE_OK:
                raise te_host.TeError("te_grid failed")
            nz, sJ, sK = g[2], g[3], g[4]

            def offset_of(name, h=h):
                o = ctypes.c_uint64()
                if L.te_field_offset(h, name.encode(), ctypes.byref(o)) != te_host.TE_OK:
                    raise te_host.TeError("te_field_offset failed")
                return o.value

            self.outs.append(_Reader(h, offset_of, ("u", "v", "w", "th", "pp3d", "qv", "tke"), sJ * sK * (nz + 1),
                                     (nz + 1, sK, sJ)))

    def go(self):
        self.ens.step(self.n)
        return [o.read() for o in self.outs]


class _Gradient:
    """J = sum of w^2 over a box of the lower half of the column; dJ/d(state at the window's start)."""
    FIELDS = ("th", "u", "v", "w", "qv", "pp3d")

    def __init__(self, case, seed):
        self.n = case["steps"]
        r = self.run_ = te_host.Run(_config(case, seed))
        r.init_state()
        r.step(SPINUP)
        r.sync()
        self.adj = te_host.Adjoint(r, every=case["every"])
        self.words = r.sJ * r.sK * (r.nz + 1)
        self.offs = {f: r.field_offset(f) for f in self.FIELDS}
        i, j = r.nx // 4, r.ny // 4
        box = te_host.Box(r, i=(i, r.nx - i), j=(j, r.ny - j), k=(1, r.nz // 2))
        self.box = box.words - self.offs["w"]
        self.seeds = np.zeros(self.words, np.float32)
        self.w = torch.empty(self.words, dtype=torch.float32, pin_memory=True)
        self.host = {f: torch.empty(self.words, dtype=torch.float32, pin_memory=True) for f in self.FIELDS}
        self.views = {f: t.numpy().reshape(r.nz + 1, r.sK, r.sJ) for f, t in self.host.items()}

    def go(self):
        L, f32, u32 = te_host.lib(), ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_uint32)
        self.adj.forward(self.n)
        if L.te_download_words(self.run_.h, self.offs["w"], ctypes.cast(self.w.data_ptr(), u32), self.words) != te_host.TE_OK:
            raise te_host.TeError("te_download_words failed")
        self.seeds[self.box] = 2.0 * self.w.numpy()[self.box]
        self.adj.zero()
        self.adj.upload(self.offs["w"], self.seeds)
        self.adj.backward()
        for f, t in self.host.items():
            if L.te_adj_download(self.adj.h, self.offs[f], ctypes.cast(t.data_ptr(), f32), self.words) != te_host.TE_OK:
                raise te_host.TeError("te_adj_download failed")
        return self.views


# The tape of one scalar's WENO advection: a memory of the caller's own layout.
H = 3  # halo cells on the low side; the high side has one more


class _Layout:
    """Word offsets of the advection tape's parameters and fields."""

    def __init__(self, case):
        self.nx, self.ny, self.nz = nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.sJ, self.sK = nx + 7, ny + 7
        self.shape = (nz + 1, self.sK, self.sJ)
        self.words = self.sJ * self.sK * (nz + 1)
        self.at, end = {}, 0
        for name, n in [("dims", 16), ("weps", 1), ("pdef", 1), ("pdefweno", 1), ("stag", 1), ("acc", 1), ("open", 2),
                        ("c1", nz + 1), ("c2", nz + 1), ("mh", nz + 1), ("mf", nz + 1), ("rho0", nz + 1),
                        ("rf0", nz + 1), ("hmetric", 2 * self.sJ + 2 * self.sK)] + \
                [(f, self.words) for f in ("s", "rru", "rrv", "rrw", "divx", "fx", "fy", "fz", "tend")]:
            self.at[name] = end
            end += (n + 63) // 64 * 64
        self.end = end


def _fields(case, seed):
    """float32 inputs: a positive scalar with a sharp-edged cloud in it, mass fluxes and their divergence."""
    lay = _Layout(case)
    nx, ny, nz = lay.nx, lay.ny, lay.nz
    g = torch.Generator().manual_seed(int(seed))
    x = torch.arange(-H, nx + 4, dtype=torch.float64)
    y = torch.arange(-H, ny + 4, dtype=torch.float64)
    z = torch.arange(0, nz + 1, dtype=torch.float64)
    wave = lambda a, n, m, p: torch.sin(2 * np.pi * (m * a / n + p))  # noqa: E731
    p = torch.rand(12, generator=g, dtype=torch.float64).tolist()
    X, Y, Z = x[None, None, :], y[None, :, None], z[:, None, None]

    def periodic(f):
        i, j = torch.remainder(x.long(), nx) + H, torch.remainder(y.long(), ny) + H
        return f[:, j][:, :, i].float().contiguous()

    noise = torch.rand((nz + 1, lay.sK, lay.sJ), generator=g, dtype=torch.float32).double()
    r2 = ((X - nx * p[0]) / (0.2 * nx)) ** 2 + ((Y - ny * p[1]) / (0.2 * ny)) ** 2 + ((Z - 0.4 * nz) / (0.25 * nz)) ** 2
    s = 0.014 * torch.exp(-Z / (0.2 * nz)) * (1 + 0.05 * wave(X, nx, 2, p[2]) * wave(Y, ny, 1, p[3]) + 0.002 * noise)
    s = torch.where(r2 < 1, s + 0.002, s) if case["pdef"] < 2 else torch.where(r2 < 1, s, torch.zeros_like(s))
    rho = torch.exp(-z / nz)
    rru = 12.0 * rho[:, None, None] * (wave(X, nx, 1, p[4]) + 0.4 * wave(Y, ny, 2, p[5]) + 0.2 * wave(Z, nz, 1, p[6]))
    rrv = 9.0 * rho[:, None, None] * (wave(X, nx, 2, p[7]) + 0.5 * wave(Y, ny, 1, p[8]) + 0.2 * wave(Z, nz, 2, p[9]))
    rrw = 4.0 * wave(X, nx, 1, p[10]) * wave(Y, ny, 1, p[11]) * torch.sin(np.pi * Z / nz)
    f = {"s": periodic(s), "rru": periodic(rru), "rrv": periodic(rrv), "rrw": periodic(rrw)}
    div = torch.zeros(lay.shape, dtype=torch.float64)
    u, v, w = (f[q].double() for q in ("rru", "rrv", "rrw"))
    rdx, rdz = 1.0 / 1000.0, nz / 20000.0
    div[:-1, :-1, :-1] = (u[:-1, :-1, 1:] - u[:-1, :-1, :-1]) * rdx + (v[:-1, 1:, :-1] - v[:-1, :-1, :-1]) * rdx + \
        (w[1:, :-1, :-1] - w[:-1, :-1, :-1]) * rdz
    f["divx"] = div.float()
    f["rho0"], f["rf0"] = (1.1 * rho).float(), (1.1 * torch.exp(-(z - 0.5) / nz)).float()
    return lay, f


# pdef: 0 a scalar of either sign (theta), 1 a positive one (vapour), 2 a positive one with sharp edges (cloud water)
_WEPS = {0: 1e-17, 1: 1e-20, 2: 1e-20}


class _Advect:
    def __init__(self, case, seed):
        lay, f = _fields(case, seed)
        nx, ny, nz, at = lay.nx, lay.ny, lay.nz, lay.at
        M = np.zeros(lay.end, np.uint32)
        F = M.view(np.float32)
        M[at["dims"]: at["dims"] + 5] = (nx, ny, nz, lay.sJ, lay.sK)
        F[at["dims"] + 5: at["dims"] + 8] = (1.0 / 1000.0, 1.0 / 1000.0, nz / 20000.0)
        F[at["weps"]] = _WEPS[case["pdef"]]
        M[at["pdef"]], M[at["pdefweno"]] = case["pdef"] > 0, case["pdef"] == 2
        M[at["stag"]] = 1
        for q, v in (("c1", 0.5), ("c2", 0.5), ("mh", 1.0), ("mf", 1.0)):
            F[at[q]: at[q] + nz + 1] = v
        F[at["hmetric"]: at["hmetric"] + 2 * lay.sJ + 2 * lay.sK] = 1.0
        for q, v in f.items():
            F[at[q]: at[q] + v.numel()] = v.reshape(-1).numpy()
        flux = {1: "s", 3: "weps", 4: "pdef"}
        tape = [("adv_flux_x_weno", (nx + 1, ny, nz), {**flux, 2: "rru", 5: "fx"}),
                ("adv_flux_y_weno", (nx, ny + 1, nz), {**flux, 2: "rrv", 5: "fy"}),
                ("adv_flux_z_weno", (nx, ny, nz + 1), {1: "s", 2: "rrw", 3: "c1", 4: "c2", 5: "weps", 6: "pdef",
                                                       7: "pdefweno", 8: "fz"}),
                ("adv_assemble", (nx, ny, nz), {1: "stag", 2: "s", 3: "fx", 4: "fy", 5: "fz", 6: "divx", 7: "rho0",
                                                8: "rf0", 9: "mh", 10: "mf", 11: "tend", 12: "acc", 13: "rru",
                                                14: "rrv", 15: "c1", 16: "c2", 17: "open"})]
        A = np.zeros((len(tape), 64), np.uint32)
        for q, (_, grid, params) in enumerate(tape):
            A[q, :3] = grid
            A[q, 4], A[q, 34] = at["dims"], at["hmetric"]
            for n, name in params.items():
                A[q, 4 + n] = at[name]
        self.names, self.args, self.memory = [t[0] for t in tape], A, M
        self.run_ = te_host.Replayer(lay.end, self.names, A)
        self.run_.upload(0, M)
        self.out = _Reader(self.run_.h, at.__getitem__, ("tend",), lay.words, lay.shape)

    def go(self):
        self.run_.encode_steps(1)
        return self.out.read()


_KINDS = {"step": _Stepped, "adaptive": _Stepped, "ensemble": _Ensemble, "gradient": _Gradient, "advect": _Advect}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, int(seed))


def run(state):
    return state.go()


# -------------------------------------------------------------------- work
def _substeps(nsound):
    return int(nsound / 3 + 0.5) + nsound // 2 + nsound


def _step_bytes(case):
    """Bytes one large step cannot do without: a three-stage step with S acoustic
    substeps is a chain of sweeps over the whole domain (each substep's pressure
    feeds its neighbours' winds in the next), and a sweep reads and writes its
    own fields once.  Per point, in words: 12 per stage for the momentum
    tendencies and mass fluxes, 3 per stage and advected scalar, 3 per stage for
    the diagnostics, 23 per substep, 8 at the end; with TKE 18 before the stages
    and 4 per stage."""
    scalars = (1 + case.get("species", 3) if case.get("moist", 1) else 1) - (1 if case.get("moist", 1) else 0)
    tke = 1 if case.get("tke") else 0
    words = 18 * tke + 3 * (12 + 3 * (scalars + tke) + 3 + 4 * tke) + 23 * _substeps(case.get("nsound", 6)) + 8
    return 4.0 * words * case["nx"] * case["ny"] * case["nz"]


def _field_bytes(case):
    return 4.0 * (case["nx"] + 7) * (case["ny"] + 7) * (case["nz"] + 1)


def work(case):
    if case["kind"] == "advect":
        pts = case["nx"] * case["ny"] * case["nz"]
        # 5 fields in, the tendency out; per face a WENO5 value (about 60 operations with its quotients)
        return {"bytes": 6.0 * _field_bytes(case), "flops": pts * (3 * 60.0 + 20.0)}
    if case["kind"] == "ensemble":
        each = [dict(m, steps=case["steps"]) for m in _member_cases(case)]
        parts = [work(m) for m in each]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    b = _step_bytes(case) * case["steps"]
    out = len(_prognostic(case)) * _field_bytes(case)
    if case["kind"] == "gradient":
        # the forward window; the reverse sweep reads the forward's values and
        # reads and writes an adjoint for each value the forward reads or writes
        b, out = 3.0 * b, len(_Gradient.FIELDS) * _field_bytes(case)
    # streaming stencils: about two operations for each byte
    return {"bytes": b + out, "flops": 2.0 * b}


# ------------------------------------------------------------------- exact
def _weno5(s1, s2, s3, s4, s5, weps):
    """WENO5 with WENO-Z type weights on Jiang-Shu indicators, in 64 bits."""
    b1 = 13 / 12 * (s1 - 2 * s2 + s3) ** 2 + 0.25 * (s1 - 4 * s2 + 3 * s3) ** 2
    b2 = 13 / 12 * (s2 - 2 * s3 + s4) ** 2 + 0.25 * (s2 - s4) ** 2
    b3 = 13 / 12 * (s3 - 2 * s4 + s5) ** 2 + 0.25 * (3 * s3 - 4 * s4 + s5) ** 2
    tau = (b1 - b3).abs()
    r = [torch.clamp(tau / (b + weps), max=1e30) for b in (b1, b2, b3)]
    m = torch.maximum(r[0], torch.maximum(r[1], r[2])).clamp(min=1.0)
    w = [c * ((q / m) ** 2 + 1 / m ** 2) for c, q in zip((0.1, 0.6, 0.3), r)]
    p = ((2 * s1 - 7 * s2 + 11 * s3) / 6, (-s2 + 5 * s3 + 2 * s4) / 6, (2 * s3 + 5 * s4 - s5) / 6)
    return (w[0] * p[0] + w[1] * p[1] + w[2] * p[2]) / (w[0] + w[1] + w[2])


def _upstream2(s1, s2, s3, weps):
    """Flux-limited second-order upstream face value."""
    d = s2 - s1
    r = (s3 - s2) / (torch.copysign(torch.full_like(d, weps), d) + d)
    phi = torch.minimum(r, torch.clamp(2 / 6 * r + 1 / 6, max=1.0)).clamp(min=0.0)
    return s2 + phi * d


def exact(case, seed):
    """The advection tape in 64 bits.  A whole step, ensemble or gradient has no
    value in 64 bits: it is defined by its binary32 operations (upwind and
    limiter branches included), bit for bit."""
    if case["kind"] != "advect":
        return None
    lay, f = _fields(case, seed)
    nx, ny, nz = lay.nx, lay.ny, lay.nz
    f = {k: v.double() for k, v in f.items()}
    a, weps = f["s"], float(np.float32(_WEPS[case["pdef"]]))

    def window(axis, n0, lo, hi):
        """a shifted by lo .. hi along an axis, over the face range (k, j, i) of that axis."""
        ext = [nz, ny, nx]
        ext[axis] = n0
        out = []
        for d in range(lo, hi + 1):
            sl = [slice(0, ext[0]), slice(H, H + ext[1]), slice(H, H + ext[2])]
            sl[axis] = slice(sl[axis].start + d, sl[axis].start + d + n0)
            out.append(a[tuple(sl)])
        return out

    def any_above(s):
        return torch.stack([q.abs() for q in s]).amax(0) > weps

    outs = {q: torch.zeros(lay.shape, dtype=torch.float64) for q in ("fx", "fy", "fz", "tend")}
    for name, axis, n0, vel in (("fx", 2, nx + 1, "rru"), ("fy", 1, ny + 1, "rrv")):
        s = window(axis, n0, -3, 2)
        sl = (slice(0, nz), slice(H, H + s[0].shape[1]), slice(H, H + s[0].shape[2]))
        u = f[vel][sl]
        up = u >= 0
        c = [torch.where(up, p, q) for p, q in zip(s[:5], s[:0:-1])]
        flux = u * _weno5(*c, weps)
        if case["pdef"]:
            flux = torch.where(any_above(c), flux, torch.zeros_like(flux))
        outs[name][sl] = flux
    jj, ii = slice(H, H + ny), slice(H, H + nx)
    w, fz = f["rrw"][:, jj, ii], outs["fz"][:, jj, ii]
    L = lambda k: a[k, jj, ii]  # noqa: E731
    for k in range(1, nz):  # face k between levels k - 1 and k
        wk = w[k]
        up = wk >= 0
        mean = 0.5 * (L(k - 1) + L(k))
        if k == 1:
            fz[k] = wk * torch.where(up, mean, _upstream2(L(2), L(1), L(0), weps))
            continue
        if k == nz - 1:
            fz[k] = wk * torch.where(wk > 0, _upstream2(L(k - 2), L(k - 1), L(k), weps), mean)
            continue
        lo = [L(max(k - 3, 0)), L(k - 2), L(k - 1), L(k), L(k + 1)]
        hi = [L(min(k + 2, nz)), L(k + 1), L(k), L(k - 1), L(k - 2)]
        c = [torch.where(up, p, q) for p, q in zip(lo, hi)]
        high = _weno5(*c, weps)
        face = high
        if k == 2:
            face = torch.where(up, _upstream2(L(0), L(1), L(2), weps), high)
        elif k == nz - 2:
            face = torch.where(up, high, _upstream2(L(k + 1), L(k), L(k - 1), weps))
        flux = wk * face
        if case["pdef"] == 2:
            ok = any_above(c)
            edge = up & (wk > 0) if k == 2 else wk < 0 if k == nz - 2 else torch.zeros_like(up)
            if k in (2, nz - 2):
                flux = torch.where(ok & ~edge, wk * high, flux)
            else:
                flux = torch.where(ok, flux, torch.zeros_like(flux))
        fz[k] = flux
    outs["fz"][:, jj, ii] = fz
    fx, fy, fzz = outs["fx"], outs["fy"], outs["fz"]
    kk = slice(0, nz)
    dx = fx[kk, jj, H + 1: H + nx + 1] - fx[kk, jj, ii]
    dy = fy[kk, H + 1: H + ny + 1, ii] - fy[kk, jj, ii]
    dz = fzz[1:, jj, ii] - fzz[kk, jj, ii]
    rdx, rdz = float(np.float32(1.0 / 1000.0)), float(np.float32(nz / 20000.0))
    rho = f["rho0"][:nz, None, None]
    outs["tend"][kk, jj, ii] = (a[kk, jj, ii] * f["divx"][kk, jj, ii] - (dx * rdx + dy * rdx + dz * rdz)) / rho
    return {"tend": outs["tend"].numpy()}
