"""The work that a user has this framework do, as cases that can be timed and checked.

Each case is one pass through the public entry points: a stretch of time steps of a forward run
(``GPUSolver``), a batch of shots (``BatchSolver``) or a whole sensitivity-kernel run
(``KernelSolver``). The kinds are those of the repository's own benchmark and workloads:

* ``forward``: one shot. Elastic, 3-SLS viscoelastic, fluid, fluid over solid, C-PML layers; regular
  boxes and warped meshes (every element irregular, what an external mesher delivers). A pass is the
  stretch between two seismogram outputs: it ends with the seismograms of the stretch on the host and
  the displacement (and potential) written out;
* ``batch``: many shots with records of different lengths on one mesh, from rest to the longest
  record, every shot's seismograms on the host;
* ``kernels``: forward run with checkpoints, adjoint run with recomputation, the kernels on the host.

``exact`` restates the same time loop in float64 with torch alone, from the arrays that the solver is
handed (mesh, mass matrices, moduli, source arrays, receivers).
"""
from __future__ import annotations

import ctypes as C
import functools

import numpy as np
import torch

from specfem3d_amd import abi
from specfem3d_amd import adjoint as A
from specfem3d_amd import pml as P
from specfem3d_amd import sources as S
from specfem3d_amd.attenuation import setup_attenuation
from specfem3d_amd.batch import BatchSolver
from specfem3d_amd.gll import get_gll
from specfem3d_amd.mesh.box import build_box, gradient_grf_model, homogeneous
from specfem3d_amd.solver import GPUSolver

H, DT, F0 = 250.0, 0.003, 3.0          # element edge (m), time step (s), Ricker frequency (Hz)
TABLE = 4000                           # steps of the source time functions of a forward run


# ------------------------------------------------------------------------------ cases
def _case(kind, nx, ny, nz, steps, **kw):
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, steps=steps, fluid=0, visco=False, warp=False, pml=0, receivers=36)
    if kind == "batch":
        c["shots"] = 8
    elif kind == "kernels":
        c["nt_dump"] = 64
    else:
        c.update(fma=True, assembly=-1)
    c.update(kw)
    return c


def listed():
    return [
        # the reference's CPU-runnable case: short steps, launches and host calls count
        dict(_case("forward", 20, 20, 20, 100, receivers=9), name="elastic_20x20x20"),
        # one shot of a survey on the 64 x 64 x 32 elastic model
        dict(_case("forward", 64, 64, 32, 160), name="elastic_64x64x32"),
        # a mesh from an external mesher: every element has its own Jacobians; odd sizes
        dict(_case("forward", 43, 37, 29, 120, warp=True), name="elastic_warped_43x37x29"),
        # the headline: fluid over a viscoelastic solid (the largest)
        dict(_case("forward", 64, 64, 32, 100, fluid=4, visco=True), name="sea_visco_64x64x32"),
        # small viscoelastic run with the Python driver's own defaults (no FMA contraction, assembly 0)
        dict(_case("forward", 21, 19, 17, 120, visco=True, fma=False, assembly=0), name="visco_default_21x19x17"),
        # a fluid alone: pressure records
        dict(_case("forward", 40, 40, 30, 150, fluid=30), name="fluid_40x40x30"),
        # C-PML layers on five sides
        dict(_case("forward", 30, 28, 18, 100, pml=3), name="cpml_30x28x18"),
        # a survey: shots of different lengths on one elastic model
        dict(_case("batch", 32, 32, 16, 200, shots=16), name="batch_elastic_32x32x16"),
        # a marine survey with attenuation
        dict(_case("batch", 18, 18, 12, 160, shots=8, fluid=2, visco=True), name="batch_sea_visco_18x18x12"),
        # sensitivity kernels, elastic and with a fluid layer
        dict(_case("kernels", 24, 24, 24, 128), name="kernels_elastic_24x24x24"),
        dict(_case("kernels", 19, 17, 16, 96, fluid=2, nt_dump=32), name="kernels_sea_19x17x16"),
    ]


def _steps_cost(c):
    """Element-steps of a pass, weighted by the bytes that a step of the case moves."""
    w = (4.0 if c["visco"] else 1.0) + (0.5 if c["warp"] else 0.0) + (1.0 if c["pml"] else 0.0)
    n = c["nx"] * c["ny"] * c["nz"] * c["steps"] * w
    return n * c.get("shots", 1) * (3.5 if c["kind"] == "kernels" else 1.0)


def draw(rng):
    """One more case of the ranges above: 6 to 64 elements a side, any of the kinds and options."""
    limit = max(_steps_cost(c) for c in listed())

    def side(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    while True:
        kind = rng.choice(("forward", "forward", "forward", "forward", "batch", "kernels"))
        top = {"forward": 64, "batch": 32, "kernels": 28}[kind]
        c = _case(kind, side(8, top), side(8, top), side(8, top // 2 + 8), rng.randrange(80, 161),
                  receivers=rng.choice((9, 16, 25, 36)))
        medium = rng.choice(("elastic", "elastic", "sea", "visco", "sea_visco", "fluid", "pml"))
        if medium in ("sea", "sea_visco"):
            c["fluid"] = max(1, c["nz"] // rng.choice((4, 6, 8)))
        c["visco"] = medium in ("visco", "sea_visco") and kind != "kernels"
        if kind == "forward":
            if medium == "fluid":
                c["fluid"] = c["nz"]
            if medium == "pml":
                c["pml"] = rng.choice((2, 3))
            c["warp"] = medium != "pml" and rng.random() < 0.4
            c["fma"] = rng.random() < 0.75
            c["assembly"] = rng.choice((-1, -1, -1, 0, 2))
        elif kind == "batch":
            c["shots"] = rng.choice((3, 8, 11, 16))
        else:
            c["nt_dump"] = rng.choice((24, 32, 64))
        if _steps_cost(c) <= limit:
            return c


# ------------------------------------------------------------------------------ what a program has in hand
@functools.lru_cache(maxsize=2)
def _model(nx, ny, nz, fluid, visco, warp, pml, receivers):
    """Mesh, attenuation and receivers of one model (the seed chooses the shots and the wavefield)."""
    lx, ly, lz = nx * H, ny * H, nz * H
    ext = (0.0, lx, 0.0, ly, -lz, 0.0)

    def bend(x, y, z):
        d = 0.25 * H * np.sin(2.0 * np.pi * x / lx) * np.sin(2.0 * np.pi * y / ly) * np.sin(np.pi * z / lz)
        return x + d, y - 0.7 * d, z + 0.8 * d

    solid = gradient_grf_model(ext, seed=11, z_top=-fluid * H, nmodes=8)
    faces = () if pml else (1, 2, 3, 4, 5)
    db = build_box(nx, ny, nz, ext, material=solid, acoustic_top_layers=fluid,
                   acoustic_material=homogeneous(1020.0, 1500.0, 0.0), stacey_faces=faces or (1, 2, 3, 4, 5),
                   warp=bend if warp else None)
    if pml:
        elems, regions = P.box_regions(db, pml)
        db.pml = P.set_damping(db, elems, regions, f0=F0)
    db.finalize(DT, stacey=not pml)
    att = setup_attenuation(db, qmu=100.0, qkappa=9000.0, f0_ref=F0) if visco else None
    n = int(round(receivers ** 0.5))
    depth = (fluid + 1) * H if 0 < fluid < nz else (0.3 * H if fluid else 0.0)
    edge = (pml + 0.5) * H
    rec = S.setup_receivers(db, [
        S.Station(f"R{i:02d}{j:02d}", "PF", float(y), float(x), 0.0, depth)
        for i, x in enumerate(np.linspace(edge, lx - edge, n)) for j, y in enumerate(np.linspace(edge, ly - edge, n))])
    return db, att, rec


def _shots(db, case, seed, count):
    """Moment tensors at random places below the fluid (in it where there is no solid) and inside the layers;
    near the receivers where the wavefield starts from rest, so that the short records have arrivals."""
    rng = np.random.default_rng([seed, 7])
    nx, ny, nz, fluid, pml = (case[k] for k in ("nx", "ny", "nz", "fluid", "pml"))
    lo, hi = (fluid + 1.0, nz - 1.0 - pml) if fluid < nz else (1.0, nz - 1.0)
    rest = case["kind"] != "forward"
    if rest:
        hi = min(hi, lo + 3.0)
    cmts = []
    for _ in range(count):
        m = rng.normal(size=6) * 1e15
        cmts.append(S.CMTSource(
            x=rng.uniform(0.3, 0.7) * nx * H, y=rng.uniform(0.3, 0.7) * ny * H,
            depth_km=rng.uniform(lo + 0.1 * (hi - lo), lo + 0.6 * (hi - lo)) * H / 1000.0, tshift=0.0,
            hdur=rng.uniform(2.0, 3.0) * F0 if rest else rng.uniform(0.8, 1.2) * F0,
            Mxx=m[0], Myy=m[1], Mzz=m[2], Mxy=m[3], Mxz=m[4], Myz=m[5]))
    s = S.setup_cmt_sources(db, cmts, DT, ricker=True)
    one = lambda v, k: v[k:k + 1]
    return [S.SourceSet(one(s.ispec, k), one(s.sourcearrays, k), s.kind, one(s.hdur, k), one(s.tshift, k), s.t0, DT,
                        one(s.located, k), acoustic=one(s.acoustic, k), kind_acoustic=s.kind_acoustic)
            for k in range(count)]


def _waves(db, seed):
    """Displacement and velocity (m, m/s) and potential and its derivative: three plane waves each."""
    rng = np.random.default_rng([seed, 3])
    n = db.nglob
    u, v = np.zeros((n, 3), np.float32), np.zeros((n, 3), np.float32)
    chi, chid = np.zeros(n, np.float32), np.zeros(n, np.float32)
    for _ in range(3):
        k = rng.normal(size=3)
        k *= 2.0 * np.pi / (rng.uniform(4.0, 8.0) * H) / np.linalg.norm(k)
        amp = rng.normal(size=3) * 1e-3
        ph = (np.float32(k[0]) * db.xstore + np.float32(k[1]) * db.ystore + np.float32(k[2]) * db.zstore)
        s, c = np.sin(ph), np.cos(ph)
        w = np.linalg.norm(k) * 2500.0
        u += s[:, None] * amp.astype(np.float32)
        v -= (c * np.float32(w))[:, None] * amp.astype(np.float32)
        chi += s * np.float32(amp[0] * 4e5)
        chid -= c * np.float32(amp[0] * 4e5 * w)
    if db.pml is not None:             # the layers are at rest: their memory variables start at zero
        inside = np.ones(n, np.float32)
        for x in (db.xstore, db.ystore, db.zstore):
            mid, width = 0.5 * (x.min() + x.max()), 0.16 * (x.max() - x.min())
            inside *= np.exp(-((x - mid) / width) ** 2)
        inside[db.ibool.reshape(db.nspec, 125)[db.pml.cpml_to_spec].ravel()] = 0.0
        u *= inside[:, None]
        v *= inside[:, None]
    el = np.zeros(n, bool)
    el[db.ibool.reshape(db.nspec, 125)[db.ispec_is_elastic].ravel()] = True
    ac = np.zeros(n, bool)
    ac[db.ibool.reshape(db.nspec, 125)[db.ispec_is_acoustic].ravel()] = True
    return u * el[:, None], v * el[:, None], chi * ac, chid * ac


def _lengths(case):
    """Record lengths of a batch: the first shot has the longest, the others down to half of it."""
    rng = np.random.default_rng([case["steps"], case["shots"]])
    return [case["steps"]] + [int(rng.integers(case["steps"] // 2, case["steps"] + 1)) for _ in range(case["shots"] - 1)]


def _in_hand(case, seed):
    db, att, rec = _model(*(case[k] for k in ("nx", "ny", "nz", "fluid", "visco", "warp", "pml", "receivers")))
    return db, att, rec, _shots(db, case, seed, case.get("shots", 1))


def prepare(case, seed):
    db, att, rec, shots = _in_hand(case, seed)
    if case["kind"] == "batch":
        b = BatchSolver(db, [(s, rec, n) for s, n in zip(shots, _lengths(case))], exact=False, attenuation=att)
        b.autotune(3)
        return dict(kind="batch", solver=b, shots=len(shots))
    if case["kind"] == "kernels":
        k = A.KernelSolver(db, shots[0], rec, case["steps"], nt_dump=case["nt_dump"], exact=False, assembly=2)
        return dict(kind="kernels", solver=k, observed=_observed(case, rec))
    g = GPUSolver(db, shots[0], rec, nstep=TABLE, nlength=case["steps"], attenuation=att, exact=not case["fma"],
                  assembly=case["assembly"], save_seismograms=("p",) if db.nspec_elastic == 0 else ("d",))
    u, v, chi, chid = _waves(db, seed)
    args = abi.Args()
    if db.nspec_elastic:
        zero = np.zeros_like(u)
        g.L.transfer_fields_el_to_device_(args.i(u.size), args.fa(u.ravel()), args.fa(v.ravel()),
                                          args.fa(zero.ravel()), g.MP)
    if db.nspec_acoustic:
        zero = np.zeros_like(chi)
        g.L.transfer_fields_ac_to_device_(args.i(chi.size), args.fa(chi), args.fa(chid), args.fa(zero), g.MP)
    return dict(kind="forward", solver=g, steps=case["steps"], displ=np.zeros(3 * db.nglob, np.float32),
                potential=np.zeros(db.nglob, np.float32))


def _observed(case, rec):
    """Records to fit: weak arrivals that the synthetics do not have."""
    t = np.arange(case["steps"])[:, None, None] / case["steps"]
    r = np.arange(rec.n)[None, :, None]
    c = np.arange(3)[None, None, :]
    return (1e-6 * np.sin(2 * np.pi * (3 * t + 0.13 * r + 0.3 * c)) * np.sin(np.pi * t)).astype(np.float32)


# ------------------------------------------------------------------------------ one pass
def run(state):
    s = state["solver"]
    if state["kind"] == "batch":
        s.reset()
        s.run()
        return [s.seismograms(k) for k in range(state["shots"])]
    if state["kind"] == "kernels":
        syn = s.forward()
        rho, mu, kappa = s.adjoint(A.waveform_adjoint_source(syn, state["observed"]))
        out = {"seismograms": syn, "rho": rho, "mu": mu, "kappa": kappa}
        if s.acoustic:
            out["rho_fluid"], out["kappa_fluid"] = s.acoustic_kernels
        return out
    if s.it + state["steps"] > s.nstep:
        s.it = 0                       # the source time function starts over
    s.seismo_current = 0               # a new stretch of records
    for _ in range(state["steps"]):
        s.step()
    n = C.c_int(state["displ"].size)
    out = {"seismograms": s.seismograms("d" if s.elastic else "p")}
    if s.elastic:
        s.L.transfer_displ_from_device_(C.byref(n), state["displ"].ctypes.data_as(C.c_void_p), s.MP)
        out["displacement"] = state["displ"]
    if s.acoustic:
        n = C.c_int(state["potential"].size)
        s.L.transfer_potential_ac_from_device_(C.byref(n), state["potential"].ctypes.data_as(C.c_void_p), s.MP)
        out["potential"] = state["potential"]
    return out


def work(case):
    """Bytes and operations of a pass: every step reads and writes the wavefield once (u and v, or chi and
    chi'), reads the inverse mass, and per local point the index, the moduli, an irregular element's ten
    Jacobian terms and the memory variables and strain (also written)."""
    nx, ny, nz, fl = case["nx"], case["ny"], case["nz"], case["fluid"]
    plane, local = (4 * nx + 1) * (4 * ny + 1), 125 * nx * ny
    steps, shots = case["steps"], 1
    if case["kind"] == "batch":
        steps, shots = 0.75 * steps, case["shots"]
    el_g, el_l = (plane * (4 * (nz - fl) + 1), local * (nz - fl)) if nz > fl else (0, 0)
    ac_g, ac_l = (plane * (4 * fl + 1), local * fl) if fl else (0, 0)
    shared = 12.0 * el_g + 4.0 * ac_g + 12.0 * el_l + 8.0 * ac_l + (40.0 * (el_l + ac_l) if case["warp"] else 0.0)
    per_shot = 48.0 * el_g + 16.0 * ac_g + (192.0 * el_l if case["visco"] else 0.0)
    if case["pml"]:
        m = case["pml"]
        inner = max(0, nx - 2 * m) * max(0, ny - 2 * m) * max(0, nz - m)
        per_shot += 125.0 * (nx * ny * nz - inner) * 20 * 8
    flops = (270.0 + (210.0 if case["visco"] else 0.0)) * el_l + 110.0 * ac_l + 21.0 * el_g + 7.0 * ac_g
    if case["kind"] == "kernels":      # forward, recomputed forward and adjoint steps; strains and kernels of each step
        shared *= 3.0
        per_shot = 3.0 * per_shot + (24.0 + 24.0) * el_l + (16.0 + 16.0) * ac_l + 24.0 * el_g + 16.0 * ac_g
        flops *= 3.7
    return {"bytes": steps * (shared + shots * per_shot), "flops": steps * shots * flops}


# ------------------------------------------------------------------------------ the same in 64 bits
class _Loop64:
    """The time loop of one wavefield in float64, from the arrays that the solver is handed."""

    def __init__(self, db, att, source, receivers, nstep, sign=1.0):
        d = self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.f = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=d).double()
        self.i = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=d).long()
        f, i = self.f, self.i
        self.db, self.att, self.sign = db, att, sign
        self.dt = float(np.float32(db.dt))
        self.dt2 = float(np.float32(np.float32(db.dt) / np.float32(2)))
        self.dtsq2 = float(np.float32(np.float32(db.dt) * np.float32(db.dt) / np.float32(2)))
        g = get_gll()
        self.hp, self.hpw, self.w2 = f(g.hprime), f(g.hprimewgll), f(g.wgllwgll_xy)
        self.ib = i(db.ibool.reshape(db.nspec, 125))
        pml = db.pml.is_cpml(db.nspec) if db.pml is not None else np.zeros(db.nspec, bool)
        self.el, self.ac = i(np.nonzero(db.ispec_is_elastic & ~pml)[0]), i(np.nonzero(db.ispec_is_acoustic)[0])
        self.nel, self.nac = db.nspec_elastic, db.nspec_acoustic
        self.kap = f(db.kappastore if att is None else att.kappastore).view(db.nspec, 125)
        self.mu = f(db.mustore if att is None else att.mustore).view(db.nspec, 125)
        self.rho = f(db.rhostore).view(db.nspec, 125)
        self.rm = torch.stack([f(db.rmassx), f(db.rmassy), f(db.rmassz)], 1)
        self.rma = f(db.rmass_acoustic)
        z = lambda *s: torch.zeros(*s, dtype=torch.float64, device=d)
        self.z = z
        if self.nel:
            self.u, self.v, self.a = z(db.nglob, 3), z(db.nglob, 3), z(db.nglob, 3)
        if self.nac:
            self.c, self.cd, self.cdd = z(db.nglob), z(db.nglob), z(db.nglob)
        if att is not None:
            n = len(self.el)
            self.R, self.old = z(n, 125, 6, 3), z(n, 125, 6)
            self.fc, self.fck = f(att.factor_common)[self.el], f(att.factor_common_kappa)[self.el]
            self.abg = [f(x) for x in (att.alphaval, att.betaval, att.gammaval)]
        self._faces()
        if pml.any():
            self._pml_arrays()
        self.stf = None
        if source is not None and source.n:
            self.src = self.ib[int(source.ispec[0])]
            self.src_ac = bool(db.ispec_is_acoustic[source.ispec[0]])
            self.src_kap = self.kap[int(source.ispec[0])]
            self.src_arr = f(source.sourcearrays[0]).view(125, 3)
            self.stf = f(source.stf_table(nstep)[:, 0].astype(np.float32)).tolist()
        h = [np.asarray(x, np.float64) for x in (receivers.hxir, receivers.hetar, receivers.hgammar)]
        self.rec_h = f((h[2][:, :, None, None] * h[1][:, None, :, None] * h[0][:, None, None, :]).reshape(-1, 125))
        self.rec = self.ib[i(receivers.ispec)]
        self.nu = f(receivers.nu)
        self.it = 0

    def _faces(self):
        db, f, i = self.db, self.f, self.i

        def points(fc, keep):
            loc = i(fc.ijk[keep][..., 0] + 5 * fc.ijk[keep][..., 1] + 25 * fc.ijk[keep][..., 2])
            e = i(fc.ispec[keep])[:, None].expand(loc.shape)
            return self.ib[e, loc].reshape(-1), e, loc, f(fc.normal[keep]).reshape(-1, 3), f(fc.jacobian2Dw[keep]).reshape(-1)

        ab = db.abs_faces
        on = np.full(ab.n, bool(db.stacey))
        g, e, loc, n, w = points(ab, on & db.ispec_is_elastic[ab.ispec])
        self.st_el = (g, n, w, f(db.rho_vp)[e, loc].reshape(-1), f(db.rho_vs)[e, loc].reshape(-1))
        g, e, loc, n, w = points(ab, on & db.ispec_is_acoustic[ab.ispec])
        rho, kap = self.rho[e, loc].reshape(-1), f(db.kappastore).view(-1, 125)[e, loc].reshape(-1)
        self.st_ac = (g, w / torch.sqrt(kap / rho) / rho)
        fr = db.free_faces
        self.free = points(fr, db.ispec_is_acoustic[fr.ispec])[0]
        g, _, _, n, w = points(db.coupling_faces, np.ones(db.coupling_faces.n, bool))
        self.couple = (g, n, w)
        self.edge = points(ab, np.ones(ab.n, bool))[0] if db.pml is not None else None

    def _geometry(self, e):
        """d(xi_a)/d(x_b) as (E, 125, 3, 3), or one factor where every element is a cube; the Jacobian."""
        db = self.db
        if not db.nspec_irregular:
            return float(db.xix_regular), float(db.jacobian_regular)
        irr = self.i(db.irregular_element_number)[e]
        m = torch.eye(3, dtype=torch.float64, device=self.dev) * float(db.xix_regular)
        m = m.expand(len(e), 125, 3, 3).clone()
        j = torch.full((len(e), 125), float(db.jacobian_regular), dtype=torch.float64, device=self.dev)
        at = irr > 0
        m[at] = self.f(db.jac9)[irr[at] - 1].transpose(1, 2).reshape(-1, 125, 3, 3)
        j[at] = self.f(db.jacobian)[irr[at] - 1]
        return m, j

    def _grad(self, x, geo):
        """(E, 125, C) -> (E, 125, C, 3): the derivatives in x, y, z."""
        e, n = x.shape[0], x.shape[-1]
        t = x.view(e, 5, 5, 5, n)
        g = torch.stack([torch.einsum("il,ekjlc->ekjic", self.hp, t), torch.einsum("jl,eklic->ekjic", self.hp, t),
                         torch.einsum("kl,eljic->ekjic", self.hp, t)], -1).view(e, 125, n, 3)
        return g * geo if isinstance(geo, float) else torch.einsum("epca,epab->epcb", g, geo)

    def _div(self, s, geo, jac):
        """Weak divergence of s (E, 125, C, 3) -> (E, 125, C)."""
        e, n = s.shape[0], s.shape[2]
        t = s * (geo * jac) if isinstance(geo, float) else torch.einsum("epcb,epab->epca", s, geo) * jac[..., None, None]
        t = t.reshape(e, 5, 5, 5, n, 3)
        w = self.w2
        f = torch.einsum("li,ekjlc->ekjic", self.hpw, t[..., 0]) * w.t()[None, :, :, None, None]
        f += torch.einsum("lj,eklic->ekjic", self.hpw, t[..., 1]) * w.t()[None, :, None, :, None]
        f += torch.einsum("lk,eljic->ekjic", self.hpw, t[..., 2]) * w.t()[None, None, :, :, None]
        return f.reshape(e, 125, n)

    @staticmethod
    def _stress(du, kap, mu):
        tr = du.diagonal(dim1=2, dim2=3).sum(-1)
        s = (du + du.transpose(2, 3)) * mu[..., None, None]
        lam = kap - 2.0 / 3.0 * mu
        for c in range(3):
            s[..., c, c] += lam * tr
        return s

    @staticmethod
    def _strain(du):
        """xx, yy, xy, xz, yz of the deviator and the trace."""
        tr = du.diagonal(dim1=2, dim2=3).sum(-1)
        sym = lambda a, b: 0.5 * (du[..., a, b] + du[..., b, a])
        return torch.stack([du[..., 0, 0] - tr / 3.0, du[..., 1, 1] - tr / 3.0, sym(0, 1), sym(0, 2), sym(1, 2), tr], -1)

    def _solid(self):
        e, ib = self.el, self.ib[self.el]
        geo, jac = self._geometry(e)
        kap, mu = self.kap[e], self.mu[e]
        du = self._grad(self.u[ib], geo)
        s = self._stress(du, kap, mu)
        if self.att is not None:
            r = self.R.sum(-1)
            xx, yy, xy, xz, yz, tr = r.unbind(-1)
            s[..., 0, 0] -= xx + tr
            s[..., 1, 1] -= yy + tr
            s[..., 2, 2] += xx + yy - tr
            for a, b, q in ((0, 1, xy), (0, 2, xz), (1, 2, yz)):
                s[..., a, b] -= q
                s[..., b, a] -= q
            new = self._strain(self._grad((self.u + self.dt * self.v)[ib], geo))
            al, be, ga = self.abg
            fac = (mu[..., None] * self.fc)[:, :, None, :].repeat(1, 1, 6, 1)
            fac[:, :, 5] = kap[..., None] * self.fck
            self.R = al * self.R + fac * (be * self.old[..., None] + ga * new[..., None])
            self.old = new
        self.a.index_add_(0, ib.reshape(-1), -self._div(s, geo, jac).reshape(-1, 3))

    def _fluid(self):
        e, ib = self.ac, self.ib[self.ac]
        geo, jac = self._geometry(e)
        s = self._grad(self.c[ib][..., None], geo) / self.rho[e][..., None, None]
        self.cdd.index_add_(0, ib.reshape(-1), -self._div(s, geo, jac).reshape(-1))

    # C-PML: recursive convolutions r <- c0 r + new c1 + old c2 and the modified strains
    def _pml_arrays(self):
        p, f = self.db.pml, self.f
        self.pe = self.i(p.cpml_to_spec)
        self.p_al, self.p_be = f(p.coef_alpha).view(-1, 125, 3, 3), f(p.coef_beta).view(-1, 125, 3, 3)
        self.p_ab, self.p_st = f(p.coef_abar), f(p.coef_strain)
        n = p.n
        self.r3, self.r1, self.rd = self.z(n, 125, 3, 3, 3), self.z(n, 125, 3, 3, 3), self.z(n, 125, 3, 3)
        w = np.asarray(get_gll().wgll, np.float64)
        self.wc = f((w[:, None, None] * w[None, :, None] * w[None, None, :]).ravel().astype(np.float32))
        self.p_old = None

    def _layers(self):
        e, ib = self.pe, self.ib[self.pe]
        geo, jac = self._geometry(e)
        th1, th2 = self.dt2 * 0.75, self.dtsq2 * 0.875
        new_u, old_u = self.u + th1 * self.v, self.p_old
        cur, new, old = (self._grad(x[ib], geo) for x in (self.u, new_u, old_u))
        al, be, st = self.p_al, self.p_be, self.p_st
        sets = ((al[:, :, 2], al[:, :, 1], be[:, :, 0]), (al[:, :, 0], al[:, :, 2], be[:, :, 1]),
                (al[:, :, 0], al[:, :, 1], be[:, :, 2]))
        conv = lambda r, k, nw, od: k[..., 0, None] * r + nw * k[..., 1, None] + od * k[..., 2, None]
        full = torch.empty_like(cur)   # d(u_c)/d(x_b), damped for the products with component c
        for b in range(3):
            for s in range(3):
                self.r3[:, :, b, s] = conv(self.r3[:, :, b, s], sets[b][s], new[..., b], old[..., b])
            q = st[:, :, 4 * b:4 * b + 4]
            full[..., b] = q[..., 0, None] * cur[..., b] + (q[..., 1:, None] * self.r3[:, :, b]).sum(2)
        part = []                      # the derivatives damped along one axis alone
        for x in range(3):
            k = al[:, :, x][..., None, :]
            self.r1[:, :, x] = k[..., 0, None] * self.r1[:, :, x] + new * k[..., 1, None] + old * k[..., 2, None]
            q = st[:, :, 12 + 2 * x:14 + 2 * x]
            part.append(q[..., 0, None, None] * cur + q[..., 1, None, None] * self.r1[:, :, x])
        mu, kap = self.mu[e], self.kap[e]
        l2m = kap + 4.0 / 3.0 * mu
        lam = l2m - 2.0 * mu
        # the axis that damps a derivative of component c in the stress that column b multiplies
        axis = {(0, 1): 2, (0, 2): 1, (1, 0): 2, (1, 2): 0, (2, 0): 1, (2, 1): 0}
        s = torch.empty_like(cur)      # s[c][b]: stress on component c for the derivative along b
        for b in range(3):
            diag = [full[..., b, b] if c == b else part[axis[(b, c)]][..., c, c] for c in range(3)]
            s[..., b, b] = sum((l2m if c == b else lam) * diag[c] for c in range(3))
            for c in range(3):
                if c != b:
                    s[..., c, b] = mu * (full[..., c, b] + part[axis[(b, c)]][..., b, c])
        f = self._div(s, geo, jac)
        for x in range(3):
            k = al[:, :, x]
            self.rd[:, :, x] = k[..., 0, None] * self.rd[:, :, x] + new_u[ib] * k[..., 1, None] + old_u[ib] * k[..., 2, None]
        ab = self.p_ab
        w = self.wc * self.rho[e] * jac
        f = f + w[..., None] * (ab[..., 0, None] * self.v[ib] + ab[..., 1, None] * self.u[ib]
                                + (ab[..., 2:, None] * self.rd).sum(2))
        self.a.index_add_(0, ib.reshape(-1), -f.reshape(-1, 3))

    def step(self, source=True, adjoint=None):
        """One Newmark step; ``adjoint``: forces (nrec, 3) at the receivers."""
        dt, dt2, dtsq2 = self.dt, self.dt2, self.dtsq2
        q = self.stf[self.it] if source and self.stf is not None else None
        self.it += 1
        if self.nel and self.db.pml is not None:
            self.p_old = self.u + self.dt2 * 0.75 * self.v + self.dtsq2 * 0.875 * self.a
        if self.nac:
            self.c += dt * self.cd + dtsq2 * self.cdd
            self.cd += dt2 * self.cdd
            self.cdd.zero_()
        if self.nel:
            self.u += dt * self.v + dtsq2 * self.a
            self.v += dt2 * self.a
            self.a.zero_()
        if self.nac:
            self._open()
            g, w = self.st_ac
            self.cdd.index_add_(0, g, -self.cd[g] * w)
            g, n, w = self.couple
            if self.nel and len(g):
                self.cdd.index_add_(0, g, self.sign * w * (self.u[g] * n).sum(1))
            if q is not None and self.src_ac:
                self.cdd.index_add_(0, self.src, -self.src_arr[:, 0] * q / self.src_kap)
            self._fluid()
            self.cdd *= self.rma
            self.cd += dt2 * self.cdd
            self._open()
        if self.nel:
            g, n, w, rp, rs = self.st_el
            vn = (self.v[g] * n).sum(1, keepdim=True)
            self.a.index_add_(0, g, -(rp[:, None] * vn * n + rs[:, None] * (self.v[g] - vn * n)) * w[:, None])
            g, n, w = self.couple
            if self.nac and len(g):
                self.a.index_add_(0, g, -self.sign * (w * self.cdd[g])[:, None] * n)
            if q is not None and not self.src_ac:
                self.a.index_add_(0, self.src, self.src_arr * q)
            if adjoint is not None:
                self.a.index_add_(0, self.rec.reshape(-1), (self.rec_h[..., None] * adjoint[:, None]).reshape(-1, 3))
            self._solid()
            if self.edge is not None:
                self._layers()
                for x in (self.u, self.v, self.a):
                    x[self.edge] = 0.0
            self.a *= self.rm
            self.v += dt2 * self.a

    def _open(self):
        for x in (self.c, self.cd, self.cdd):
            x[self.free] = 0.0

    def record(self):
        if self.nel:
            return torch.einsum("rab,rb->ra", self.nu, (self.rec_h[..., None] * self.u[self.rec]).sum(1))
        p = -(self.rec_h * self.cdd[self.rec]).sum(1)
        return torch.stack([p, p * 0, p * 0], 1)


def exact(case, seed):
    db, att, rec, shots = _in_hand(case, seed)
    if case["kind"] == "batch":
        out = []
        for s, n in zip(shots, _lengths(case)):
            loop, seis = _Loop64(db, att, s, rec, n), []
            for _ in range(n):
                loop.step()
                seis.append(loop.record())
            out.append(torch.stack(seis).cpu().numpy())
        return out
    if case["kind"] == "kernels":
        return _kernels64(db, shots[0], rec, case)
    loop, seis = _Loop64(db, att, shots[0], rec, TABLE), []
    u, v, chi, chid = _waves(db, seed)
    if loop.nel:
        loop.u, loop.v = loop.f(u), loop.f(v)
    if loop.nac:
        loop.c, loop.cd = loop.f(chi), loop.f(chid)
    for _ in range(case["steps"]):
        loop.step()
        seis.append(loop.record())
    out = {"seismograms": torch.stack(seis).cpu().numpy()}
    if loop.nel:
        out["displacement"] = loop.u.reshape(-1).cpu().numpy()
    if loop.nac:
        out["potential"] = loop.c.cpu().numpy()
    return out


def _kernels64(db, source, rec, case):
    n = case["steps"]
    loop, seis, frames = _Loop64(db, None, source, rec, n), [], []
    for _ in range(n):
        loop.step()
        seis.append(loop.record())
        frames.append((loop.u.clone(),) + ((loop.c.clone(), loop.cdd.clone()) if loop.nac else ()))
    syn = torch.stack(seis)
    adj = syn - loop.f(_observed(case, rec))
    back = _Loop64(db, None, None, rec, n, sign=-1.0)
    shape = (db.nspec, 125)
    kl = {k: back.z(*shape) for k in ("rho", "mu", "kappa") + (("rho_fluid", "kappa_fluid") if loop.nac else ())}
    ib, ia = back.ib[back.el], back.ib[back.ac]
    geo, _ = back._geometry(back.el)
    geo_a, _ = back._geometry(back.ac)
    for it in range(1, n + 1):
        back.step(source=False, adjoint=adj[n - it] if it < n else None)
        b = frames[n - it]
        kl["rho"][back.el] += back.dt * (back.a[ib] * b[0][ib]).sum(-1)
        s, t = back._strain(back._grad(back.u[ib], geo)), back._strain(back._grad(b[0][ib], geo))
        kl["kappa"][back.el] += back.dt * s[..., 5] * t[..., 5]
        kl["mu"][back.el] += back.dt * (s[..., 0] * t[..., 0] + s[..., 1] * t[..., 1]
                                        + (s[..., 0] + s[..., 1]) * (t[..., 0] + t[..., 1])
                                        + 2.0 * (s[..., 2:5] * t[..., 2:5]).sum(-1))
        if loop.nac:
            ga, gb = (back._grad(x[ia][..., None], geo_a) for x in (back.c, b[1]))
            kl["rho_fluid"][back.ac] += back.dt * (ga * gb).sum((-1, -2))
            kl["kappa_fluid"][back.ac] += back.dt * back.c[ia] * b[2][ia]
    out = {"seismograms": syn.cpu().numpy()}
    out.update({k: x.view(db.nspec, 5, 5, 5).cpu().numpy() for k, x in kl.items()})
    return out
