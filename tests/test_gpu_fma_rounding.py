"""FMA builds round every operation where they always did.

Records and kernels of a weak first arrival are mostly what the rounding of each step leaves behind the
front, so a sum taken in another order, or with other bits, shows there first: 1e-5 to 1e-3 of the output
where strong arrivals move by 1e-7. ``golden/fma_rounding.npz`` holds such outputs as the library gave them
when its element launches scattered colour by colour (written by golden/make_fma_rounding_fixture.py);
sums in the colour order reproduce them. Tolerance 2e-5 of the 2-norm, what a program may see between two
builds in single precision; equal roundings give equal bits.

The other tests follow from the same rounding: a field that is read between steps, the interval of the
checkpoints and the number of shot groups held at a time change no bit."""
import os

import numpy as np
import pytest

from conftest import rel_l2, smooth_warp

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "fma_rounding.npz")
DT = 0.008
# (elements a side, fluid layers, warped: 0 no, 1 every element, 2 the upper half, viscoelastic, steps)
FORWARD = {"elastic": (5, 0, False, False, 45), "elastic_warped": (6, 0, True, False, 45), "sea": (5, 1, False, False, 45),
           "sea_visco": (5, 1, True, True, 45), "fluid": (4, 4, False, False, 40), "fluid_warped": (4, 4, True, False, 40),
           "elastic_mixed": (6, 0, 2, False, 45), "sea_visco_mixed": (6, 1, 2, True, 45)}
KERNELS = {"kernels": (5, 0, False, 48), "kernels_warped": (6, 0, True, 48), "kernels_sea": (6, 2, False, 48),
           "kernels_mixed": (6, 0, 2, 48)}
BATCH = {"batch_2": (2, False, 0), "batch_3": (3, False, 0), "batch_visco": (2, True, 0), "batch_mixed": (2, False, 2), "batch_sea": (2, False, 1)}
CASES = [*FORWARD, *KERNELS, *BATCH]


def upper_half(L):
    """Elements below the middle stay cubes."""
    def w(x, y, z):
        d = 0.05 * L * np.sin(np.pi * x / L) * np.sin(np.pi * y / L) * np.sin(2 * np.pi * np.maximum(0.0, 0.5 + z / L))
        return x + 0.5 * d, y - 0.3 * d, z + 0.4 * d
    return w


def corner_to_corner(n, fluid, warped, hdurs=(4.0,)):
    """A gradient box with shots in one bottom corner (of the fluid, if that is all) and receivers in the opposite
    ones: the steps end when the first arrival has come through."""
    from specfem3d_amd import sources as S
    from specfem3d_amd.mesh.box import build_box, gradient_grf_model, homogeneous
    L = 500.0 * n
    ext = (0.0, L, 0.0, L, -L, 0.0)
    db = build_box(n, n, n, ext, material=gradient_grf_model(ext, seed=0, corr_len=700.0), acoustic_top_layers=fluid,
                   acoustic_material=homogeneous(1020.0, 1500.0, 0.0), warp=[None, smooth_warp(L), upper_half(L)][warped],
                   stacey_faces=(1, 2, 3, 4, 5))
    db.finalize(DT, stacey=True)
    assert warped != 2 or 0 < db.nspec_irregular < db.nspec
    shots = [S.setup_cmt_sources(db, [S.CMTSource(300.0 + 50.0 * k, 400.0, 0.9 * L / 1000.0, 0.0, h, 1e13, -2e13, 0.7e13,
                                                  0.3e13, -0.5e13, 0.2e13)], DT, ricker=True) for k, h in enumerate(hdurs)]
    rec = S.setup_receivers(db, [S.Station(f"R{i}", "T", 0.9 * L, (0.1 + 0.4 * i) * L, 0.0, 0.6 * L) for i in range(3)])
    return db, shots, rec


def attenuation(db):
    from specfem3d_amd.attenuation import setup_attenuation
    return setup_attenuation(db, qmu=60.0, qkappa=200.0, f0_ref=4.0)


def adjoint_source(nstep, nrec):
    t, r, c = np.arange(nstep)[:, None, None] / nstep, np.arange(nrec)[None, :, None], np.arange(3)[None, None, :]
    return (np.sin(2 * np.pi * (2 * t + 0.17 * r + 0.3 * c)) * np.sin(np.pi * t)).astype(np.float32)


def kernel_solver(case, nt_dump=16):
    from specfem3d_amd.adjoint import KernelSolver
    n, fluid, warped, nstep = KERNELS[case]
    db, (src,), rec = corner_to_corner(n, fluid, warped)
    return KernelSolver(db, src, rec, nstep, nt_dump=nt_dump, exact=False, assembly=2)


def batch_solver(case):
    from specfem3d_amd.batch import BatchSolver
    assembly, visco, warped = BATCH[case]
    db, shots, rec = corner_to_corner(8, 2 if case == "batch_sea" else 1 if visco else 0, warped, (4.0, 5.0, 6.0))
    return BatchSolver(db, [(s, rec, n) for s, n in zip(shots, (48, 45, 36))], exact=False, shots_per_group=8,
                       assembly=assembly, attenuation=attenuation(db) if visco else None)


def outputs(case):
    """Arrays of one case by name."""
    from specfem3d_amd.solver import GPUSolver
    if case in KERNELS:
        ks = kernel_solver(case)
        out = {"seis": ks.forward()}
        out.update(zip(("rho", "mu", "kappa"), ks.adjoint(adjoint_source(ks.nstep, ks.receivers.n))))
        if ks.acoustic:
            ac = np.asarray(ks.db.ispec_is_acoustic, bool)
            out = {"seis": out["seis"], "rho_fluid": ks.acoustic_kernels[0][ac], "kappa_fluid": ks.acoustic_kernels[1][ac]}
        ks.close()
        return out
    if case in BATCH:
        b = batch_solver(case)
        b.run()
        out = {f"shot{k}": b.seismograms(k) for k in range(3)}
        b.close()
        return out
    n, fluid, warped, visco, nstep = FORWARD[case]
    db, (src,), rec = corner_to_corner(n, fluid, warped)
    kind = "p" if fluid == n else "d"
    g = GPUSolver(db, src, rec, nstep=nstep, exact=False, assembly=2, attenuation=attenuation(db) if visco else None,
                  save_seismograms=(kind,))
    g.run()
    out = {"seis": g.seismograms(kind).copy()}
    g.close()
    return out


@pytest.mark.parametrize("case", CASES)
def test_outputs_of_weak_arrivals(case):
    print(f"[gpu] FMA rounding {case}", flush=True)
    with np.load(GOLDEN) as f:
        for name, x in outputs(case).items():
            ref = f[f"{case}/{name}"]
            assert np.abs(ref).max() > 0
            e = rel_l2(x, ref)
            print(f"[gpu]   {name} {e:.2e}", flush=True)
            assert e < 2e-5, (name, e)


@pytest.mark.parametrize("assembly", [-1, 0, 2])
@pytest.mark.parametrize("case", ["elastic", "sea_visco", "fluid"])
def test_fields_read_between_steps(case, assembly):
    """A transfer to the host ends the fusion of sum, corrector and predictor for a step and changes no bit."""
    from specfem3d_amd.solver import GPUSolver
    n, fluid, warped, visco, _ = FORWARD[case]
    db, (src,), rec = corner_to_corner(n, fluid, warped)
    print(f"[gpu] fields read between steps {case} assembly={assembly}", flush=True)
    out = []
    for read in (False, True):
        g = GPUSolver(db, src, rec, nstep=24, exact=False, assembly=assembly, attenuation=attenuation(db) if visco else None,
                      save_seismograms=("p",) if fluid == n else ("d",))
        for k in range(24):
            g.step()
            if read and k % 3 != 1:
                if g.elastic:
                    g.fields()
                if g.acoustic:
                    g.potentials()
        out.append([g.seis_d.copy(), g.seis_p.copy(), *(g.fields() if g.elastic else ()),
                    *(g.potentials() if g.acoustic else ())])
        g.close()
    assert max(np.abs(x).max() for x in out[0]) > 0
    assert all(np.array_equal(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("case", list(KERNELS))
def test_checkpoint_interval_changes_no_bit(case):
    print(f"[gpu] checkpoint intervals {case}", flush=True)
    out = []
    for nt_dump in (7, 16, 48):
        ks = kernel_solver(case, nt_dump)
        r = [ks.forward(), *ks.adjoint(adjoint_source(ks.nstep, ks.receivers.n))]
        out.append(r + list(ks.acoustic_kernels or ()))
        ks.close()
    assert np.abs(out[0][1]).max() > 0
    for o in out[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(out[0], o))


@pytest.mark.parametrize("assembly,visco", [(2, False), (3, False), (3, True)])
def test_groups_held_at_a_time_change_no_bit(assembly, visco):
    """Ten shots are two groups of eight; with one group's local forces held at a time, each group is summed
    into accel before the next, and the update is a pass of its own."""
    from specfem3d_amd.batch import BatchSolver
    db, shots, rec = corner_to_corner(4, 1, False, [4.0 + 0.2 * k for k in range(10)])
    print(f"[gpu] groups held, assembly {assembly}, visco {visco}", flush=True)
    out = []
    for groups in (2, 1):
        b = BatchSolver(db, [(s, rec, 40 - k) for k, s in enumerate(shots)], exact=False, shots_per_group=8, assembly=assembly,
                        attenuation=attenuation(db) if visco else None)
        b.set_tuning("local_groups", groups)
        assert b.L.sf_batch_get_tuning(b.h, b"local_groups") == groups
        b.run()
        out.append([f(k) for k in range(10) for f in (b.seismograms, b.displ, b.potential)])
        b.close()
    assert max(np.abs(x).max() for x in out[0]) > 0
    assert all(np.array_equal(x, y) for x, y in zip(*out))


@pytest.mark.parametrize("nx,nz,nshots,visco,assembly", [(5, 5, 9, False, 2), (12, 10, 9, False, 2), (14, 10, 9, False, 3),
                                                         (14, 10, 3, True, 2), (32, 20, 3, True, 3)])
def test_assembly_after_a_trial(nx, nz, nshots, visco, assembly):
    """The line between the two roundings of the update, in elements x shots (a multiple of eight): 25000, with
    attenuation 160000."""
    from specfem3d_amd import sources as S
    from specfem3d_amd.batch import BatchSolver
    from specfem3d_amd.mesh.box import build_box, homogeneous
    assert (nx * nx * nz * (-(-nshots // 8) * 8) >= (160000 if visco else 25000)) == (assembly == 3)
    L = 500.0 * nx
    db = build_box(nx, nx, nz, (0.0, L, 0.0, L, -500.0 * nz, 0.0), material=homogeneous(2300.0, 2800.0, 1500.0))
    db.finalize(DT)
    src = S.setup_cmt_sources(db, [S.CMTSource(0.4 * L, 0.4 * L, 0.6, 0.0, 4.0, 1e13, 1e13, 1e13, 0.0, 0.0, 0.0)], DT, ricker=True)
    rec = S.setup_receivers(db, [S.Station("R", "T", 0.6 * L, 0.6 * L, 0.0, 0.0)])
    b = BatchSolver(db, [(src, rec, 12)] * nshots, exact=False, attenuation=attenuation(db) if visco else None)
    print(f"[gpu] trial of {nx}x{nx}x{nz} elements x {nshots} shots, attenuation {visco}", flush=True)
    assert b.autotune(2)["assembly"] == assembly
    b.close()
