"""Gather assembly fused with the Newmark update: fields read and written between the steps, where the
sum is taken early, the acceleration is not known to be zero, or both. Without FMA contraction every
path sums in the oracle's order, so the fields equal its bit for bit."""
import ctypes as C

import numpy as np
import pytest

from conftest import small_elastic_box, smooth_warp

pytestmark = pytest.mark.gpu


def put_fields(g, u, v, a):
    n = C.c_int(u.size)
    p = [x.ctypes.data_as(C.c_void_p) for x in (u, v, a)]
    g.L.transfer_fields_el_to_device_(C.byref(n), *p, g.MP)


@pytest.mark.parametrize("assembly", [0, 1])
@pytest.mark.parametrize("n,warp", [(1, False), (2, True), (5, False)])
def test_fields_between_steps(oracle_mod, n, warp, assembly):
    from specfem3d_amd.solver import GPUSolver
    db, src, rec = small_elastic_box(n=n, warp=smooth_warp(500.0 * n) if warp else None)
    o = oracle_mod.OracleSolver(db, src, rec, "f32")
    o.stf_table = src.stf_table(40)
    o.run(6)
    g = GPUSolver(db, src, rec, nstep=40, exact=True, assembly=assembly)
    print(f"[gpu] gather n={n} warp={warp} assembly={assembly}", flush=True)
    for _ in range(6):
        g.step()
    rng = np.random.default_rng(n)
    u, v, a = (rng.normal(size=3 * db.nglob).astype(np.float32) * s for s in (1e-3, 1e-1, 1e1))
    put_fields(g, u, v, a)            # an acceleration that is nonzero everywhere
    o.displ[:], o.veloc[:], o.accel[:] = u, v, a
    for k in range(6):
        g.step()
        o.run(1)
        if k % 2:                     # sum and corrector before the next update
            for x, y in zip(g.fields(), (o.displ, o.veloc, o.accel)):
                assert np.array_equal(x, y), k
    for x, y in zip(g.fields(), (o.displ, o.veloc, o.accel)):
        assert np.array_equal(x, y)
    g.close()


@pytest.mark.parametrize("order", [None, "morton"])
@pytest.mark.parametrize("n", [2, 3, 6])
def test_mixed_elements(oracle_mod, n, order):
    """Cubes and irregular elements in one workgroup (five elements, a lane one line of points), element
    counts with every remainder: 8, 27, 216; the launch order moves the slots, not the sums."""
    from specfem3d_amd.solver import GPUSolver
    L = 500.0 * n

    def bend(x, y, z):                # the element corners inside x < 3L/4, y < 3L/4 move, the others stay
        d = 30.0 * ((x > 0) & (x < 0.75 * L) & (y > 0) & (y < 0.75 * L) & (z < 0) & (z > -L))
        return x + d, y - 0.5 * d, z + 0.7 * d

    db, src, rec = small_elastic_box(n=n, warp=bend)
    print(f"[gpu] mixed n={n} irregular={db.nspec_irregular} of {db.nspec}", flush=True)
    assert db.nspec_irregular > 0 and (n < 3 or db.nspec_irregular < db.nspec)
    ref = oracle_mod.OracleSolver(db, src, rec, "f32").run(60)
    g = GPUSolver(db, src, rec, nstep=60, exact=True, assembly=1, element_order=order)
    out = g.run().copy()
    g.close()
    assert np.abs(ref).max() > 0 and np.array_equal(out, ref)
    g = GPUSolver(db, src, rec, nstep=60, exact=False, assembly=-1)
    fast = g.run().copy()
    g.close()
    e = np.linalg.norm((fast - ref).astype(np.float64)) / np.linalg.norm(ref.astype(np.float64))
    assert e < 1e-5, e


@pytest.mark.parametrize("n,warp", [(2, False), (3, True), (5, False)])
def test_potentials_between_steps(oracle_mod, n, warp):
    """The fluid's sums, fused with its update and free surface, under a solid bottom layer: potentials put
    between the steps (nonzero on the free surface too) and read back after every step, every second, or at
    the end."""
    from specfem3d_amd import sources as S
    from specfem3d_amd.mesh.box import build_box, homogeneous
    from specfem3d_amd.solver import GPUSolver
    L = 500.0 * n
    ext = (0.0, L, 0.0, L, -L, 0.0)
    db = build_box(n, n, n, ext, material=homogeneous(2300.0, 2800.0, 1500.0), acoustic_top_layers=n - 1,
                   acoustic_material=homogeneous(1020.0, 1500.0, 0.0), warp=smooth_warp(L) if warp else None,
                   stacey_faces=(1, 2, 3, 4, 5))
    db.finalize(0.004, stacey=True)
    src = S.setup_cmt_sources(db, [S.CMTSource(0.43 * L, 0.57 * L, 0.3 * L / 1000.0, 0.0, 0.06, 3e13, 2e13, 3e13,
                                               1e12, 0.0, 0.0)], 0.004)
    assert db.ispec_is_acoustic[src.ispec].all()
    wet = np.unique(db.ibool[np.asarray(db.ispec_is_acoustic, bool)].ravel()).astype(np.int64)
    wet = wet - int(db.ibool.min())
    rng = np.random.default_rng(n)
    put = [np.zeros(db.nglob, np.float32) for _ in range(3)]
    for x, s in zip(put, (1e2, 1e4, 1e6)):
        x[wet] = rng.normal(size=wet.size).astype(np.float32) * np.float32(s)
    for every in (1, 2, 12):
        o = oracle_mod.OracleSolver(db, src, None, "f32")
        o.stf_table = src.stf_table(40)
        g = GPUSolver(db, src, None, nstep=40, exact=True, assembly=1)
        print(f"[gpu] fluid gather n={n} warp={warp} every={every}", flush=True)
        for k in range(12):
            if k == 4:
                nn = C.c_int(db.nglob)
                g.L.transfer_fields_ac_to_device_(C.byref(nn), *[x.ctypes.data_as(C.c_void_p) for x in put], g.MP)
                o.pot[:], o.potd[:], o.potdd[:] = put
            g.step()
            o.run(1)
            if (k + 1) % every == 0:
                for x, y in zip(g.potentials(), (o.pot, o.potd, o.potdd)):
                    assert np.array_equal(x, y), (every, k)
        g.close()


@pytest.mark.parametrize("nsrc", [1, 256, 257])
def test_source_values(oracle_mod, nsrc):
    """Source time functions as launch arguments (up to 256) and through device memory, sources of
    neighbouring elements adding to shared points in the reference's order."""
    from specfem3d_amd import sources as S
    from specfem3d_amd.solver import GPUSolver
    n, dt = 7, 0.004
    db, _, rec = small_elastic_box(n=n, dt=dt)
    L = 500.0 * n
    cmt = []
    for q in range(nsrc):
        e = (q * 2) % 343
        x, y, z = (0.5 + e % 7) * 500.0, (0.5 + (e // 7) % 7) * 500.0, (0.5 + e // 49) * 500.0
        cmt.append(S.CMTSource(x, y, z / 1000.0, 0.0, 0.05 + 1e-4 * q, 1e13, 1e13 + q * 1e10, -1e13, 0.0, 1e12, 0.0))
    src = S.setup_cmt_sources(db, cmt, dt)
    assert src.n == nsrc and x < L
    ref = oracle_mod.OracleSolver(db, src, rec, "f32").run(12)
    g = GPUSolver(db, src, rec, nstep=12, exact=True, assembly=1)
    print(f"[gpu] {nsrc} sources", flush=True)
    out = g.run().copy()
    g.close()
    assert np.abs(ref).max() > 0 and np.array_equal(out, ref)


@pytest.mark.parametrize("n,warp,nt_dump", [(2, False, 7), (3, True, 40), (5, False, 16)])
def test_kernel_run_low_parts(oracle_mod, n, warp, nt_dump):
    """FMA kernel runs carry u and v with low parts through fused and separate updates, snapshots, history
    frames and fields put to zero. Tolerance: the moduli, masses and tables in single precision (about
    eight factors of 2^-24 on the way from displacement to displacement) and the rounding of the forces
    in each of 40 steps, 2^-24 (8 + sqrt(40)) = 8.5e-7, times 6 for the fields of a product."""
    from specfem3d_amd.adjoint import KernelSolver
    nstep, tol = 40, 5e-6
    db, src, rec = small_elastic_box(n=n, warp=smooth_warp(500.0 * n) if warp else None, dt=0.008)
    t = np.arange(nstep)[:, None, None] / nstep
    r, c = np.arange(rec.n)[None, :, None], np.arange(3)[None, None, :]
    adj = (np.sin(2 * np.pi * (2 * t + 0.17 * r + 0.3 * c)) * np.sin(np.pi * t)).astype(np.float32)
    ref = oracle_mod.kernel_run(db, src, rec, nstep, adj.astype(np.float64), nt_dump, "f64")
    print(f"[gpu] low parts n={n} warp={warp} nt_dump={nt_dump}", flush=True)
    ks = KernelSolver(db, src, rec, nstep, nt_dump=nt_dump, exact=False, assembly=-1)
    seis = ks.forward()
    k = ks.adjoint(adj)
    seis2, k2 = ks.seis_d[: nstep].copy(), ks.adjoint(adj)      # the same run again gives the same bits
    ks.close()
    assert all(np.array_equal(a, b) for a, b in zip(k, k2)) and np.array_equal(seis, seis2[: len(seis)])
    for name, a, b in zip(("seis", "rho", "mu", "kappa"), (seis,) + tuple(k), ref):
        e = np.linalg.norm(a.ravel().astype(np.float64) - b.ravel()) / np.linalg.norm(b)
        print(f"[gpu]   {name} {e:.2e}", flush=True)
        assert np.abs(b).max() > 0 and e < tol, (name, e)
