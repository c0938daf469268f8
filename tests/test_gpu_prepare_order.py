"""The fluid prepared after the solid: the coupling points take their terms all the same."""
import numpy as np
import pytest

from conftest import small_coupled_box

pytestmark = pytest.mark.gpu


class SolidFirst:
    """The library with prepare_fields_acoustic_device put behind prepare_fields_elastic_device."""

    def __init__(self, lib):
        self.lib, self.late = lib, None

    def __getattr__(self, name):
        f = getattr(self.lib, name)
        if name == "prepare_fields_acoustic_device_":
            return lambda *a: setattr(self, "late", (f, a))
        if name == "prepare_fields_elastic_device_":
            def both(*a):
                f(*a)
                g, b = self.late
                g(*b)
            return both
        return f


@pytest.mark.parametrize("exact,assembly", [(True, 1), (False, 2)])
def test_fluid_prepared_after_the_solid(monkeypatch, exact, assembly):
    from specfem3d_amd import abi
    from specfem3d_amd.solver import GPUSolver
    db, src, rec = small_coupled_box(n=3, dt=0.006, nrec=3, seed=2)
    lib = abi.load()
    print(f"[gpu] solid prepared first, exact={exact}", flush=True)
    out = []
    for load in (lambda: lib, lambda: SolidFirst(lib)):
        monkeypatch.setattr(abi, "load", load)
        g = GPUSolver(db, src, rec, nstep=60, exact=exact, assembly=assembly)
        g.run()
        out.append([g.seis_d.copy(), *g.fields(), *g.potentials()])
        g.close()
    assert all(np.abs(x).max() > 0 for x in out[0])
    assert all(np.array_equal(x, y) for x, y in zip(*out))
