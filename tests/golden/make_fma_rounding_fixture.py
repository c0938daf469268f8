"""Write golden/fma_rounding.npz: outputs of the FMA builds on the cases of tests/test_gpu_fma_rounding.py.

Run on a GPU, with the package whose rounding is to be kept first on the path:

    PYTHONPATH=<tree> python tests/golden/make_fma_rounding_fixture.py [out.npz]

The fixture was written by the library of commit f9a7498, whose element launches scattered their forces
colour by colour. (The values have no other source: no closed form and no reference run has this rounding.)
"""
import os
import sys

import numpy as np

import specfem3d_amd  # the tree on the path, before the test's own is put in front of it

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(1, os.path.dirname(HERE))

if __name__ == "__main__":
    import test_gpu_fma_rounding as T
    out = {f"{c}/{k}": v for c in T.CASES for k, v in T.outputs(c).items()}
    path = sys.argv[1] if len(sys.argv) > 1 else os.path.join(HERE, "fma_rounding.npz")
    np.savez_compressed(path, **out)
    print("wrote", path, "with", specfem3d_amd.__file__, {k: v.shape for k, v in out.items()})
