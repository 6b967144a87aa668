"""Kernels at the sizes where their blocking can go wrong (edges of panels and tiles,
remainders, the smallest and largest of their range), against the CPU oracle (GPU tests)."""
import numpy as np
import pytest

import rpcf

pytestmark = pytest.mark.gpu


def pair(prm):
    return rpcf.Simulation(rpcf.HIP_LIB, prm), rpcf.Simulation(rpcf.ORACLE_LIB, prm)


# nz below, at and above whole panels of 16 columns and waves of 64 columns, and the largest
@pytest.mark.parametrize("nz", [5, 16, 17, 31, 49, 65, 76, 129, 251])
@pytest.mark.parametrize("profile", [(1.0, 0.0, -1.0), (0.5, 0.5, 0.0)])
def test_inverses_bit_identical(nz, profile):
    prm = rpcf.make_params(6, 6, 4 * (nz - 1), n_pi_x=2.0, n_pi_y=1.0, Re=900.0, dt=0.004, u_profile=profile)
    g, o = pair(prm)
    for eq in (0, 1):
        for p in range(g.s["P"]):
            assert np.array_equal(g.get_inverse(eq, p), o.get_inverse(eq, p)), (eq, p)
    g.close(), o.close()
