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


# spectral arrays below and above the size that crosses through pinned buffers (8 MB), whole
# and partial pieces, contiguous and padded pencils: what goes in comes out, bit for bit, and
# the caller's padding is left alone
@pytest.mark.parametrize("grid", [(24, 24, 64), (192, 192, 240), (192, 192, 256)])
@pytest.mark.parametrize("pad", [0, 3])
def test_state_crosses_the_boundary_unchanged(grid, pad):
    prm = rpcf.make_params(*grid)
    with rpcf.Simulation(rpcf.HIP_LIB, prm) as sim:
        P, nz = sim.s["P"], sim.s["nz"]
        rng = np.random.default_rng(3)
        v, e = (rng.standard_normal((P, nz + pad)) + 1j * rng.standard_normal((P, nz + pad)) for _ in range(2))
        sim.set_state(v, e)
        a, b = sim.get_state()
        assert np.array_equal(a, v[:, :nz]) and np.array_equal(b, e[:, :nz])
        out = np.full((2, P, nz + pad), 7.0 + 1j)
        ptr = [x.view(np.float64).ctypes.data_as(rpcf.binding._dp) for x in out]
        assert sim.dll.rpcf_get_state(sim.h, ptr[0], ptr[1], nz + pad) == 0
        assert np.array_equal(out[0, :, :nz], a) and np.array_equal(out[1, :, :nz], b)
        assert (out[:, :, nz:] == 7.0 + 1j).all()
