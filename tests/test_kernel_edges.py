"""Kernels at the sizes where their blocking can go wrong (edges of panels and tiles,
remainders, the smallest and largest of their range), against the CPU oracle (GPU tests)."""
import numpy as np
import pytest

import rpcf
from helpers import rel

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


# lengths without a compiled plan: N odd and even, row tiles of the Chebyshev products whole,
# one row over and partial (N/2 + 1 = 8 .. 126 rows), the largest N; ragged pencil tiles; x and
# span lengths with radices 2 to 8, 3 and 5.  The library's bars: 1e-12 after one step, 1e-13
# for a transform of one field.
@pytest.mark.parametrize("N,mx,my", [(15, 30, 20), (25, 36, 54), (27, 20, 30), (30, 54, 24), (36, 50, 36), (45, 24, 90),
                                     (50, 40, 60), (75, 72, 18), (81, 48, 20), (125, 12, 30), (160, 18, 24),
                                     (225, 12, 12), (243, 10, 12), (250, 12, 10)])
def test_lengths_without_compiled_plans(N, mx, my):
    channel = N % 2 == 0
    prm = rpcf.make_params(mx, my, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=900.0, Ro=0.1, dt=0.002,
                           u_profile=(1.0, 0.0, -1.0) if channel else (0.0, 1.0, 0.0), flow_control=int(channel))
    g, o = pair(prm)
    v, e = rpcf.seed_state(g.dll, prm, 5, 0.1, 3, 8, 0.5)
    for s in (g, o):
        s.set_state(v, e)
        s.nonlinear()
    assert rel(g.get_nonlinear()[1], o.get_nonlinear()[1]) < 1e-12
    for s in (g, o):
        s.step(1)
    for a, b in zip(g.get_state(), o.get_state()):
        assert rel(a, b) < 1e-12
    for padded in (True, False):
        assert rel(g.spec_to_phys(v, padded), o.spec_to_phys(v, padded)) < 1e-13
    g.close(), o.close()


XY_LENGTHS = [24, 30, 32, 36, 40, 48, 50, 54, 60, 64, 72, 80, 90, 96, 100, 108, 120, 128, 144, 150, 160, 162, 180, 192,
              200, 216, 240, 250, 256, 270, 288, 300, 320, 324, 360, 384, 400, 512]


# span transforms of every compiled length and one longer than them: tiles of 8 and 16 columns
# whole, partial and of one column (nx/2 = 3 .. 18 columns in, nx/2 + 1 out), every butterfly's
# zeroed and dropped rows
@pytest.mark.parametrize("my", XY_LENGTHS)
def test_span_transforms(my):
    g, o = pair(rpcf.make_params((10, 24, 50, 54)[XY_LENGTHS.index(my) % 4], my, 40, n_pi_x=2.0, n_pi_y=1.0))
    rng = np.random.default_rng(my)
    a = rng.standard_normal((g.s["P"], g.s["nz"])) + 1j * rng.standard_normal((g.s["P"], g.s["nz"]))
    p, q = g.spec_to_phys(a), o.spec_to_phys(a)
    assert rel(p, q) < 1e-13
    f = rng.standard_normal(q.shape)
    assert rel(g.phys_to_spec(f), o.phys_to_spec(f)) < 1e-13
    g.close(), o.close()


# the x transforms and products of every compiled length: whole and partial tiles of row pairs
# (5, 12 and 27 pairs).  The library's bar for N after one evaluation.  (512 is refused for mx.)
@pytest.mark.parametrize("mx", XY_LENGTHS[:-1])
def test_lamb_vector(mx):
    prm = rpcf.make_params(mx, (10, 24, 54)[XY_LENGTHS.index(mx) % 3], 40, n_pi_x=2.0, n_pi_y=1.0, Re=900.0, Ro=0.1,
                           dt=0.002)
    g, o = pair(prm)
    rng = np.random.default_rng(mx)
    shape = g.s["P"], g.s["nz"]
    f = [(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / (1.0 + np.arange(g.s["nz"])) ** 2
         for _ in range(6)]
    for s in (g, o):
        for i in range(6):
            s.set_field(i, f[i])
        s.nonlinear()
    for a, b in zip(g.get_nonlinear(), o.get_nonlinear()):
        assert rel(a, b) < 1e-12
    g.close(), o.close()


# padded values by products: blocks of one, two and four groups of 16 pencils, of groups of 8, whole
# and ragged groups; N odd and even, rows below N/2 that fill tiles, leave one over or are few
@pytest.mark.parametrize("N,mx,my", [(4, 24, 24), (5, 30, 24), (16, 128, 384), (32, 24, 36), (36, 30, 24), (45, 128, 192),
                                     (45, 60, 90), (64, 128, 192), (75, 24, 54), (100, 12, 30), (128, 128, 96),
                                     (192, 24, 36)])
def test_padded_values(N, mx, my):
    g, o = pair(rpcf.make_params(mx, my, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=900.0, Ro=0.1, dt=0.002))
    rng = np.random.default_rng(N + mx)
    shape = g.s["P"], g.s["nz"]
    f = [(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / (1.0 + np.arange(g.s["nz"])) ** 2
         for _ in range(6)]
    for s in (g, o):
        for i in range(6):
            s.set_field(i, f[i])
        s.nonlinear()
    for a, b in zip(g.get_nonlinear(), o.get_nonlinear()):
        assert rel(a, b) < 1e-12
    assert rel(g.spec_to_phys(f[0]), o.spec_to_phys(f[0])) < 1e-13
    g.close(), o.close()


# velocity recovery: half a wave, one to four coefficients a lane, whole, one over and partial;
# pencils that fill blocks of 4 and 8 and not.  Sums of at most N/2 terms without cancellation:
# N/2 2^-53 = 1.4e-14 relative at most.
@pytest.mark.parametrize("N", [4, 5, 30, 32, 36, 60, 64, 72, 120, 128, 135, 160, 192, 200, 225, 250])
def test_velocity(N):
    g, o = pair(rpcf.make_params(12 if N % 2 else 18, 18, 4 * N, n_pi_x=2.0, n_pi_y=1.0))
    rng = np.random.default_rng(N)
    shape = g.s["P"], g.s["nz"]
    state = [rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for _ in range(2)]
    for s in (g, o):
        s.set_state(*state)
        s.velocity()
    for i in range(6):
        assert rel(g.get_field(i), o.get_field(i)) < 1e-13, i
    g.close(), o.close()


# solves of an odd base profile by conjugate parity blocks, at N odd and even, the smallest pair
# counts, row pairs that fill whole and partial batches of every column group, the largest N: the
# full inverses' results after one step.  2e-13 is the bound of the even profiles' blocks with
# remainders (2^-9 of the 1e-11 the blocks alone leave).  Without stored remainders the same values are formed from the full inverses.
@pytest.mark.parametrize("N", [4, 5, 6, 12, 27, 48, 64, 75, 96, 125, 128, 160, 250])
@pytest.mark.parametrize("precision", [0, 2])
def test_odd_profile_solves(N, precision, monkeypatch):
    def step(p, full):
        monkeypatch.setenv("RPCF_FULL_INVERSE", str(int(full)))
        prm = rpcf.make_params(24, 24, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=1300.0, Ro=0.1, dt=0.002,
                               u_profile=(0.0, 1.0, 0.0), precision=p)
        with rpcf.Simulation(rpcf.HIP_LIB, prm) as s:
            if N < 12:  # no room for a seed that satisfies the wall conditions
                rng = np.random.default_rng(N)
                shape = s.s["P"], s.s["nz"]
                s.set_state(*(rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for _ in range(2)))
            else:
                s.set_state(*rpcf.seed_state(s.dll, prm, 0, 0.1, 4, min(24, N - 5), 5.0 / 6.0, True))
            s.bootstrap()
            return s.get_state()

    a, f = step(precision, False), step(precision, True)
    e = max(rel(x, y) for x, y in zip(a, f))
    print("N=%d precision %d: blocks vs full inverses %.2e" % (N, precision, e))
    assert e < 2e-13
    if precision == 2:
        b = step(0, False)
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


# x and span lengths whose run-time plan has no room in LDS for its twiddles beside the tile, and
# the longest that have: one row pair or column, and a few.  The library's bars, as above.
@pytest.mark.parametrize("mx,my", [(486, 10), (500, 18), (540, 12), (12, 400), (24, 1000), (18, 1620), (12, 1728), (6, 3240)])
def test_long_lengths(mx, my):
    prm = rpcf.make_params(mx, my, 24, n_pi_x=2.0, n_pi_y=1.0, Re=900.0, Ro=0.1, dt=0.002)
    g, o = pair(prm)
    rng = np.random.default_rng(mx + my)
    shape = g.s["P"], g.s["nz"]
    f = [(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / (1.0 + np.arange(g.s["nz"])) ** 2
         for _ in range(6)]
    for s in (g, o):
        for i in range(6):
            s.set_field(i, f[i])
        s.nonlinear()
    for a, b in zip(g.get_nonlinear(), o.get_nonlinear()):
        assert rel(a, b) < 1e-12
    p, q = g.spec_to_phys(f[0]), o.spec_to_phys(f[0])
    assert rel(p, q) < 1e-13
    f = rng.standard_normal(q.shape)
    assert rel(g.phys_to_spec(f), o.phys_to_spec(f)) < 1e-13
    g.close(), o.close()


# profiles that are not even keep both FP64 inverses whole at every size: the state after a step is,
# bit for bit, that of RPCF_FULL_INVERSE=1
@pytest.mark.parametrize("N,mx", [(32, 24), (64, 24), (75, 24), (96, 24), (128, 24), (160, 24), (40, 192)])
@pytest.mark.parametrize("profile", [(0.0, 1.0, 0.0), (0.5, 0.5, 0.0)])
@pytest.mark.parametrize("precision", [0, 2])
def test_other_profiles_solve_with_the_full_inverses(N, mx, profile, precision, monkeypatch):
    def step(full):
        monkeypatch.setenv("RPCF_FULL_INVERSE", str(full))
        prm = rpcf.make_params(mx, mx, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=1300.0, Ro=0.1, dt=0.002,
                               u_profile=profile, precision=precision)
        with rpcf.Simulation(rpcf.HIP_LIB, prm) as s:
            s.set_state(*rpcf.seed_state(s.dll, prm, 0, 0.1, 4, 24, 5.0 / 6.0, True))
            s.bootstrap()
            return s.get_state()

    for a, b in zip(step(0), step(1)):
        assert np.array_equal(a, b)


# a member alone and beside others whose blocks together outnumber the compute units (16-sample
# chunks in the padded p2s, wider blocks in the padded s2p): the same bits.  N with and without a
# compiled plan, with the centre row N/2 in a tile of its own (32, 96, 128, 192) and not.
@pytest.mark.parametrize("N,mx,my,members", [(24, 96, 96, 2), (32, 96, 96, 2), (45, 60, 90, 4), (48, 96, 96, 2),
                                             (96, 96, 96, 2), (128, 48, 96, 2), (192, 48, 96, 2)])
def test_member_alone_and_in_a_full_group(N, mx, my, members):
    def prm(i):
        return rpcf.make_params(mx, my, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=900.0 + 100 * i, Ro=0.1, dt=0.002,
                                u_profile=(1.0, 0.0, -1.0), flow_control=1)

    def initial(i):
        return rpcf.seed_state(rpcf.load(rpcf.HIP_LIB), prm(i), i, 0.1, 4, 12, 5.0 / 6.0, True)

    ids = list(range(members))
    with rpcf.Group(rpcf.HIP_LIB, prm(0), members) as g:
        for i in ids:
            g.init(i, prm(i))
            g.set_state(i, *initial(i))
        g.bootstrap(ids)
        g.step(ids, 2)
        got = [g.get_state(i) for i in ids]
    for i in (0, members - 1):
        with rpcf.Simulation(rpcf.HIP_LIB, prm(i)) as s:
            s.set_state(*initial(i))
            s.bootstrap()
            s.step(2)
            for a, b in zip(s.get_state(), got[i]):
                assert np.array_equal(a, b), i


# the padded p2s in chunks of 16 samples (more blocks than compute units) at the lengths the grids
# above leave out: chunks of 12 and 16 samples, row tiles in one block and in two
@pytest.mark.parametrize("N,mx,my", [(24, 128, 192), (48, 128, 192), (96, 128, 192), (192, 96, 96)])
def test_padded_p2s_with_many_blocks(N, mx, my):
    g, o = pair(rpcf.make_params(mx, my, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=900.0, Ro=0.1, dt=0.002))
    rng = np.random.default_rng(N)
    shape = g.s["P"], g.s["nz"]
    f = [(rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / (1.0 + np.arange(g.s["nz"])) ** 2
         for _ in range(6)]
    for s in (g, o):
        for i in range(6):
            s.set_field(i, f[i])
        s.nonlinear()
    for a, b in zip(g.get_nonlinear(), o.get_nonlinear()):
        assert rel(a, b) < 1e-12
    g.close(), o.close()


# even profiles solve with the parity blocks and their v remainders at every size up to the longest
# compiled one: N odd (no centre row) and even, the smallest pair counts, row pairs that fill whole
# and partial batches of every column group; inverses of a few kB and (N = 40) of more than 0.2 GB.  The full
# inverses' results after one step, to the library's bar -- and not their bits, which would mean
# that the full inverses were read.
@pytest.mark.parametrize("N,mx", [(4, 24), (5, 24), (6, 24), (12, 24), (15, 24), (27, 24), (32, 24), (36, 24), (45, 24),
                                  (48, 24), (60, 24), (64, 24), (75, 24), (81, 24), (96, 24), (125, 24), (128, 24),
                                  (160, 24), (192, 24), (40, 192)])
def test_even_profile_solves(N, mx, monkeypatch):
    def step(full):
        monkeypatch.setenv("RPCF_FULL_INVERSE", str(full))
        prm = rpcf.make_params(mx, mx, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=1300.0, Ro=0.1, dt=0.002,
                               u_profile=(1.0, 0.0, -1.0), flow_control=1)
        with rpcf.Simulation(rpcf.HIP_LIB, prm) as s:
            if N < 12:  # no room for a seed that satisfies the wall conditions
                rng = np.random.default_rng(N)
                shape = s.s["P"], s.s["nz"]
                s.set_state(*(rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for _ in range(2)))
            else:
                s.set_state(*rpcf.seed_state(s.dll, prm, 0, 0.1, 4, min(24, N - 5), 5.0 / 6.0, True))
            s.bootstrap()
            return s.get_state()

    for a, f in zip(step(0), step(1)):
        print("N=%d: blocks vs full inverses %.2e" % (N, rel(a, f)))
        assert rel(a, f) < 1e-12
        assert not np.array_equal(a, f)


# past N = 192 the FP64 solves of even profiles read the full inverses, whose results the remainders
# in BF16 no longer restore: the library's bar against the oracle after one step
@pytest.mark.parametrize("N", [200, 216, 225, 240, 243, 250])
def test_even_profile_past_the_compiled_lengths(N):
    prm = rpcf.make_params(12, 12, 4 * N, n_pi_x=2.0, n_pi_y=1.0, Re=1300.0, Ro=0.1, dt=0.002,
                           u_profile=(1.0, 0.0, -1.0), flow_control=1)
    g, o = pair(prm)
    for s in (g, o):
        s.set_state(*rpcf.seed_state(s.dll, prm, 0, 0.1, 4, 24, 5.0 / 6.0, True))
        s.bootstrap()
    for a, b in zip(g.get_state(), o.get_state()):
        print("N=%d: one step against the oracle %.2e" % (N, rel(a, b)))
        assert rel(a, b) < 1e-12
    g.close(), o.close()
