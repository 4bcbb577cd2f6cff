"""The grid kernels' shared quotients (plain range), their general form outside it, and the two
ways the strips report their maxima: bitwise the oracle at states that sit on the borders.

The oracle divides and takes roots in IEEE arithmetic.  Inside the plain range (density and
pressure within 2^+-100) the kernels' quotients are the compiler's division without its range
scalings; velocities may be of any size, down to subnormal numbers, and of either zero sign.
Outside it a row falls back to full divisions, so both must give the oracle's bits (results that
are themselves subnormal excepted: nothing here makes one).
"""
import ctypes as C

import numpy as np
import pytest

from oracle import pygrid as G
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import _native as N
from quick_gpu_cfd_for_neural_network_with_converging_inputs_airfoil2d_version_amd import euler2d as E

from .grid_cases import cut_body

pytestmark = pytest.mark.gpu


def solver(nx, ny, cases, flux, scale=1.0, velocity=0.3, mco=0.7, seed=5):
    """Random states: density about 1, pressure about `scale`, velocities `velocity` times the
    sound speed; one half of the first case has velocities of exactly +0 / -0."""
    par = E.params2d_default()
    par.limiter, par.flux = E.LIM_FIRST_ORDER, flux
    s = E.Solver2D(nx, ny, 0.0, 1.0, 0.0, 0.7, cases, par)
    rng = np.random.default_rng(seed)
    for c in range(cases):
        r = rng.uniform(0.5, 2.0, (ny, nx))
        p = scale * rng.uniform(0.5, 2.0, (ny, nx))
        u, v = (velocity * np.sqrt(scale) * rng.uniform(-1, 1, (ny, nx)) for _ in range(2))
        if c == 0:
            u[: ny // 2], v[: ny // 2] = 0.0, -0.0
        s.set_primitive_field(c, r, u, v, p)
        s.set_mco(c, mco)
    return s


def check(s, steps):
    ref = G.run(s, 1e300, steps)
    with s.device_session() as d:
        status, message = d.run(1e300, steps)
        d.pull()
    assert status == ref["status"], message
    assert (s.nsteps, s.nreject) == (ref["nsteps"], ref["nreject"])
    for got, want in ((s.U, ref["u"]), (s.t, ref["t"]), (s.dt, ref["dt"])):
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("flux", [E.FLUX_HLLC, E.FLUX_AUSMPUP])
@pytest.mark.parametrize("scale, velocity", [
    (1.0, 0.3), (1.0, 3.0),          # plain
    (1.0, 1e-120), (1.0, 1e-290),    # plain, with velocities whose products underflow
    (2.0 ** -99, 0.3), (2.0 ** 98, 0.3),    # the last plain pressures: some cells on either side
    (2.0 ** -140, 0.3), (2.0 ** 140, 0.3),  # general
])
def test_states_at_the_borders_of_the_plain_range(flux, scale, velocity):
    check(solver(70, 9, 2, flux, scale, velocity), 6)


@pytest.mark.parametrize("flux", [E.FLUX_HLLC, E.FLUX_AUSMPUP])
def test_one_odd_row_among_plain_ones(flux):
    s = solver(130, 12, 1, flux)
    q = s.field(0)
    q[3, 7, 40] = 2.0 ** 101  # energy beyond the plain range in one cell: its row takes the general form
    check(s, 3)


def test_reference_mach_number_outside_the_plain_range():
    check(solver(64, 8, 2, E.FLUX_AUSMPUP, mco=2.0 ** -120), 4)


@pytest.mark.parametrize("mco", [0.0, float("nan"), 2.0 ** -120])
def test_reference_mach_number_that_hllc_does_not_read(mco):
    """HLLC reads no reference Mach number, so none may take its grid from the shared quotients (the
    three stages of 4 cases of 512 x 512: 116 us, 150 in the general form)."""
    check(solver(64, 8, 2, E.FLUX_HLLC, mco=mco), 4)
    best = {}
    for value in (0.7, mco):
        with solver(512, 512, 4, E.FLUX_HLLC, mco=value).device_session() as d:
            us, err = (C.c_double * 3)(), N.err_buffer()
            for _ in range(5):
                assert not d.lib.ugrid_profile(d.handle, 10, us, err, N.ERR_LEN), err.value
                best.setdefault(str(value), []).append(sum(us))
    plain, other = (min(v) for v in best.values())
    print("stages us, mco 0.7:", plain, f"mco {mco}:", other, flush=True)
    assert other < 1.2 * plain


@pytest.mark.parametrize("cases", [1023, 1025])  # strips' partials in the decision kernel's table / atomics
def test_many_cases(cases):
    check(solver(3, 4, cases, E.FLUX_HLLC), 5)


@pytest.mark.parametrize("nx, ny, cases", [(1, 1, 1), (62, 1, 3), (63, 65, 1), (124, 130, 2), (500, 77, 5)])
def test_strip_lengths(nx, ny, cases):
    check(solver(nx, ny, cases, E.FLUX_HLLC), 4)


@pytest.mark.parametrize("bc", [(0, 0, 0, 0), (1, 1, 2, 2), (2, 1, 0, 0), (2, 2, 1, 2)])
@pytest.mark.parametrize("nx, ny", [(2, 2), (2, 7), (70, 3), (1, 5)])  # ghosts filled on the device, and by the host
def test_downloaded_ghosts(bc, nx, ny):
    """Ghost cells of a downloaded state, while steps remain and after the last, and of a state
    downloaded again after more steps; before the first step they are the uploaded ones."""
    s = solver(nx, ny, 3, E.FLUX_HLLC)
    if (nx < 2 and (bc[0] != 1 or bc[1] != 1)):
        pytest.skip("the reference's fill of a one-cell reflect or periodic axis reads another ghost")
    s.par.bc = list(bc)
    s.U[:] = np.where(s.U == 0.0, 7.0, s.U)  # ghost cells as the caller left them
    first = s.U.copy()
    with s.device_session() as d:
        d.pull()
        np.testing.assert_array_equal(s.U, first)
        done = 0
        for steps in (2, 3):
            s.U[:] = first
            s.t[:], s.dt[:] = 0.0, 0.0
            done += steps
            ref = G.run(s, 1e300, done)
            d.run(1e300, steps)
            d.pull()
            if steps == 2:
                np.testing.assert_array_equal(s.U, ref["u"])
        inner = s.U.reshape(3, 4, ny + 4, nx + 4)[:, :, 2:-2, 2:-2]
        np.testing.assert_array_equal(inner, ref["u"].reshape(3, 4, ny + 4, nx + 4)[:, :, 2:-2, 2:-2])
        np.testing.assert_array_equal(s.U, ref["u"])


@pytest.mark.parametrize("cases", [3, 1023, 1025])  # norms by the strips' partials / by atomics
def test_many_cases_implicit(cases):
    """Backward Euler with refused candidates (each formed again from the same iterate) and steps of
    more updates than one round of launches holds."""
    s = solver(5, 4, cases, E.FLUX_HLLC)
    s.par.time_integrator, s.par.cfl, s.par.pseudo_cfl = E.TIME_BACKWARD_EULER, 2.0, 1000.0
    ref = G.run_implicit(s, 1e300, 2)
    assert ref["updates"] > 16
    with s.device_session() as d:
        status, _ = d.run(1e300, 2)
        got = d.implicit_stats()
        d.pull()
    assert status == ref["status"]
    for key in ("updates", "retries", "checks", "initial_defect", "final_defect"):
        assert got[key] == ref[key], key
    np.testing.assert_array_equal(s.U, ref["u"])
    np.testing.assert_array_equal(s.t, ref["t"])


@pytest.mark.parametrize("halvings", [1, 6, 7, 8, 9, 12, 13])  # within, at and past one pre-check's steps, and too many
@pytest.mark.parametrize("flux", [E.FLUX_HLLC, E.FLUX_AUSMPUP])
def test_halvings_of_a_step_on_a_cut_grid(flux, halvings):
    par = E.params2d_default()
    par.limiter, par.flux = E.LIM_FIRST_ORDER, flux
    par.dt_fixed = 2.0 ** (halvings - 11)  # 2^-11 is admissible in the smallest cut cells
    s, _, _ = cut_body("circle", 52, 40, par, shock=-0.6)
    ref = G.run(s, 1e300, 1)
    assert ref["nreject"] == halvings and ref["status"] == (2 if halvings == 13 else 1)
    check(s, 1)
