"""RK4 and SSP-RK3 in stage pairs (2-flavour boxes, periodic and open in z): against the oracle at
shapes that leave the x groups (8 to 16 rows), the z segments and the
last direction chunk partly filled, boxes narrower than the stencils' reach,
and mixed with the paths that keep other records of the state."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nx, nz, refinement (nv = 10 nn^2 + 2), z-segment length (0: the plan's own)
SHAPES = [(1, 40, 2, 0), (2, 3, 1, 0), (3, 1, 1, 0), (5, 4, 3, 3), (8, 17, 2, 5), (9, 33, 3, 32), (12, 16, 4, 1),
          (13, 29, 2, 7), (25, 70, 3, 0)]
H = 0.125


def geo(nx, nz):
    return dict(x0=-nx * H / 2, x1=nx * H / 2, z0=-nz * H / 2, z1=nz * H / 2, dx=H, dz=H)


INIT = dict(ipt=5, alpha=0.85, eps0=0.1, sigma=1.0, lnue=0.6, lnueb=0.5, seed=77)
PHYS = dict(ko=0.1, mu=1.3, pmo=0.7)


def make(N, nx, nz, nn, **kw):
    g = N.NuOsc(nv=nn, CFL=0.4, **geo(nx, nz), **PHYS, **kw)
    g.fillInitValue(**INIT)
    return g


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("scheme", ["rk4", "srk3"])
def test_pairs_match_oracle(nuosc_mod, oracle_mod, shape, precision, scheme):
    """FP64: 1e-12 per field over 9 steps (a few roundings each).  FP32: one
    rounding (2^-24) per store of Y3, A and u' and about four per stage update,
    grown by at most e^(gamma t) < 2: 9 steps x 8 x 2^-24 x 2 = 8.6e-6."""
    nx, nz, nn, zlen = shape
    g = make(nuosc_mod, nx, nz, nn, precision=precision)
    o = oracle_mod.OracleSim(nn=nn, cfl=0.4, **geo(nx, nz), **PHYS)
    o.fill_init(**INIT)
    if zlen:
        g.set_zlen(zlen)
    for n in (1, 2, 6):     # odd and even numbers of exchanges of the state copies
        (g.step_rk4 if scheme == "rk4" else g.step_srk3)(n)
        (o.step if scheme == "rk4" else o.step_srk3)(n)
    a, b = g.get_state(), o.get_state()
    tol = 1e-12 if precision == 64 else 9 * 8 * 2.0 ** -24 * 2
    for f in range(8):
        assert np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[:4] if f < 4 else b[4:])), f
    assert abs(g.phy_time - 9 * g.dt) < 1e-12


@pytest.mark.parametrize("precision", [64, 32])
def test_pairs_split_and_segments_bitwise(nuosc_mod, precision):
    """The state does not depend on how the steps are split into calls, on
    graph replay, on the z segments or on profiling."""
    runs = []
    for kw, zlen, calls in ((dict(use_graph=True), 0, (7,)), (dict(use_graph=False), 0, (1, 2, 1, 3)),
                            (dict(use_graph=True), 5, (3, 4)), (dict(use_graph=True), 64, (5, "profile"))):
        g = make(nuosc_mod, 11, 37, 3, precision=precision, **kw)
        if zlen:
            g.set_zlen(zlen)
        for n in calls:
            if n == "profile":
                ms = g.profile_stages(2)
                assert ms[0] > 0 and ms[2] > 0 and ms[1] == ms[3] == 0
            else:
                g.step_rk4(n)
        runs.append(g.get_state())
    for r in runs[1:]:
        assert np.array_equal(r, runs[0])


def test_pairs_mixed_with_other_paths(nuosc_mod, oracle_mod):
    """RK4 steps between SSP-RK3 steps, uploads, renormalisation, changed
    physics and calRHS, each of which leaves other records of the state."""
    g = make(nuosc_mod, 9, 21, 2)
    o = oracle_mod.OracleSim(nn=2, cfl=0.4, **geo(9, 21), **PHYS)
    o.fill_init(**INIT)
    g.step_rk4(1)
    o.step(1)
    g.step_srk3(2)
    o.step_srk3(2)
    g.step_rk4(2)
    o.step(2)
    st = g.get_state()
    g.calRHS(st)
    g.set_state(st)
    g.step_rk4(1)
    o.step(1)
    g.set_mu(0.4)
    g.set_pmo(-0.3)
    oracle_mod.lib().orc_set_physics(o._p, 0.4, -0.3, 1)
    g.set_renorm(True)
    g.step_rk4(3)
    o.step(3)
    a, b = g.get_state(), o.get_state()
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))


# open z: nx, nz, refinement, ghost sites, z-segment length (segments that begin
# at the second site or end at the last but one, boxes of three sites)
OPEN_SHAPES = [(1, 3, 1, 2, 1), (1, 4, 4, 2, 3), (1, 40, 2, 3, 7), (2, 3, 2, 2, 2), (3, 5, 1, 2, 1), (5, 33, 3, 2, 0),
               (9, 20, 2, 3, 32), (13, 29, 2, 2, 7)]


@pytest.mark.parametrize("shape", OPEN_SHAPES)
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("scheme", ["rk4", "srk3"])
def test_open_pairs_match_oracle(nuosc_mod, oracle_mod, shape, precision, scheme):
    """A pulse entering through z0, all couplings on.  FP64: 1e-12 per field as
    above.  FP32: besides the 8 roundings a step of the periodic box, the
    extrapolated ghost values (weights 7 and 17 in sum) reach the edge sites'
    stages through the stencil (8/12 and 1/12) times dt/h = 0.4, 2.4 more a
    stage at most: 9 steps x 18 x 2^-24 x 2 = 1.9e-5."""
    nx, nz, nn, gz, zlen = shape
    zc = -nz * H / 2 - 0.3
    init = dict(ipt=0, alpha=0.85, eps0=0.3, sigma=0.5, lnue=0.6, lnueb=0.5)
    g = nuosc_mod.NuOsc(nv=nn, CFL=0.4, gz=gz, bc=nuosc_mod.BC_OPEN_Z, zc=zc, precision=precision, **geo(nx, nz), **PHYS)
    o = oracle_mod.OracleSim(nn=nn, cfl=0.4, gz=gz, bc=1, zc=zc, **geo(nx, nz), **PHYS)
    g.fillInitValue(**init)
    o.fill_init(**init)
    if zlen:
        g.set_zlen(zlen)
    for n in (1, 2, 6):
        (g.step_rk4 if scheme == "rk4" else g.step_srk3)(n)
        (o.step if scheme == "rk4" else o.step_srk3)(n)
    a, b = g.get_state(), o.get_state()
    tol = 1e-12 if precision == 64 else 9 * 18 * 2.0 ** -24 * 2
    for f in range(8):
        assert np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[:4] if f < 4 else b[4:])), f
    assert g.phy_time == pytest.approx(o.phy_time, rel=1e-14)


@pytest.mark.parametrize("precision", [64, 32])
def test_open_pairs_segments_bitwise(nuosc_mod, precision):
    """The state does not depend on the z segments, on graph replay or on how
    the steps are split into calls."""
    runs = []
    for use_graph, zlen, calls in ((True, 0, (7,)), (False, 1, (1, 2, 1, 3)), (True, 5, (3, 4)), (True, 64, (5, 2))):
        g = nuosc_mod.NuOsc(nv=3, CFL=0.4, bc=nuosc_mod.BC_OPEN_Z, zc=-3.0, precision=precision, use_graph=use_graph,
                            **geo(11, 37), **PHYS)
        g.fillInitValue(ipt=0, alpha=0.85, eps0=0.3, sigma=0.5, lnue=0.6, lnueb=0.5)
        if zlen:
            g.set_zlen(zlen)
        for n in calls:
            g.step_rk4(n)
        runs.append(g.get_state())
    for r in runs[1:]:
        assert np.array_equal(r, runs[0])


@pytest.mark.parametrize("nx,nn", [(1, 5), (2, 6), (3, 4), (5, 8), (7, 1)])
@pytest.mark.parametrize("precision", [64, 32])
def test_open_ghost_waves(nuosc_mod, oracle_mod, nx, nn, precision):
    """4 nx ghost sites of 1 to 11 direction chunks, four waves to a block: blocks
    within one site, over several, and a partly filled last one.  Tolerances of
    test_open_pairs_match_oracle, for 3 steps."""
    nz = 9
    zc = -nz * H / 2 - 0.3
    init = dict(ipt=0, alpha=0.85, eps0=0.3, sigma=0.5, lnue=0.6, lnueb=0.5)
    g = nuosc_mod.NuOsc(nv=nn, CFL=0.4, gz=2, bc=nuosc_mod.BC_OPEN_Z, zc=zc, precision=precision, **geo(nx, nz), **PHYS)
    o = oracle_mod.OracleSim(nn=nn, cfl=0.4, gz=2, bc=1, zc=zc, **geo(nx, nz), **PHYS)
    g.fillInitValue(**init)
    o.fill_init(**init)
    g.step_rk4(3)
    o.step(3)
    a, b = g.get_state(), o.get_state()
    tol = 1e-12 if precision == 64 else 3 * 18 * 2.0 ** -24 * 2
    for f in range(8):
        assert np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[:4] if f < 4 else b[4:])), f


@pytest.mark.parametrize("precision", [64, 32])
def test_autotuned_steps_bitwise(nuosc_mod, precision):
    """Steps on tuned segment lengths, on a second handle through the cached
    ones, and on the plan: the same state."""
    runs = []
    for tune in (0, 2, 2):
        g = make(nuosc_mod, 31, 83, 3, precision=precision)
        if tune:
            zlen, ms = g.autotune(tune)
            assert zlen == g.plan()[0] and (ms > 0) == (len(runs) == 1)
        g.step_rk4(3)
        g.step_srk3(1)
        runs.append(g.get_state())
    for r in runs[1:]:
        assert np.array_equal(r, runs[0])


@pytest.mark.parametrize("shape", [(1, 40, 2, 7), (5, 33, 3, 0), (9, 20, 2, 5)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("scheme", ["rk4", "srk3"])
def test_open_renormalised_pairs_match_oracle(nuosc_mod, oracle_mod, shape, precision, scheme):
    """Open z with renormalisation in every step: the new state is renormalised
    after its sums were formed, and its ghost sites follow.  Tolerances of
    test_open_pairs_match_oracle, one more rounding a step."""
    nx, nz, nn, zlen = shape
    zc = -nz * H / 2 - 0.3
    init = dict(ipt=0, alpha=0.85, eps0=0.3, sigma=0.5, lnue=0.6, lnueb=0.5)
    g = nuosc_mod.NuOsc(nv=nn, CFL=0.4, bc=nuosc_mod.BC_OPEN_Z, zc=zc, precision=precision, renorm=True, **geo(nx, nz), **PHYS)
    o = oracle_mod.OracleSim(nn=nn, cfl=0.4, bc=1, zc=zc, renorm=1, **geo(nx, nz), **PHYS)
    g.fillInitValue(**init)
    o.fill_init(**init)
    if zlen:
        g.set_zlen(zlen)
    for n in (1, 2, 6):
        (g.step_rk4 if scheme == "rk4" else g.step_srk3)(n)
        (o.step if scheme == "rk4" else o.step_srk3)(n)
    a, b = g.get_state(), o.get_state()
    tol = 1e-12 if precision == 64 else 9 * 19 * 2.0 ** -24 * 2
    for f in range(8):
        assert np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[:4] if f < 4 else b[4:])), f
