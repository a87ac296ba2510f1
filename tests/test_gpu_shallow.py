"""Boxes that are shallow in z, and those of 12 directions, step stage by stage
where that is faster than stage pairs: the route on both sides of the line, and
its results against the oracle, mixed with the other scheme's route, in batches
and through uploads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 0.125
INIT = dict(ipt=5, alpha=0.85, eps0=0.1, sigma=1.0, lnue=0.6, lnueb=0.5, seed=77)
PHYS = dict(ko=0.1, mu=1.3, pmo=0.7)


def geo(nx, nz):
    return dict(x0=-nx * H / 2, x1=nx * H / 2, z0=-nz * H / 2, z1=nz * H / 2, dx=H, dz=H)


def make(N, nx, nz, nn, precision, **kw):
    g = N.NuOsc(nv=nn, CFL=0.4, precision=precision, **geo(nx, nz), **PHYS, **kw)
    g.fillInitValue(**INIT)
    return g


# nx, nz, nn, precision, open z, in pairs
@pytest.mark.parametrize("nx,nz,nn,precision,open_z,pairs", [
    (1, 1, 2, 64, False, True), (700, 1, 2, 64, False, True), (701, 5, 2, 64, False, False), (701, 6, 2, 64, False, True),
    (701, 3, 2, 64, True, True), (234, 7, 4, 32, False, False), (234, 8, 4, 32, True, True), (501, 11, 1, 64, False, False),
    (501, 12, 1, 64, False, True), (501, 39, 1, 64, True, False), (500, 40, 1, 32, False, True), (500, 41, 1, 32, True, False)])
def test_route(nuosc_mod, nx, nz, nn, precision, open_z, pairs):
    kw = dict(bc=nuosc_mod.BC_OPEN_Z) if open_z else {}
    g = make(nuosc_mod, nx, nz, nn, precision, **kw)
    ms = g.profile_stages(1)
    assert (ms[1] == 0 and ms[3] == 0) == pairs and ms[0] > 0 and ms[2] > 0
    g.close()


@pytest.mark.parametrize("nx,nz,nn", [(701, 1, 2), (701, 3, 2), (352, 4, 3), (503, 5, 1), (501, 42, 1)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("open_z", [False, True])
def test_matches_oracle(nuosc_mod, oracle_mod, nx, nz, nn, precision, open_z):
    """RK4 and SSP-RK3 steps in turn, an upload between.  FP64: 1e-12 per field
    over 9 steps (a few roundings each).  FP32: at most 18 roundings of 2^-24 a
    step (8 stores and stage updates, 10 for the extrapolated ghost values), grown
    by less than 2: 9 x 18 x 2^-24 x 2."""
    if open_z and nz < 3:
        pytest.skip("the open boundary needs three sites")
    kw, okw, init = {}, {}, INIT
    if open_z:
        init = dict(ipt=0, alpha=0.85, eps0=0.3, sigma=0.5, lnue=0.6, lnueb=0.5)
        kw, okw = dict(bc=nuosc_mod.BC_OPEN_Z, zc=-nz * H / 2 - 0.3), dict(bc=1, zc=-nz * H / 2 - 0.3)
    g = nuosc_mod.NuOsc(nv=nn, CFL=0.4, precision=precision, **geo(nx, nz), **PHYS, **kw)
    o = oracle_mod.OracleSim(nn=nn, cfl=0.4, **geo(nx, nz), **PHYS, **okw)
    g.fillInitValue(**init)
    o.fill_init(**init)
    for n, srk in ((1, False), (2, True), (2, False), (1, True), (3, False)):
        (g.step_srk3 if srk else g.step_rk4)(n)
        (o.step_srk3 if srk else o.step)(n)
        if n == 1:
            g.set_state(g.get_state())
    a, b = g.get_state(), o.get_state()
    tol = 1e-12 if precision == 64 else 9 * 18 * 2.0 ** -24 * 2
    for f in range(8):
        assert np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[:4] if f < 4 else b[4:])), f


@pytest.mark.parametrize("precision", [64, 32])
def test_schemes_of_different_routes(nuosc_mod, oracle_mod, precision):
    """703 x 6 x 42 in FP64 and 703 x 10 x 42 in FP32 step RK4 in pairs and SSP-RK3
    stage by stage: each leaves records the other does not use."""
    nz = {64: 6, 32: 10}[precision]
    g = make(nuosc_mod, 703, nz, 2, precision)
    o = oracle_mod.OracleSim(nn=2, cfl=0.4, **geo(703, nz), **PHYS)
    o.fill_init(**INIT)
    for n, srk in ((1, False), (1, True), (1, True), (2, False), (1, False), (3, True)):
        (g.step_srk3 if srk else g.step_rk4)(n)
        (o.step_srk3 if srk else o.step)(n)
    g.renormalize()
    o.renormalize()
    g.step_srk3(1)
    o.step_srk3(1)
    a, b = g.get_state(), o.get_state()
    tol = 1e-12 if precision == 64 else 10 * 18 * 2.0 ** -24 * 2
    for f in range(8):
        assert np.max(np.abs(a[f] - b[f])) <= tol * np.max(np.abs(b[:4] if f < 4 else b[4:])), f


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("shapes", [[(703, 2, 2), (360, 4, 3), (505, 1, 1)], [(703, 2, 2), (12, 20, 2), (1, 30, 1), (360, 3, 3)]])
def test_batch_equals_alone(nuosc_mod, precision, persistent, shapes):
    """Batches of shallow runs, and of shallow and deep ones, over odd and even
    numbers of steps, with members stepped alone in between."""
    N = nuosc_mod
    alone = [make(N, *s, precision) for s in shapes]
    mixed = [make(N, *s, precision) for s in shapes]
    b = N.Batch(precision=precision)
    for g in mixed:
        b.add(g)
    if persistent:
        b.set_launch(N.BATCH_PERSISTENT)
    for n in (3, 2):
        b.step(n)
        for g in alone:
            g.step_rk4(n)
    for g in (alone[0], mixed[0], alone[1], mixed[1]):
        g.step_srk3(1)
    before = [g.get_state() for g in mixed]
    zl, ms = b.autotune(1)
    assert ms > 0
    for g, s in zip(mixed, before):
        assert np.array_equal(g.get_state(), s)
    b.step(2)
    for a, m in zip(alone, mixed):
        a.step_rk4(2)
        assert np.array_equal(a.get_state(), m.get_state())
    b.close()
