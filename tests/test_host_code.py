"""The host code of the handles and batches on a stand-in HIP runtime
(fake_hip.cpp): no GPU, every launch and allocation can be made to fail, and a
kernel that is given another state's records is counted."""
import ctypes as C

import numpy as np
import pytest

import fake_hip
import nuosc_amd as N

H = 0.125


@pytest.fixture(scope="session")
def fake_lib(tmp_path_factory):
    return fake_hip.load(fake_hip.build(tmp_path_factory.mktemp("fake")))


@pytest.fixture
def fake(fake_lib, monkeypatch):
    monkeypatch.setattr(N, "_lib", fake_lib)
    fake_lib.fake_reset()
    yield fake_lib
    assert fake_lib.fake_mistakes() == 0
    assert fake_lib.fake_device_bytes() == 0 and fake_lib.fake_graphs() == 0


def make(nx=9, nz=40, nn=2, seed=7, **kw):
    g = N.NuOsc(nv=nn, x0=-nx * H / 2, x1=nx * H / 2, z0=-nz * H / 2, z1=nz * H / 2, dx=H, dz=H, **kw)
    g.fillInitValue(ipt=5, seed=seed)
    return g


def value(g):
    return g.get_field(0).flat[0]


@pytest.mark.parametrize("kw", [dict(), dict(precision=32), dict(nx=701, nz=2), dict(bc=N.BC_OPEN_Z), dict(nflavor=3),
                                dict(adv=N.ADV_CFD2), dict(renorm=True), dict(use_graph=False)])
def test_steps(fake, kw):
    """The stand-in itself: every route steps, in any order of the schemes."""
    with make(**kw) as g:
        g.step_rk4(3)
        g.step_srk3(2)
        g.step_rk4(2)
        g.set_state(g.get_state())
        g.step_srk3(1)
        assert value(g) % 1000 == 7 + 8


@pytest.mark.parametrize("kw", [dict(), dict(precision=32), dict(nx=701, nz=2), dict(bc=N.BC_OPEN_Z), dict(nflavor=3),
                                dict(renorm=True)])
@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("scheme", ["step_rk4", "step_srk3", "profile_stages"])
def test_failed_launch_in_a_step(fake, kw, use_graph, scheme):
    """Whichever launch of a step fails, the call says so and the next step does
    not take the records the failed one left."""
    with make(use_graph=use_graph, **kw) as g:
        g.step_rk4(1)
        pairs = g.plan()[0] == 15 and "nflavor" not in kw
        for n in range(1, 15):
            before, t = value(g), g.phy_time
            fake.fake_fail(b"launch", n)
            try:
                getattr(g, scheme)(1)
            except N.NuOscError:
                assert g.phy_time == t
                if pairs:   # (the other routes write the state in place)
                    assert value(g) == before
            fake.fake_fail(b"launch", 1 << 30)
            g.step_srk3(1)
            g.step_rk4(1)
            assert fake.fake_mistakes() == 0, n


@pytest.mark.parametrize("what", ["analysis", "pair_sums", "renorm"])
def test_failed_refresh(fake, what):
    """fillInitValue and renormalize that fail half-way leave no records of the
    state before."""
    with make() as g:
        g.step_rk4(1)
        fake.fake_fail(what.encode(), 1)
        with pytest.raises(N.NuOscError):
            if what == "renorm":
                g.renormalize()
            else:
                g.fillInitValue(ipt=5, seed=50)
        g.step_rk4(1)
        assert value(g) == (9 if what == "renorm" else 51)


@pytest.mark.parametrize("what", ["launch", "hipGraphLaunch"])
def test_failed_batch_step(fake, what):
    sims = [make(seed=10), make(nx=701, nz=2, seed=20)]
    b = N.Batch()
    for g in sims:
        b.add(g)
    b.step(1)
    for n in range(1, 10):
        before = [value(g) for g in sims]
        fake.fake_fail(what.encode(), n)
        sims[0].set_mu(1.0 + n)   # (a new capture)
        try:
            b.step(1)
        except N.NuOscError:
            assert [value(g) for g in sims] == before
        fake.fake_fail(what.encode(), 1 << 30)
        for g in sims:
            g.step_rk4(1)
        b.step(2)
        assert fake.fake_mistakes() == 0, n
    b.close()
    for g in sims:
        g.close()


def test_failed_instantiation(fake):
    """A captured step that cannot be instantiated is given back (the fixture
    counts graphs), and the next call captures it again."""
    with make() as g:
        b = N.Batch()
        for n in range(2):
            fake.fake_fail(b"hipGraphInstantiate", 1)
            with pytest.raises(N.NuOscError):
                g.step_rk4(1)
        g.step_rk4(3)
        b.add(g)
        for n in range(2):
            fake.fake_fail(b"hipGraphInstantiate", 1)
            with pytest.raises(N.NuOscError):
                b.step(1)
        b.step(2)
        assert value(g) == 7 + 5
        b.close()


def test_transfer_with_another_device_current(fake):
    """A handle on device 1 moves fields whichever device its caller has current."""
    with make(device=1) as g:
        for current in (0, 1):
            fake.hipSetDevice(current)
            a = np.full((8, *g.shape), 3.0 + current)
            g.set_state(a)
            assert np.array_equal(g.get_state(), a)
            g.analysis()
    fake.hipSetDevice(0)
    with N.NuOsc(nv=2, device=1) as g:
        fake.hipSetDevice(0)
        g.fillInitValue(ipt=5, seed=4)   # the first slot
        assert value(g) == 4
        dev = C.c_int()
        fake.hipGetDevice(C.byref(dev))
        assert dev.value == 0


def test_fewer_slots_than_asked_for(fake):
    """A transfer that gets some of its slots goes on with those."""
    with make(nx=128, nz=128) as g:   # 44 MB: eight slots
        a = np.full((8, *g.shape), 3.0)
        for what in (b"hipHostMalloc", b"hipEventCreate"):
            fake.fake_fail(what, 2)
            g.set_state(a)
            assert np.array_equal(g.get_state(), a)


def test_no_slot_leaves_nothing_queued(fake):
    """Calls that fail for want of a slot return once the copies that they queued
    from their own memory are done."""
    with N.NuOsc(nv=2) as g:
        for call in (lambda: g.p3_slice([0, 1], [0, 2]), lambda: g.fillInitValue(ipt=0)):
            fake.fake_fail(b"hipHostMalloc", 1)
            with pytest.raises(N.NuOscError) as e:
                call()
            assert e.value.code == N.NUOSC_ENOMEM
            assert fake.fake_pending() == 0


def test_slot_events_release_to_the_system(fake):
    """hipEventReleaseToSystem (0x80000000): the fence that makes a kernel's writes
    to a slot visible to the host."""
    with make():
        assert fake.fake_event_flags() & 0x80000000


# best lengths of the two pair kernels; planned: 15 and 25
@pytest.mark.parametrize("nx,best", [(100, (15, 25)), (101, (64, 16)), (102, (15, 32)), (103, (8, 25)), (104, (40, 33))])
def test_autotune_takes_each_kernels_best(fake, nx, best):
    """The tuner never leaves a kernel slower than it was planned, gives each its
    own length, and a second handle of the grid gets the same from the cache."""
    zl = [8, 16, 32, 64, 128, 256]
    want = [min([p, *zl], key=lambda z: abs(z - b)) for p, b in zip((15, 25), best)]
    for pair in (1, 2):
        fake.fake_best_zlen(pair, best[pair - 1])
    for handle in range(2):
        with make(nx=nx, nz=300) as g:
            got, ms = g.autotune(1)
            assert (ms > 0) == (handle == 0) and got == want[0] == g.plan()[0]
            g.step_rk4(1)
            assert [fake.fake_last_zlen(p) for p in (1, 2)] == want
            g.step_srk3(1)
            assert [fake.fake_last_zlen(p) for p in (3, 4)] == [15, 20]


def test_autotune_tries_the_length_in_force(fake):
    fake.fake_best_zlen(1, 47)
    fake.fake_best_zlen(2, 47)
    with make(nx=110, nz=300) as g:
        g.set_zlen(47)
        assert g.autotune(1)[0] == 47


# best lengths of the two pair kernels (pair 2 the steeper), length after tuning; planned: 24
@pytest.mark.parametrize("best,want", [((24, 24), 24), ((16, 64), 64), ((128, 128), 128), ((30, 20), 24)])
def test_batch_autotune_times_both_pairs(fake, best, want):
    """The batch is left on the length that is fastest for both kernels together,
    the planned one included."""
    for pair in (1, 2):
        fake.fake_best_zlen(pair, best[pair - 1])
    sims = [make(nx=20 + k, nz=300, seed=k) for k in range(2)]
    b = N.Batch()
    for g in sims:
        b.add(g)
    zlen, ms = b.autotune(1)
    assert zlen in (16, 32, 64, 128, 256) and ms > 0
    b.step(3)
    assert [fake.fake_last_zlen(p) for p in (1, 2)] == [want, want]
    assert [value(g) for g in sims] == [3, 4]
    b.close()
    for g in sims:
        g.close()


def test_batch_members_own_plans(fake):
    """set_zlen(0): each member's own lengths, one for each kernel."""
    with make(nz=300) as g:
        b = N.Batch()
        b.add(g)
        b.set_zlen(0)
        b.step(1)
        assert [fake.fake_last_zlen(p) for p in (1, 2)] == [15, 25]
        b.close()


@pytest.mark.parametrize("kw,copies", [(dict(), 3), (dict(precision=32), 4), (dict(nx=701, nz=2), 4), (dict(nflavor=3), 4),
                                       (dict(adv=N.ADV_CFD2), 4), (dict(bc=N.BC_OPEN_Z), 3), (dict(nx=701, nz=6), 3)])
def test_state_copies(fake, kw, copies):
    """FP64 stage pairs hold three copies of the state, the others four; the
    estimate says so too."""
    with make(**kw) as g:
        es, fields = g.precision // 8, g.nvar
        nvp = -(-g.nv * es // 128) * 128 // es
        copy = (g.nx + 7) * (g.nz + (4 if "bc" in kw else 0)) * fields * nvp * es
        assert copies * copy < g.device_bytes() < (copies + 0.5) * copy
        est = N.estimate_device_bytes(nv=2, x0=-g.nx * H / 2, x1=g.nx * H / 2, z0=-g.nz * H / 2, z1=g.nz * H / 2, dx=H,
                                      dz=H, **kw)
        assert g.device_bytes() <= est < g.device_bytes() + (1 << 20)
