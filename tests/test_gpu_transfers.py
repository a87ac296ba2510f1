"""Field transfers through pinned slots: states of one piece, of a few and of
many slots with a ragged last one come back bit for bit, from several threads
at once, and slices agree with the fields they are made of."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 0.125


def make(N, nx, nz, nn, **kw):
    g = N.NuOsc(nv=nn, x0=-nx * H / 2, x1=nx * H / 2, z0=-nz * H / 2, z1=nz * H / 2, dx=H, dz=H, **kw)
    g.fillInitValue(ipt=5, alpha=0.9, eps0=0.1, sigma=1.0, lnue=0.6, lnueb=0.5, seed=5)
    return g


# 8 (or 18) fields of 12 .. 1.0e6 values: one slot holds 524288
@pytest.mark.parametrize("nx,nz,nn,nflavor", [(1, 1, 1, 2), (3, 5, 2, 3), (16, 33, 4, 2), (41, 39, 5, 3), (67, 61, 5, 2)])
@pytest.mark.parametrize("precision", [64, 32])
def test_round_trip(nuosc_mod, nx, nz, nn, nflavor, precision):
    g = make(nuosc_mod, nx, nz, nn, precision=precision, nflavor=nflavor)
    rng = np.random.default_rng(nx)
    a = rng.normal(size=(g.nvar, *g.shape)).astype(np.float32 if precision == 32 else np.float64).astype(np.float64)
    g.set_state(a)
    assert np.array_equal(g.get_state(), a)
    for f in (0, g.nvar - 1):
        assert np.array_equal(g.get_field(f), a[f])
    p3 = g.p3_slice(np.arange(g.nx), np.arange(g.nv))
    assert np.array_equal(p3, (a[0] - a[1]) * (1.0 / g.g0()[0]))
    with pytest.raises(nuosc_mod.NuOscError):
        g.get_field(g.nvar)


def test_threads(nuosc_mod):
    """Four handles transfer at once (more slots asked for than there are)."""
    sims = [make(nuosc_mod, 40 + k, 50, 5) for k in range(4)]
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(4):
            a = rng.normal(size=(8, *sims[k].shape))
            sims[k].set_state(a)
            if not np.array_equal(sims[k].get_state(), a):
                bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_more_transfers_than_slots(nuosc_mod):
    """Four handles with states of 57 MB, eight slots each of the sixteen there
    are: the later ones wait for a slot."""
    sims = [make(nuosc_mod, 60, 60 + k, 5) for k in range(4)]
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(3):
            a = rng.normal(size=(8, *sims[k].shape))
            assert a.nbytes >= 32 << 20
            sims[k].set_state(a)
            if not np.array_equal(sims[k].get_state(), a):
                bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
