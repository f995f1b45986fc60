"""The pair walks at the edges of their tiles, batches and dispatch rules,
against the oracle after initialization and one time step (1e-12, as the
other parity tests: sums of at most a few thousand FP64 terms in another
order)."""
import os
import sys

import numpy as np
import pytest
from scipy.spatial import cKDTree

import ccake_amd  # noqa: F401
from ccake_amd import batching, config
from parity_metrics import DERIVS, STATE
from test_gpu_parity import Pair, compare, ints_equal
from test_milne3 import DERIVS3, STATE3, Pair3, compare3

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "hostemu"))

pytestmark = pytest.mark.gpu


def cloud(n, half, seed=3):
    """n jittered points with flow, charges and a smooth energy profile."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(np.sqrt(n)))
    g = np.linspace(-half, half, m) if m > 1 else np.zeros(1)
    x, y = (a.ravel()[:n] + rng.uniform(-0.01, 0.01, n) for a in np.meshgrid(g, g))
    e = (5.0 + 20.0 * np.exp(-(x * x + y * y) / 8.0)) / config.HBARC_GEVFM
    f = 0.02 * np.cos(x + 0.3 * y)
    return dict(x=x, y=y, e=e, ux=0.1 * x / (half + 1), uy=-0.05 * y / (half + 1), rhoB=f * e, rhoS=0.5 * f * e,
                rhoQ=-f * e)


# one particle; a tile and its neighbours; the last size of the kept summation
# order (8,192 with a hypersurface) and the first beyond it; 40 cells per
# radius: more than 64 key rows within reach of a tile
@pytest.mark.parametrize("n,half,cells,particlization,shear", [
    (1, 0.5, 4, 0, 1), (63, 0.4, 4, 0, 1), (64, 0.4, 1, 1, 1), (65, 0.4, 4, 0, 0), (300, 0.5, 40, 0, 1),
    (300, 0.5, 40, 1, 1), (8192, 4.5, 4, 1, 1), (8193, 4.5, 4, 1, 1), (8192, 4.5, 4, 0, 0)])
def test_walk_edges(dev, orc, n, half, cells, particlization, shear):
    eta = 0.08 if shear else 0.0
    cfg = config.base_params(t0=0.6, dt=0.01, particlization=particlization, eta_mode=config.ETA_CONSTANT,
                             constant_eta_over_s=eta, cells_per_rc=cells, x_subcells=4)
    p = Pair(dev, orc, cfg, cloud(n, half))
    p.initialize()
    ints_equal(p.g, p.o, "BTRACK")
    p.step(1)
    ints_equal(p.g, p.o, "BTRACK")
    compare(p.g, p.o, STATE + DERIVS, what=f"n={n} cells={cells} surface={particlization} shear={shear}")
    p.close()


# 3+1D: tiles of 16 targets; one particle, a tile and its neighbours, several
# cell rows in a tile (1 and 8 cells per radius), 24 cells per radius (more than
# 64 cell rows within reach), each number of waves per tile, both kernels, with
# and without the shear sums
@pytest.mark.parametrize("n,cells,waves,factorized,shear", [
    (1, 2, 4, 0, 1), (15, 2, 2, 0, 1), (16, 2, 1, 1, 1), (17, 1, 4, 0, 0), (70, 8, 4, 1, 1), (343, 24, 4, 0, 1),
    (1000, 2, 1, 0, 1), (1000, 2, 2, 1, 0), (1000, 2, 4, 0, 0), (1331, 3, 4, 1, 1)])
def test_milne_walk_edges(dev, orc, n, cells, waves, factorized, shear):
    m = int(np.ceil(round(n ** (1 / 3), 9)))
    rng = np.random.default_rng(n)
    g = (np.arange(m) - 0.5 * (m - 1)) * 0.17
    x, y, eta = (a.ravel()[:n] + rng.uniform(-0.02, 0.02, n) for a in np.meshgrid(g, g, g))
    e = (5.0 + 20.0 * np.exp(-(x * x + y * y + eta * eta) / 2.0)) / config.HBARC_GEVFM
    f = 0.02 * np.cos(x + 0.3 * y)
    d = dict(x=x, y=y, eta=eta, e=e, ux=0.1 * x, uy=-0.05 * y, ueta=0.03 * eta, rhoB=f * e, rhoS=0.5 * f * e, rhoQ=-f * e)
    cfg = config.base_params(dim=3, hEta=0.2, factorized_kernel=factorized, t0=0.6, dt=0.01, particlization=0,
                             eta_mode=config.ETA_CONSTANT, constant_eta_over_s=0.08 if shear else 0.0,
                             cells_per_rc=cells, x_subcells=4)
    p = Pair3(dev, orc, cfg, d)
    p.g.nslices(waves)
    p.g.initialize()
    assert p.o.initialize() == 0
    ints_equal(p.g, p.o, "BTRACK")
    p.g.advance_timestep(cfg["dt"], 2)
    assert p.o.advance_timestep(cfg["dt"], 2) == 0
    ints_equal(p.g, p.o, "BTRACK")
    compare3(p.g, p.o, STATE3 + DERIVS3, what=f"n={n} cells={cells} waves={waves} factorized={factorized} shear={shear}")
    p.close()


# the cell sort: radix blocks of 1,024 (one, a partial one, 17 over the scan's 16
# waves, the most its one workgroup takes and one more) and runs of empty cells
@pytest.mark.parametrize("n", [1, 1023, 1025, 16385, 17409, 262144, 262145])
def test_sort_and_counts(dev, n):
    rng = np.random.default_rng(n)
    half = max(1.0, 0.12 * np.sqrt(n))
    r = rng.uniform(-half, half, (n, 2))
    r[r[:, 0] > 0.0, 0] += 3.0 * half                 # two clouds with empty cells between
    cfg = config.base_params(t0=0.6, dt=0.01, particlization=0, cells_per_rc=1, x_subcells=1)
    eos = ccake_amd.Eos(dev, 0, 0.75)
    ev = ccake_amd.Event(dev, eos, cfg, n)
    ev.upload("CCAKE_F_X", r[:, 0])
    ev.upload("CCAKE_F_Y", r[:, 1])
    ev.build_neighbors()
    want = cKDTree(r).query_ball_point(r, 2.0 * cfg["hT"], return_length=True) - 1
    assert np.array_equal(ev.download_int("CCAKE_I_BTRACK"), want)
    ev.close()
    eos.close()


# single-precision weights (relative error 5.2e-8 at most) with each number of
# waves per tile and with single-wave slices: a smoothed field is a sum of
# positive terms, so its error stays below that; the gradients cancel
@pytest.mark.parametrize("slices", [8, 4, 2])
@pytest.mark.parametrize("shear", [0, 1])
def test_single_precision_weights(dev, slices, shear):
    d = cloud(2500, 2.5)
    cfg = config.base_params(t0=0.6, dt=0.01, particlization=0, eta_mode=config.ETA_CONSTANT,
                             constant_eta_over_s=0.08 if shear else 0.0, cells_per_rc=4, x_subcells=4)
    eos = ccake_amd.Eos(dev, 0, 0.75)
    got = []
    for pp in (0, 1):
        ev = ccake_amd.Event(dev, eos, dict(cfg, pair_precision=pp), len(d["x"]))
        ccake_amd.load_event(ev, d)
        ev.nslices(slices)
        ev.initialize()
        ev.get_time_derivatives()
        got.append({f: ev.download(ccake_amd.FIELDS["CCAKE_F_" + f]) for f in ("SIGMA_LAB", "S", "GRADP0", "GRADE0", "GRADV0")})
        got[-1]["BTRACK"] = ev.download_int("CCAKE_I_BTRACK")
        ev.close()
    eos.close()
    assert np.array_equal(got[0].pop("BTRACK"), got[1].pop("BTRACK"))
    for f, a in got[0].items():
        err = np.max(np.abs(got[1][f] - a)) / np.max(np.abs(a))
        assert 0.0 < err <= (5.2e-8 if f == "SIGMA_LAB" else 2e-6), (f, err)


# above 2,000 neighbours r comes from the square root instruction (2.7e-8 at most,
# at twice which a pair's weight can be off) and the errors' mean is taken out: of
# -3.3e-9 in r, so 6.6e-9 in a density, no more than 2e-9 is left
def test_single_precision_weights_of_many_neighbours(dev):
    d = cloud(66000, 2.4)
    cfg = config.base_params(t0=0.6, dt=0.01, particlization=0, eta_mode=config.ETA_CONSTANT, constant_eta_over_s=0.08,
                             cells_per_rc=4, x_subcells=4)
    eos = ccake_amd.Eos(dev, 0, 0.75)
    got = []
    for pp in (0, 1):
        ev = ccake_amd.Event(dev, eos, dict(cfg, pair_precision=pp), len(d["x"]))
        ccake_amd.load_event(ev, d)
        ev.initialize()
        ev.get_time_derivatives()
        got.append({f: ev.download(ccake_amd.FIELDS["CCAKE_F_" + f]) for f in ("SIGMA_LAB", "S", "GRADP0", "GRADE0", "GRADV0")})
        got[-1]["BTRACK"] = ev.download_int("CCAKE_I_BTRACK")
        ev.close()
    eos.close()
    assert np.array_equal(got[0]["BTRACK"], got[1].pop("BTRACK")) and np.mean(got[0].pop("BTRACK")) >= 2000
    for f, a in got[0].items():
        err = np.max(np.abs(got[1][f] - a)) / np.max(np.abs(a))
        print(f, err)
        assert 0.0 < err <= (5.4e-8 if f in ("SIGMA_LAB", "S") else 2e-6), (f, err)
    assert abs(np.mean(got[1]["SIGMA_LAB"] / got[0]["SIGMA_LAB"] - 1.0)) <= 2e-9


# An event for which one slice of partial sums is set aside (262,144 particles
# are 4,096 tiles: whole rounds of the chip's SIMDs) runs its tiles of 8 waves in
# no more device memory: the diffusion pass, which stores every slice's sums,
# then takes one slice, and a slice count whose sums would not fit is refused.
# The autotuner takes what it is given as far as that goes.
def test_partial_sums_fit(dev, monkeypatch):
    n = 262144
    m = 512
    x, y = (a.ravel() for a in np.meshgrid(np.arange(m) * 0.1, np.arange(m) * 0.1))
    cfg = config.base_params(t0=0.6, dt=0.01, particlization=0, cells_per_rc=4, x_subcells=4, using_diffusion=1,
                             kappa_over_T2=[0.1, 0, 0, 0, 0.1, 0, 0, 0, 0.1], diffusion_regulator=1)
    f = 0.02 * np.cos(x + 0.3 * y)
    e = 10.0 + np.cos(0.1 * x) + np.cos(0.1 * y)
    d = dict(x=x, y=y, e=e, ux=0.05 * np.sin(0.2 * x), uy=0.05 * np.sin(0.3 * y), rhoB=f * e, rhoS=0.5 * f * e, rhoQ=-f * e)
    eos = ccake_amd.Eos(dev, 0, 0.75)
    a = []
    for one in (False, True):
        if one:                                  # one wave per tile
            monkeypatch.setenv("CCAKE_PAIR_SLICES", "1")
        ev = ccake_amd.Event(dev, eos, cfg, n)
        ccake_amd.load_event(ev, d)
        assert ev.nslices() == 1
        for s in (2, 3, 4, 16):
            with pytest.raises(RuntimeError):
                ev.nslices(s)
        ev.nslices(1)
        ev.initialize()
        ev.get_time_derivatives()
        a.append([ev.download(ccake_amd.FIELDS["CCAKE_F_" + f]) for f in ("GRADP0", "GRADV0", "DEXT_Q0")])
        ev.close()
    monkeypatch.delenv("CCAKE_PAIR_SLICES")
    for u, v in zip(*a):
        assert np.max(np.abs(u - v)) <= 1e-12 * np.max(np.abs(u)) > 0.0
    assert any(np.any(u != v) for u, v in zip(*a))      # the tile's eight waves ran, then one
    for slices in ((1, 2, 4), (4, 8)):
        t = batching.autotune(dev, eos, dict(cfg, using_diffusion=0, pair_precision=1), [d], cells_per_rc=(4,), slices=slices, steps=1)
        assert t["slices"] == 1
    eos.close()


# A recorded batch above the kept order's 8,192 particles whose second event ends,
# which leaves less than that: the first event goes on in the form it began with,
# so as it does beside an event that has not ended.  (Its lines of 128 particles
# are whole tiles, each in a cell row of its own, sorted anew in every stage, so
# that its tiles and their segments are the same either way.)
def test_a_batch_keeps_its_form_as_events_end(dev, monkeypatch):
    def lines(nx, ny, gev):
        x, y = (a.ravel() for a in np.meshgrid((np.arange(nx) - 0.5 * nx) * 0.05, np.arange(ny) * 0.45))
        y[y > 0.0] += 0.075                          # the first line is the box's edge, the others mid-cell
        e = gev * (1.0 + 0.2 * np.cos(x) * np.cos(y)) / config.HBARC_GEVFM
        z = np.zeros_like(x)
        return dict(x=x, y=y, e=e, ux=0.1 * np.sin(x), uy=0.1 * np.sin(y), rhoB=0.02 * e, rhoS=z, rhoQ=z)

    monkeypatch.setenv("CCAKE_SORT_SKIN", "0")
    T = 150.0 / config.HBARC_MEVFM
    eos = ccake_amd.Eos(dev, 0, T)
    cfg = dict(config.lumpy_params(dt=0.002), particlization=1, e_freeze=eos.efreeze(T), cells_per_rc=4, x_subcells=8)
    got = []
    for gev in (0.2, 20.0):                          # the second event: cold, or as hot as the first
        ics = [lines(128, 50, 20.0), lines(128, 20, gev)]
        b = ccake_amd.Batch(dev, eos, cfg, [6400, 2560])
        ccake_amd.load_event(b, ccake_amd.concat_ics(ics))
        b.initialize()
        for _ in range(12):
            live = b.batch_continue_evolution(max_tau=30.0)
            b.advance_timestep(cfg["dt"], 2)
        got.append([bool(q) for q in live])
        got.append(np.stack([b.download(ccake_amd.FIELDS["CCAKE_F_" + f])[:6400] for f in ("UX", "UY", "E", "GRADP0", "GRADV0")]))
        b.close()
    eos.close()
    assert got[0] == [True, False] and got[2] == [True, True]
    print("differ by", np.max(np.abs(got[1] - got[3]), axis=1))
    assert np.array_equal(got[1], got[3])


# NaN or infinity in one particle stays within its range (0 times either is NaN):
# the walks of the tiles that meet it are done again; 3+1D sums are then formed
# outside the matrix cores, so in another order (a few hundred terms: 1e-13), and
# without the pairs just out of range that single-precision weights (error 5.2e-8)
# give the square of that at most, 3e-15 of a whole weight
@pytest.mark.parametrize("case,slices", [("small", 0), ("small", 4), ("small", 2), ("recorded", 0), ("mixed", 0),
                                         ("diffusion", 0), ("milne", 0), ("milne_fact", 1)])
def test_a_non_finite_value_stays_within_its_range(dev, case, slices):
    from run_nonfinite import check
    assert check(dev, case, slices, stepped=False, tol=1e-13 if case in ("mixed", "milne", "milne_fact") else 0.0)
