"""A non-finite value in one particle (test infrastructure): it may reach the
particles within the cutoff of the one that holds it, in their pair sums, and
no other.  Two lumpy events in a batch, or one 3+1D event, are evaluated with
and without the value; every particle out of its range must keep its fields
bit for bit.  Where the value leaves its holder without an EoS solution (whose
gradient record then stays as it was), the particles of its own event out of
its range must stay finite, and so after a time step with a velocity that is
not finite, whose second stage has a position that is not: that particle is in
range of none.  Prints "OK".

Usage (through tests/hostemu/emu.sh): run_nonfinite.py CASE [SLICES]
CASE: small, recorded, mixed, diffusion, milne or milne_fact.
"""
from __future__ import annotations

import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

import ccake_amd  # noqa: E402
from ccake_amd import config, ic  # noqa: E402

F = ccake_amd.FIELDS
OUT = [("SIGMA_LAB", 0), ("S", 0), ("RHOB", 0), ("GRADP0", 0), ("GRADP0", 1), ("GRADE0", 0), ("GRADBULK0", 0),
       ("GRADBULK0", 1), ("GRADV0", 0), ("GRADV0", 1), ("GRADV0", 3), ("GRADSHEAR0", 0), ("DIVSHEAR0", 1), ("DUDT0", 0)]


def evaluate(dev, eos, cfg, d, counts, slices, bad, step=False):
    """The fields after one derivative evaluation, or one time step, `bad` =
    (column, particle, value) set after the initialization."""
    if counts is None:
        ev = ccake_amd.Event(dev, eos, cfg, len(d["x"]))
    else:
        ev = ccake_amd.Batch(dev, eos, cfg, counts)
    if slices:
        ev.nslices(slices)
    ccake_amd.load_event(ev, d)
    if cfg.get("using_diffusion"):
        for k in range(12):
            ev.upload(F["CCAKE_F_Q0"] + k, 0.0)
    ev.initialize()
    if bad:
        col, i, v = bad
        a = ev.download(F["CCAKE_F_" + col])
        a[i] = v
        ev.upload(F["CCAKE_F_" + col], a)
    try:
        if step:
            ev.advance_timestep(cfg["dt"], 2)
        else:
            ev.get_time_derivatives()
    except ccake_amd.CcakeError as e:          # the particle's own state may have no EoS solution
        print("  reported:", e, flush=True)
    out = OUT + [("DUDT0", 1)]
    if cfg.get("dim") == 3:
        out = out + [("GRADP0", 2), ("GRADV0", 8), ("DUDT0", 2)]
    if cfg.get("using_diffusion"):
        out = out + [("DEXT_Q0", k) for k in range(2)]
    r = {f: ev.download(F["CCAKE_F_" + f[0]] + f[1]) for f in out}
    r["BTRACK"] = ev.download_int("CCAKE_I_BTRACK").astype(float)
    ev.close()
    return r


def check(dev, case, slices, stepped=True, tol=0.0):
    """Whether every value tried stays in its range (fields out of it within
    tol of their largest magnitude, bit for bit by default)."""
    eos = ccake_amd.Eos(dev, 0, 150.0 / config.HBARC_MEVFM)
    milne = case.startswith("milne")
    if milne:
        rng = np.random.default_rng(5)
        g = np.arange(-2.5, 3.0) * 0.17
        x, y, eta = (a.ravel() + rng.uniform(-0.02, 0.02, a.size) for a in np.meshgrid(np.arange(-11.5, 12.0) * 0.17, g, g))
        e = (5.0 + 20.0 * np.exp(-(x * x + y * y + eta * eta) / 2.0)) / config.HBARC_GEVFM
        f = 0.02 * np.cos(x + 0.3 * y)
        d = dict(x=x, y=y, eta=eta, e=e, ux=0.1 * x, uy=-0.05 * y, ueta=0.03 * eta, rhoB=f * e, rhoS=0.5 * f * e,
                 rhoQ=-f * e)
        cfg = config.base_params(dim=3, hEta=0.2, factorized_kernel=int(case == "milne_fact"), t0=0.6, dt=0.01,
                                 particlization=0, eta_mode=config.ETA_CONSTANT, constant_eta_over_s=0.08, cells_per_rc=2)
        counts, n0 = None, len(x)
        r = np.stack([x, y, eta])
    else:
        # short key rows, so that a tile holds many and the one across the events' border holds both
        ics = [ic.lumpy(seed=0xCCA4E001 + k, spacing=0.2, half_width=hw, e_cutoff_gev=0.15) for k, hw in enumerate((3.2, 3.0))]
        counts = [len(q["x"]) for q in ics]
        d, n0 = ccake_amd.concat_ics(ics), counts[0]
        cfg = dict(config.lumpy_params(), particlization=int(case == "recorded"), pair_precision=int(case == "mixed"))
        if case == "diffusion":
            cfg.update(using_diffusion=1, kappa_over_T2=[0.1, 0, 0, 0, 0.1, 0, 0, 0, 0.1], diffusion_regulator=1)
        r = np.stack([d["x"], d["y"]])
    h = cfg["hT"]
    clean = evaluate(dev, eos, cfg, d, counts, slices, None)
    ok = True
    # the highest rows of event 0 share a tile with the lowest of event 1
    far = [int(np.argmax(r[1, :n0])), int(np.argmin(np.abs(r[0, :n0]) + np.abs(r[1, :n0])))]
    cols = ["EXT_BULK", "EXT_SHV0"] + (["EXT_S"] if not milne else []) + (["EXT_Q0"] if case == "diffusion" else [])
    for col in cols:
        for value in (np.nan, np.inf):
            for i in far if col == "EXT_BULK" else far[:1]:
                got = evaluate(dev, eos, cfg, d, counts, slices, (col, i, value))
                dist = np.sqrt(((r - r[:, i:i + 1]) ** 2).sum(0))
                # a bad density reaches its neighbours' pressures in the smoothing, and theirs in the gradients
                reach = (4.0 if col == "EXT_S" else 2.0) * h
                out = dist > reach * (1 + 1e-12)
                if counts is not None:
                    out[n0:] = True
                same = out.copy()
                if col == "EXT_S":
                    same[:n0] = False
                wrong = {k: int(np.sum(np.abs(v - clean[k])[same] > tol * np.max(np.abs(clean[k]))))
                         + int(np.sum(~np.isfinite(v[out]))) for k, v in got.items()}
                wrong = {k: w for k, w in wrong.items() if w}
                hit = sum(int(np.sum(~np.isfinite(v))) for v in got.values())
                print(case, slices, col, value, i, "out of range", int(out.sum()), "non-finite", hit, "changed out of range",
                      wrong, flush=True)
                ok = ok and not wrong and hit > 0
    if not stepped:
        return ok
    # the first stage spreads it over its range, the second theirs to the densities over theirs and on to the gradients
    clean = evaluate(dev, eos, cfg, d, counts, slices, None, True)
    i = int(np.argmin(r[0, :n0]))
    got = evaluate(dev, eos, cfg, d, counts, slices, ("UX", i, np.nan), True)
    out = np.sqrt(((r - r[:, i:i + 1]) ** 2).sum(0)) > 6.0 * h + 0.05
    if counts is not None:
        out[n0:] = True
    wrong = {k: int(np.sum(~np.isfinite(v[out]))) for k, v in got.items()}
    if counts is not None:
        wrong.update({(k, "second event"): int(np.sum(v[n0:] != clean[k][n0:])) for k, v in got.items()})
    wrong = {k: w for k, w in wrong.items() if w}
    hit = sum(int(np.sum(~np.isfinite(v))) for v in got.values())
    print(case, slices, "UX nan", i, "out of range", int(out.sum()), "non-finite", hit, "changed out of range", wrong, flush=True)
    ok = ok and not wrong and hit > 0
    return ok


def main():
    case, slices = sys.argv[1], int(sys.argv[2]) if len(sys.argv) > 2 else 0
    assert ccake_amd.LIB_PATH.endswith("libccake_emu.so"), ccake_amd.LIB_PATH
    if check(ccake_amd.Device(0), case, slices):
        print("OK", flush=True)


if __name__ == "__main__":
    main()
