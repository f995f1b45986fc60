"""Tables with a single node along some axes (test infrastructure): a cell's
corners along such an axis have the weights 1 and 0, and the second one's values
are read all the same.  Under AddressSanitizer, and with the thermodynamics at
the table's nodes equal to the table's.  Prints "OK".

Usage (through tests/hostemu/emu.sh): run_one_node_axis.py
"""
from __future__ import annotations

import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

import ccake_amd  # noqa: E402
from ccake_amd import config, eos_tables  # noqa: E402


def main():
    assert ccake_amd.LIB_PATH.endswith("libccake_emu.so"), ccake_amd.LIB_PATH
    dev = ccake_amd.Device(0)
    T_FO = 150.0 / config.HBARC_MEVFM
    for dims in ((8, 1, 1, 1), (8, 1, 1, 3), (8, 3, 1, 1), (8, 3, 3, 1), (8, 3, 3, 3)):
        tab, dims, mins, maxs = eos_tables.tanh_conformal_table(dims=dims)
        eos = ccake_amd.Eos(dev, config.EOS_TABLE, T_FO, dims, mins, maxs, tab)
        t = np.asarray(tab).reshape(tuple(dims) + (17,))
        for i in (0, 1, dims[0] - 1):
            at = [i] + [n - 1 for n in dims[1:]]
            x = [mins[a] if n == 1 else mins[a] + at[a] * ((maxs[a] - mins[a]) / (n - 1.0)) for a, n in enumerate(dims)]
            r = eos.full_thermo(0, x)
            want = t[tuple(at)]
            assert np.all(np.isfinite(r)) and np.allclose(r, want, rtol=1e-10, atol=1e-10), (dims, at, r, want)
        # the device's copies: an inversion from a state on the table (solvable or not, without charges' axes)
        n = 64
        ev = ccake_amd.Event(dev, eos, dict(config.lumpy_params(), particlization=0), n)
        g = np.linspace(-0.4, 0.4, 8)
        x, y = (a.ravel() for a in np.meshgrid(g, g))
        z = np.zeros(n)
        ccake_amd.load_event(ev, dict(x=x, y=y, e=np.full(n, 20.0), ux=z, uy=z, rhoB=z, rhoS=z, rhoQ=z))
        try:
            ev.initialize()
        except ccake_amd.CcakeError as e:
            print(dims, "reported:", e, flush=True)
        ev.close()
        eos.close()
        print(dims, "ok", flush=True)
    print("OK", flush=True)


if __name__ == "__main__":
    main()
