"""The slice counts that an event takes (test infrastructure): every one up to
the one it was created with, which nslices() then returns, and none beyond.
The sizes are 1 tile, one that leaves the chip's SIMDs half empty, and whole
rounds of them (one slice).  Prints "OK".

Usage (through tests/hostemu/emu.sh): run_slices.py
"""
from __future__ import annotations

import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import ccake_amd  # noqa: E402
from ccake_amd import config  # noqa: E402


def main():
    assert ccake_amd.LIB_PATH.endswith("libccake_emu.so"), ccake_amd.LIB_PATH
    dev = ccake_amd.Device(0)
    eos = ccake_amd.Eos(dev, 0, 150.0 / config.HBARC_MEVFM)
    created = set()
    for dim, n in ((2, 64), (2, 131072), (2, 196608), (2, 262144), (3, 64), (3, 262144)):
        cfg = dict(config.lumpy_params(dim=dim), particlization=0)
        ev = ccake_amd.Batch(dev, eos, cfg, [n - n // 3, n // 3]) if dim == 2 else ccake_amd.Event(dev, eos, cfg, n)
        cap = ev.nslices()
        created.add(cap)
        took = [s for s in range(1, 17) if accepts(ev, s)]
        print(dim, n, "created with", cap, "accepts", took, flush=True)
        assert took == list(range(1, cap + 1))
        # what a caller with a wish of its own sets
        assert all(ev.nslices(min(s, cap)) == min(s, cap) for s in range(1, 17))
        ev.close()
    assert 1 in created and 16 in created
    print("OK", flush=True)


def accepts(ev, s):
    try:
        return ev.nslices(s) == s
    except ccake_amd.CcakeError:
        return False


if __name__ == "__main__":
    main()
