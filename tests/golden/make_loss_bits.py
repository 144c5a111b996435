"""Write ``loss_bits.npz`` and ``energy_bits.npz`` (the values of ``test_gpu_loss_bits.py``'s cases) from the built library, on
a GPU.  The committed files are from commit 9ab37b9's library.

    python tests/golden/make_loss_bits.py [output folder]
"""
from __future__ import annotations

import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(HERE))
sys.path.insert(0, os.path.dirname(os.path.dirname(HERE)))

from test_gpu_loss_bits import CASES, ENERGIES, energies, key, statistics  # noqa: E402

if __name__ == "__main__":
    folder = sys.argv[1] if len(sys.argv) > 1 else HERE
    out = {}
    for case in CASES:
        for suffix, value in zip(("_loss", "_clip", "_eloc"), statistics(case)):
            out[key(case) + suffix] = value
    np.savez_compressed(os.path.join(folder, "loss_bits.npz"), **out)
    np.savez_compressed(os.path.join(folder, "energy_bits.npz"), **{key(c): energies(c) for c in ENERGIES})
