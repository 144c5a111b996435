"""Write ``loss_bits.npz``: loss, clipping state and local energies of ``test_gpu_loss_bits.py``'s cases from the built
library, on a GPU.  The committed file is from commit 9ab37b9's library.

    python tests/golden/make_loss_bits.py [output file]
"""
from __future__ import annotations

import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(HERE))
sys.path.insert(0, os.path.dirname(os.path.dirname(HERE)))

from test_gpu_loss_bits import CASES, FILE, key, statistics  # noqa: E402

if __name__ == "__main__":
    out = {}
    for case in CASES:
        for suffix, value in zip(("_loss", "_clip", "_eloc"), statistics(case)):
            out[key(case) + suffix] = value
    np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else FILE, **out)
