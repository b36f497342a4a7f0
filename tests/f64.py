"""float32 arrays as float64 for the tests."""
from __future__ import annotations

import numpy as np


def f64_of_bits(x):
    """float32 values as float64 from their bits (a process in which some library
    has set the CPU to flush subnormals converts them to zero)."""
    u = np.ascontiguousarray(x).view(np.uint32).astype(np.int64)
    e = (u >> 23) & 255
    frac = (u & 0x7FFFFF) | np.where(e > 0, 1 << 23, 0)
    return np.where(u >> 31, -1.0, 1.0) * np.ldexp(frac.astype(np.float64),
                                                   np.maximum(e, 1) - 150)
