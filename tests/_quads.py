"""The library's choice between quads (four slices side by side) and single slices:
its own functions, called on the host, and the distance of the angles restated."""
import ctypes
import os
import re

import numpy as np
import torch  # noqa: F401  (its HIP runtime is the one to load first)
from ctrecon import _lib, load

_LIB = load()
with open(os.path.join(os.path.dirname(_lib.__file__), "..", "csrc", "ctr_api.cpp")) as _f:
    MAX_RIM_TEXELS, ALIGN_MAX_RIM_TEXELS = (float(v) for v in re.search(
        r"QUAD_MAX_RIM_TEXELS = ([0-9.]+), ALIGN_MAX_RIM_TEXELS = ([0-9.]+);", _f.read()).groups())


def rim_texels(ang, D, stride):
    """Mean distance of the rims of strips at neighbouring angles of a subset."""
    a = np.asarray(ang, np.float64)[::stride]
    step = np.abs(np.remainder(np.diff(a) + 90.0, 180.0) - 90.0)
    return float(step.mean() * np.pi / 180.0 * 0.5 * D) if len(a) > 1 else 0.0


def stack_quads(nx, ny, px, pa, ss, dn, ang, passes=2 ** 31 - 1):
    """Layers of an OS-EM, TV OS-EM or AART (passes: its subsets in all) stack that run
    as quads."""
    nq = _LIB._ZN3ctr14stack_quads_ofEiiiiii(dn, nx, ny, px, pa // ss, passes)
    return nq if nq and rim_texels(ang, max(nx, ny), ss) <= MAX_RIM_TEXELS else 0


def align_quads(nx, ny, px, pa, dn, ang):
    """Layers of an alignment forward that run as quads."""
    nq = _LIB._ZN3ctr14align_quads_ofEiiiii(dn, nx, ny, px, pa)
    return nq if nq and rim_texels(ang, max(nx, ny), 1) <= ALIGN_MAX_RIM_TEXELS else 0


def fbp_kernels(nx, ny, zp, dn):
    """Layers of an FBP call that run as quads, and the kernels of its backprojection
    (slices side by side, rows, angle shares, as digits)."""
    nq = _LIB._ZN3ctr12fbp_quads_ofEiiii(dn, nx, ny, zp)
    parts = [((nq + 3) // 4, 1)] * (nq > 0) + [(dn - nq, 0)] * (nq < dn)
    return nq, {_LIB._ZN3ctr10fbp_kernelEiiii(nx, ny, units, quads) for units, quads in parts}


def batch_quads(sides, na):
    """Slices of a batch that run as quads (angles close enough to share windows)."""
    runs = {n: sides.count(n) for n in set(sides)}
    if len(runs) == 1:
        n = sides[0]
        return _LIB._ZN3ctr14stack_quads_ofEiiiiii(len(sides), n, n, n, na, 2 ** 31 - 1)
    part = {n: k if k >= 3 and k % 4 >= 2 else k // 4 * 4 for n, k in runs.items()}
    blocks = sum(q * ((n + 63) // 64) * ((na + 1) // 2) for n, q in part.items())
    bp = sum((q + 3) // 4 * ((n + 63) // 64) * ((n + 15) // 16) for n, q in part.items())
    nq = sum(part.values())
    take = _LIB._ZN3ctr17batch_takes_quadsExxx
    take.argtypes, take.restype = [ctypes.c_longlong] * 3, ctypes.c_bool
    return nq if take(blocks, bp, len(sides) - nq) else 0
