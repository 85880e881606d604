"""The library's choice between quads (four slices side by side) and single slices,
restated, with its lines read from the sources: which layers of a stack run as
quads, and which of the FBP backprojection's kernels a call takes."""
import os
import re

import numpy as np

_CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ct-xafs_analysis_amd", "csrc")
_TEXT = {f: open(os.path.join(_CSRC, f)).read() for f in ("ctr_api.cpp", "ctr_internal.h", "ctr_kernels.hip")}


def const(name):
    for text in _TEXT.values():
        m = re.search(r"constexpr [^;]*?\b" + name + r" = ([0-9.]+)", text)
        if m:
            return float(m.group(1)) if "." in m.group(1) else int(m.group(1))
    raise KeyError(name)


def _cdiv(a, b):
    return (a + b - 1) // b


def per_quad(px, na):
    return _cdiv(px, 64) * _cdiv(na, const("QA"))


def rim_texels(ang, D, stride):
    """Mean distance of the rims of strips at neighbouring angles of a subset."""
    a = np.asarray(ang, np.float64)[::stride]
    step = np.abs(np.remainder(np.diff(a) + 90.0, 180.0) - 90.0)
    return float(step.mean() * np.pi / 180.0 * 0.5 * D) if len(a) > 1 else 0.0


def one_joins(D, pq):
    return D <= const("QUAD_ONE_OVER_SIDE") and pq * D <= const("QUAD_ONE_OVER_WORK")


def quads_of(n, D, pq, bp):
    if n < 3:
        return 0
    one = n % 4 == 1
    nq = n - 1 if one and not one_joins(D, pq) else n
    least = const("QUAD_MIN_BLOCKS" + ("" if not one else
                                       "_ONE_SMALL" if D <= const("QUAD_ONE_OVER_SIDE") else "_ONE_LARGE"))
    return nq if nq * pq >= 4 * least and _cdiv(nq, 4) * bp >= const("QUAD_MIN_BP_BLOCKS") else 0


def stack_quads(nx, ny, px, pa, ss, dn, ang):
    """Layers of an OS-EM, TV OS-EM or AART stack that run as quads."""
    D = max(nx, ny)
    nq = quads_of(dn, D, per_quad(px, pa // ss), _cdiv(nx, 64) * _cdiv(ny, 4 * const("QBP_ROWS")))
    return nq if nq and rim_texels(ang, D, ss) <= const("QUAD_MAX_RIM_TEXELS") else 0


def align_quads(nx, ny, px, pa, dn, ang):
    """Layers of an alignment forward that run as quads."""
    D = max(nx, ny)
    if dn < 3 or D > 3840:
        return 0
    one = dn % 4 == 1
    into = one and dn > 8 and one_joins(D, per_quad(px, pa))
    nq = dn - 1 if one and not into else dn
    least = const("ALIGN_QUAD_MIN_BLOCKS" + ("_ONE_IN" if into else "_ONE_BESIDE" if one else ""))
    return nq if nq * per_quad(px, pa) >= 4 * least and rim_texels(ang, D, 1) <= const("QUAD_MAX_RIM_TEXELS") else 0


def fbp_kernels(nx, ny, zp, dn):
    """The backprojection kernels <slices, rows, angle shares> of an FBP call."""
    nq = dn if dn >= 3 and dn % 4 >= 2 else dn // 4 * 4
    units = _cdiv(nq, 4)
    if units * _cdiv(nx, 64) * _cdiv(ny, 4) < const("FBP_QUAD_MIN_BLOCKS") or zp > const("FBP_QUAD_MAX_ZP"):
        nq = units = 0
    lines = [int(v) for v in re.findall(r"blocks\((?:16|8)\) >= (\d+)", _TEXT["ctr_kernels.hip"])]
    blocks = lambda rows, n: _cdiv(nx, 64) * _cdiv(ny, rows) * n            # noqa: E731
    out = set()
    if units:
        out.add("4,4,0" if blocks(16, units) >= lines[0] else "4,4,4")
    if dn > nq:
        rest = dn - nq
        out.add("1,4,0" if blocks(16, rest) >= lines[1] else "1,8,4" if blocks(8, rest) >= lines[2] else "1,4,8")
    return out
