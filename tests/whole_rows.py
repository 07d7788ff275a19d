"""Products that take whole rows to a workgroup, by the variant of the kernel that the plan picks for them (one GPU of 256 CUs), and the
plan as the library makes it."""
import ctypes as C

import cases as K

BLOCKS = [K.Q4_0, K.Q5_0, K.Q5_1, K.Q8_0]
# (rows, columns, tokens, rows of a workgroup, its wavefronts): the remainders of workgroups, of the layout's 256 rows and of shares of the
# columns, odd counts of steps; up to eight tokens, up to sixteen, and tiles of tokens
_UP_TO_8 = [(33, 480, 5, 16, 8), (300, 2080, 8, 16, 16), (4130, 160, 3, 32, 8), (4097, 2080, 8, 32, 16), (8255, 160, 5, 64, 8),
            (8193, 2080, 3, 64, 16), (16385, 480, 6, 64, 4)]
_UP_TO_16 = [(33, 480, 9, 16, 8), (300, 2080, 16, 16, 16), (4130, 288, 12, 32, 8), (4097, 2080, 9, 32, 16), (8255, 288, 16, 64, 8),
             (12289, 2080, 11, 64, 16), (16385, 288, 9, 64, 4)]
_TILES = [(33, 96, 17, 16, 8), (300, 2080, 31, 16, 16), (2080, 288, 17, 32, 8), (2049, 2080, 33, 32, 16), (4130, 288, 20, 64, 8),
          (4097, 2080, 17, 64, 16)]
VARIANTS = {ty: _UP_TO_8 + _UP_TO_16 + _TILES for ty in BLOCKS}
VARIANTS[K.Q4_K] = [(33, 512, 5, 16, 8), (300, 2304, 8, 16, 16), (4130, 768, 3, 32, 8), (4097, 2304, 8, 32, 16), (8255, 768, 5, 64, 8),
                    (8193, 2304, 3, 64, 16), (33, 512, 9, 16, 8), (300, 2304, 16, 16, 8), (4130, 768, 12, 32, 8), (8255, 768, 16, 32, 4),
                    (33, 512, 17, 16, 8), (2049, 768, 17, 32, 8)]
VARIANTS[K.Q6_K] = [(33, 512, 5, 16, 8), (300, 2304, 8, 16, 16), (4130, 768, 3, 32, 8), (4097, 2304, 5, 32, 16), (8255, 768, 8, 64, 8),
                    (16383, 2048, 3, 64, 16), (16385, 512, 6, 64, 4), (33, 512, 9, 16, 8), (300, 2304, 17, 16, 16), (2049, 768, 9, 32, 8),
                    (2049, 2304, 9, 32, 16), (4130, 768, 15, 64, 8), (4097, 2048, 9, 64, 16)]
# products in a chain: rows that are columns of another matrix
CHAINED = {ty: [(512, 2080, 8, 16, 16), (4352, 288, 3, 32, 8), (4352, 2080, 8, 32, 16), (8448, 288, 5, 64, 8), (8448, 2080, 8, 64, 16),
                (4352, 288, 12, 32, 8), (8448, 288, 16, 64, 8), (4352, 288, 20, 64, 8), (2304, 2080, 24, 32, 16), (4352, 288, 40, 64, 8)]
           for ty in BLOCKS}
CHAINED[K.Q4_K] = [(512, 2304, 8, 16, 16), (4352, 768, 3, 32, 8), (4352, 2304, 8, 32, 16), (8448, 768, 5, 64, 8), (8448, 2304, 8, 64, 16),
                   (4352, 768, 12, 32, 8), (8448, 768, 16, 32, 4), (2304, 768, 24, 32, 8), (2304, 768, 40, 32, 8)]
CHAINED[K.Q6_K] = [(512, 2304, 8, 16, 16), (4352, 768, 3, 32, 8), (4352, 2304, 8, 32, 16), (8448, 768, 5, 64, 8), (16640, 512, 6, 64, 4),
                   (2304, 768, 12, 32, 8), (4352, 768, 24, 64, 8), (2304, 768, 40, 64, 8)]


class MatView(C.Structure):  # csrc/matview.h
    _fields_ = [("p", C.c_void_p * 4), ("s", C.c_uint32 * 4), ("type", C.c_uint32), ("rows", C.c_uint32), ("cols", C.c_uint32), ("nb", C.c_uint32)]


class _WholeRows(C.Structure):
    _fields_ = [("rows", C.c_uint32), ("waves", C.c_uint32)]


def views(ty, rows, cols):
    mats = (MatView * len(rows))()
    for m, r in zip(mats, rows):
        m.type, m.rows, m.cols = ty, r, cols
    return mats


def planned(lib, ty, rows, cols, tokens, xs=None, ys=None):
    """(rows, wavefronts) of a workgroup that owns whole rows in the launch of these products, (0, 0) where columns are shared."""
    f = getattr(lib, "_ZN2nh18planned_whole_rowsEPKNS_7MatViewEPKjPKPKfPKPfj")
    f.restype = _WholeRows
    n = len(rows)
    toks = (C.c_uint32 * n)(*(tokens if isinstance(tokens, (list, tuple)) else [tokens] * n))
    p = f(views(ty, rows, cols), toks, (C.c_void_p * n)(*xs) if xs else None, (C.c_void_p * n)(*ys) if ys else None, C.c_uint32(n))
    return p.rows, p.waves
