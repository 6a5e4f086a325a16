"""The oracle in extended precision (x87 long double, 64-bit mantissa): the
same source with its double types widened, for tests that measure rounding."""
import copy
import types

import numpy as np

from oracle import chan_oracle as O


class _Numpy:
    """numpy whose new arrays are extended by default."""
    def __getattr__(self, k):
        return getattr(np, k)

    @staticmethod
    def zeros(shape, dtype=np.longdouble):
        return np.zeros(shape, dtype)

    @staticmethod
    def empty(shape, dtype=np.longdouble):
        return np.empty(shape, dtype)


def _load():
    with open(O.__file__) as f:
        src = f.read()
    for a, b in (("np.complex128", "np.clongdouble"), ("np.float64", "np.longdouble"), ("float(", "np.longdouble("),
                 ("math.cos(", "np.cos("), ("math.sin(", "np.sin("), ("import numpy as np\n", "np = _extended_numpy\n")):
        assert a in src
        src = src.replace(a, b)
    m = types.ModuleType("chan_oracle_extended")
    m.__dict__["_extended_numpy"] = _Numpy()
    import sys
    sys.modules[m.__name__] = m          # its dataclasses look their module up
    exec(compile(src, m.__name__, "exec"), m.__dict__)
    for k in ("RKA", "RKB", "RKC", "RKD"):
        setattr(m, k, [np.longdouble(v) for v in getattr(O, k)])
    return m


X = _load()


def wide(a):
    """A double scalar or array as an extended one."""
    if isinstance(a, np.ndarray):
        return a.astype(np.clongdouble if a.dtype.kind == "c" else np.longdouble)
    return np.longdouble(a)


def wide_grid(g):
    """The grid with its operators, as they are in double, as extended values."""
    g = copy.copy(g)
    for k, v in list(vars(g).items()):
        if isinstance(v, (np.ndarray, float)):
            setattr(g, k, wide(v))
    g.ikx, g.ikz = 1j * g.kx, 1j * g.kz
    return g


def error(a, ref):
    """2-norm of a - ref over that of ref (extended)."""
    return float(np.linalg.norm((a - ref).ravel()) / np.linalg.norm(ref.ravel()))
