"""The plain cases of the eager path in C++ (``csrc/mx_host.cpp``), loaded when first asked for.

``host.f(...)`` does the work of a function of ``kernels/`` in one call -- its allocations, its launches, its views -- or returns
``None``, with nothing launched, for every call that is not plain: then the Python function goes on itself.
"""

from __future__ import annotations


def __getattr__(name: str):
    if name.startswith("__"):
        raise AttributeError(name)
    from kohakuwullm_amd import _lib

    _lib.load()
    library = _lib.product()
    try:
        from kohakuwullm_amd import _host
    except ImportError as error:
        raise _lib.MXFP8LibraryError(f"kohakuwullm_amd/_host.so cannot be loaded ({error}): `make -C kohakuwullm_amd/csrc` builds it") from error
    _host.bind(_lib.LIB_PATH, library, _lib.own_invoke, _lib)
    globals().update({n: getattr(_host, n) for n in dir(_host) if not n.startswith("_") and n != "bind"})
    return globals()[name]
