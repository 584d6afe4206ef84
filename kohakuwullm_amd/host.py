"""The plain cases of the eager path in C++ (``csrc/mx_host.cpp``), loaded when first asked for.

``host.f(...)`` does the work of a function of ``kernels/`` in one call -- its allocations, its launches, its views -- or returns
``None``, with nothing launched, for every call that is not plain: then the Python function goes on itself.  Without the extension
(not built, or built against another PyTorch) no call is plain: the same kernels, behind slower host code, and a warning.
"""

from __future__ import annotations


_told = False


def _declined(*args):
    """What every function here is while the extension cannot be used."""


def __getattr__(name: str):
    if name.startswith("__"):
        raise AttributeError(name)
    import torch

    from kohakuwullm_amd import _lib

    try:
        _lib.load()
    except _lib.MXFP8LibraryError:  # the Python function says so where it would call the library
        return _declined
    try:
        from kohakuwullm_amd import _host

        built = getattr(_host, "torch_version", "another release")
        if not torch.__version__.startswith(built):
            raise ImportError(f"built against PyTorch {built}, this is {torch.__version__}")
    except ImportError as error:
        if not _told:
            import warnings

            warnings.warn(f"kohakuwullm_amd/_host.so cannot be used ({error}): launches take the slower Python way.  "
                          "`make -C kohakuwullm_amd/csrc` builds it.", RuntimeWarning, stacklevel=3)
        globals().update({"_told": True, name: _declined})
        return _declined
    _host.bind(_lib.LIB_PATH, _lib.product(), _lib.own_invoke, _lib)
    globals().update({n: getattr(_host, n) for n in dir(_host) if callable(getattr(_host, n)) and not n.startswith("_") and n != "bind"})
    return globals()[name]
