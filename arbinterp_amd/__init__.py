"""MI355X-native Lekien-Marsden tricubic / quadcubic interpolation.

`from arbinterp_amd.ARBInterp import tricubic, quadcubic` is the drop-in for
the reference's `from ARBInterp.ARBInterp import tricubic, quadcubic`.
"""
from .ARBInterp import tricubic, quadcubic, __version__  # noqa: F401


def release_memory():
    """Give device memory kept from dropped fields (at most 512 MB) back to the
    device; returns its bytes."""
    from . import _native as N
    return N.lib().arb_release_memory()
