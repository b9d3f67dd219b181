"""The host path of eager calls: the extension module ``_native``, or what stands for it where that cannot be loaded.

``_native`` is built for one Python and one torch.  Every call that it serves has a Python path behind it -- the same kernels
of ``libbsi_hip.so``, more host time a call -- so that another interpreter, or another torch, has a slower package and not
none.  That is said once, when the package is imported."""
from __future__ import annotations

import warnings

import torch

# torch.compile leaves a graph at a BSI layer, which runs as it does eagerly (one break a layer; its launches are no operators
# that a graph could hold).  Dynamo's advice to report the builtin it breaks at is of no use to anybody.
warnings.filterwarnings("ignore", message=r"Dynamo does not know how to trace the builtin `bsipytorch_amd\._native\.")


class PythonPath:
    """``_native``'s functions for a process without it: every call is left to the Python path."""

    _generation = 0
    layer_call = torch.nn.Module.__call__

    @staticmethod
    def _not_served(*args):
        return None

    build = build_keys = hybrid = ewah_streams = dot_streams = linear = scalar_query = dot = _not_served
    bind = bind_layer = forget = _not_served

    @classmethod
    def configure(cls, *flags):
        cls._generation += 1

    @classmethod
    def build_key(cls, x: torch.Tensor, decimals: int, Sb: int):
        if x.is_inference() or x.dim() < 1 or x.numel() == 0:
            return None
        return (x.data_ptr(), tuple(x.shape), x.dtype, x._version, cls._generation, decimals, Sb)


try:
    from . import _native as native
except ImportError as why:
    warnings.warn(f"bsipytorch_amd: the native host path cannot be loaded ({why}); eager calls take the Python path, which costs "
                  "the host more a call.  `make -C bsipytorch_amd/csrc` builds it for this Python and torch.", RuntimeWarning)
    native = PythonPath
