"""The native host path of the modules (csrc/host_passes.cpp): loads the extension, loudly when it is not built."""
from . import _lib

_lib.load()   # the kernels' library, which the extension calls, with its interface version checked

try:
    from ._host import Due, Route, Setup, cast_weights, gating, linear_step, mlp_step, route, set_kernel_timing
except ImportError as exc:
    raise ImportError("fp8_gmm_amd/_host.so is missing or does not load: build the extensions "
                      "(`make -C fp8_gmm_amd/csrc -j8`)") from exc

__all__ = ["Due", "Route", "Setup", "cast_weights", "gating", "linear_step", "mlp_step", "route", "set_kernel_timing"]
