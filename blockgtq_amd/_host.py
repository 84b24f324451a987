"""Loader of the native host side (csrc/bgtq_host.cpp): layer handles that issue a whole decode
step or an append in one call.  There is no Python substitute: a missing extension raises."""
import os

from . import _capi
from .build import HOST_PATH

_mod = None


def module():
    """The extension module, loaded and set up once."""
    global _mod
    if _mod is None:
        _capi.lib()                                  # the library the extension calls, layout-checked
        if not os.path.exists(HOST_PATH):
            raise _capi.BgtqError(f"{HOST_PATH} is missing: build it with `python -m blockgtq_amd.build`")
        import importlib.util
        from . import ops
        spec = importlib.util.spec_from_file_location("_bgtq_host", HOST_PATH)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.setup(_capi.BgtqError, ops._note_path)
        _mod = mod
    return _mod


def layer(li, plans, k_packed, k_norms, v_packed, v_norms, k_row_width, norm_width, v_row_width, n_q,
          k_layout, v_layout, scale, baked, buf_k, buf_v):
    """A native handle of layer ``li`` over its plans and cache, or None where the cache is not on the GPU (the general
    path then says so).  The cache tensors are one layer's, or all layers' stacked; the handle's ``holds`` takes the
    same arguments and says whether it still is what this would make of them."""
    if not (plans.is_cuda and k_packed.is_cuda):
        return None

    def one(t, dims=4):
        return t[li] if t is not None and t.dim() == dims + 1 else t
    return module().Layer(plans, one(k_packed), one(k_norms), one(v_packed), one(v_norms, 3), k_row_width, norm_width,
                          v_row_width, n_q, k_layout, v_layout, scale, baked, one(buf_k), one(buf_v))
