"""ctypes binding of libdwoconv1d_hip.so (the declarations of include/dwoconv1d_hip.h)."""
import ctypes
import os

HERE = os.path.dirname(os.path.abspath(__file__))
# DWOCONV1D_LIB overrides the library location (e.g. an instrumented build)
LIB_PATH = os.environ.get("DWOCONV1D_LIB") or os.path.join(HERE, "libdwoconv1d_hip.so")
HOST_PATH = os.path.join(HERE, "_host.so")

F32, BF16, F16 = 0, 1, 2
NCHW, NHWC, GROUPED = 0, 1, 2

_vp, _i, _sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t

# name -> (restype, argtypes); kept in the order of the header
SIGNATURES = {
    "dwo_version": (_i, []),
    "dwo_status_string": (ctypes.c_char_p, [_i]),
    "dwo_init": (_i, []),
    "dwo_taps_bytes": (_sz, [_i, _i]),
    "dwo_build_taps": (_i, [_vp, _i, _i, _vp]),
    "dwo_taps_grouped": (_i, [_vp, _i]),
    "dwo_taps_get": (_i, [_vp, _i, _i, ctypes.POINTER(_i), ctypes.POINTER(_i)]),
    "dwo_fprop": (_i, [_vp, _vp, _vp, _vp, _vp] + [_i] * 8 + [_vp]),
    "dwo_dgrad": (_i, [_vp, _vp, _vp, _vp] + [_i] * 8 + [_vp]),
    "dwo_wgrad_scratch_bytes": (_sz, [_i] * 8),
    "dwo_wgrad": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _sz] + [_i] * 8 + [_vp]),
    "dwo_wgrad_static": (_i, [_vp, _vp, _vp, _vp, _vp] + [_i] * 8 + [_vp]),
    "dwo_set_wgrad_reduction": (_i, [_i]),
    "dwo_pointwise_fprop_nhwc": (_i, [_vp] * 7 + [_i] * 8 + [_vp]),
    "dwo_pointwise_fprop": (_i, [_vp] * 7 + [_i] * 9 + [_vp]),
    "dwo_layernorm_nhwc": (_i, [_vp, _vp, _vp, _vp, _sz, _i, ctypes.c_float, _i, _i, _vp]),
    "dwo_nchw_layernorm_nhwc": (_i, [_vp, _vp, _vp, _vp, _i, _i, _i, _i, ctypes.c_float, _i, _vp]),
    "dwo_nhwc_scale_add_nchw": (_i, [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp]),
    "dwo_pointwise_wgrad_scratch_bytes": (_sz, [_i, _i]),
    "dwo_pointwise_wgrad": (_i, [_vp] * 5 + [_sz, _sz] + [_i] * 3 + [_vp]),
    "dwo_pointwise_forward": (_i, [_vp] * 4 + [_sz] + [_i] * 3 + [_vp]),
    "dwo_block_scratch_bytes": (_sz, [_i]),
    "dwo_ln_rows": (_i, [_vp] * 5 + [_sz, _i, ctypes.c_float] + [_i] * 3 + [_vp]),
    "dwo_ln_rows_backward": (_i, [_vp] * 9 + [_sz, _sz] + [_i] * 5 + [_vp]),
    "dwo_ln_tile": (_i, [_vp] * 5 + [_i] * 4 + [ctypes.c_float] + [_i] * 2 + [_vp]),
    "dwo_ln_tile_backward": (_i, [_vp] * 8 + [_sz] + [_i] * 7 + [_vp]),
    "dwo_ln_patch": (_i, [_vp] * 5 + [_i] * 4 + [ctypes.c_float] + [_i] * 2 + [_vp]),
    "dwo_ln_patch_backward": (_i, [_vp] * 8 + [_sz] + [_i] * 7 + [_vp]),
    "dwo_block_tail": (_i, [_vp] * 4 + [_i] * 8 + [_vp]),
    "dwo_block_tail_backward": (_i, [_vp] * 6 + [_sz] + [_i] * 7 + [_vp]),
    "dwo_linear_wgrad_scratch_bytes": (_sz, [_sz, _i, _i]),
    "dwo_linear_rows": (_i, [_vp] * 4 + [_sz] + [_i] * 4 + [_vp]),
    "dwo_linear_planes": (_i, [_vp] * 6 + [_i] * 5 + [_vp]),
    "dwo_block_mlp": (_i, [_vp] * 8 + [_i] * 4 + [_vp]),
    "dwo_linear_norm_planes": (_i, [_vp] * 3 + [ctypes.c_float] + [_vp] * 4 + [ctypes.c_float, _vp] + [_i] * 5 + [_vp]),
    "dwo_linear_wgrad": (_i, [_vp] * 5 + [_sz, _sz] + [_i] * 4 + [_vp]),
}

_lib = None


def load():
    """Load the built library; there is no fallback when it is missing."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            "libdwoconv1d_hip.so is not built (expected at %s); run "
            "`python -m oriented1d_amd.build` -- this operator has no CPU or PyTorch fallback"
            % LIB_PATH)
    lib = ctypes.CDLL(LIB_PATH)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = res, args
    _lib = lib
    return lib


_ready = set()
_host = None


def host(index):
    """The native call path (csrc/dwo_host.cpp) with the kernels set up on CUDA device ``index``
    (below zero for a tensor that is on no CUDA device: the call itself refuses those)."""
    global _host
    if index >= 0 and index not in _ready:
        import torch

        ready(torch.device("cuda", index))
    if _host is None:
        load()
        if not os.path.exists(HOST_PATH):
            raise RuntimeError("%s is not built; run `python -m oriented1d_amd.build`" % HOST_PATH)
        import torch  # noqa: F401  (the extension links against its libraries)
        from . import _host as native

        native.bind(LIB_PATH)
        _host = native
    return _host


def ready(device):
    """The loaded library with its kernels set up on ``device`` (a torch CUDA device): the first
    use on a device runs ``dwo_init`` there, so no later call does anything but launch kernels."""
    import torch

    lib = load()
    index = device.index if device.index is not None else torch.cuda.current_device()
    if index not in _ready:
        with torch.cuda.device(index):
            check(lib.dwo_init(), "dwo_init")
        _ready.add(index)
    return lib


def check(status, what):
    if status != 0:
        msg = load().dwo_status_string(status).decode()
        raise RuntimeError("%s failed: %s (status %d)" % (what, msg, status))
