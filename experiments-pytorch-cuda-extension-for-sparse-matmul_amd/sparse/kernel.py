"""Loader of the HIP library and the ``sparse_ops`` boundary object.

Takes the place of ``sparse/kernel.py:6-16`` of the reference, which JIT-builds a
torch C++/CUDA extension at import time.  Here a prebuilt C-ABI shared object
(``csrc/libbsa_hip.so``, made by ``csrc/build.py`` with hipcc for gfx950) is
opened with ctypes; torch tensors cross the boundary as raw device pointers and
the current HIP stream.  If the library is missing the import fails loudly:
there is no fallback path.
"""
import contextlib
import ctypes
import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (loads the HIP runtime the library binds to)

_CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc")
LIBRARY_PATH = os.path.join(_CSRC, "libbsa_hip.so")

BSA_F32, BSA_F16, BSA_BF16 = 0, 1, 2
BSA_SDD, BSA_DSD, BSA_DDS = 0, 1, 2
BSA_OK, BSA_ERR_INVALID, BSA_ERR_LAUNCH, BSA_ERR_UNSUPPORTED = 0, -1, -2, -3
MODES = {"sdd": BSA_SDD, "dsd": BSA_DSD, "dds": BSA_DDS}

_vp, _i, _i64, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float

# name -> (restype, argtypes); mirrors include/bsa.h one to one
SIGNATURES = {
    "bsa_version": (_i, []),
    "bsa_last_error": (ctypes.c_char_p, []),
    "bsa_layout_workspace_bytes": (ctypes.c_size_t, [_i, _i]),
    "bsa_layout_build": (_i, [_vp, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _vp]),
    "bsa_layout_finish": (_i, [_vp, _vp, _i, _i, _i, _vp, _vp, _vp, _vp, _vp]),
    "bsa_schedule_capacity": (_i64, [_i, _i, _i, _i]),
    "bsa_schedule_build": (_i, [_vp, _i, _i, _i, _i, _i, _i, _vp, _i64, _vp, _vp]),
    "bsa_matmul_workspace_bytes": (ctypes.c_size_t, [_i, _i, _i, _i, _i, _i]),
    "bsa_matmul": (_i, [_i, _i, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _i, _i, _vp, ctypes.c_size_t,
                        _i, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp]),
    "bsa_matmul_noalloc": (_i, [_i, _i, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _i, _i, _i,
                                _i, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp]),
    "bsa_matmul_dsd_block64": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i, _vp]),
    "bsa_matmul_dds_panels": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _vp]),
    "bsa_matmul_dds_panels_limits": (None, [_vp]),
    "bsa_weight_grad_shares": (_i, [_i, _i, _i]),
    "bsa_weight_grad": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp, ctypes.c_size_t, _vp]),
    "bsa_run_schedule_bytes": (ctypes.c_int64, [_i, _i]),
    "bsa_run_schedule_build": (_i, [_vp, _vp, _i, _i, _i, _i, _vp, ctypes.c_int64, _vp, _vp]),
    "bsa_matmul_dsd_runs": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _i, _i, _i, _i, _vp]),
    "bsa_softmax_forward": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "bsa_softmax_backward": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _f, _vp]),
    "bsa_to_sparse": (_i, [_i, _vp, _vp, _vp, _i, _i, _i, _i, _vp]),
    "bsa_to_dense": (_i, [_i, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _vp]),
    "bsa_attention_workspace_bytes": (ctypes.c_size_t, [_i, _i, _i, _i]),
    "bsa_attention_forward": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _vp, ctypes.c_size_t,
                                   _i, _i, _i, _i, _i, _f, _i, _vp]),
    "bsa_attention_backward_workspace_bytes": (ctypes.c_size_t, [_i, _i, _i, _i, _i, _i]),
    "bsa_attention_backward_scores": (_i, [_i, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i,
                                           _i, _i, _vp, ctypes.c_size_t, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "bsa_attention_backward": (_i, [_i] + [_vp] * 10 + [_vp, _vp, _vp, _i, _i, _i, _i, _vp, _vp, _vp, _i, _i, _i, _i,
                                                        _vp, ctypes.c_size_t, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "bsa_attention_gradients": (_i, [_i] + [_vp] * 10 + [_vp, _vp, _vp, _i, _i, _i, _i, _vp, _vp, _vp, _i, _i, _i, _i,
                                                        _vp, ctypes.c_size_t, _i, _i, _i, _i, _i, _f, _i, _vp]),
}


class BsaError(RuntimeError):
    """A C-ABI call returned a nonzero status."""


def load_library(path: str = LIBRARY_PATH) -> ctypes.CDLL:
    if not os.path.exists(path):
        raise ImportError(
            f"{path} is missing: build it with `python {os.path.join(_CSRC, 'build.py')}` "
            "(hipcc, --offload-arch=gfx950). There is no fallback implementation.")
    lib = ctypes.CDLL(path)
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)      # AttributeError if the symbol is not exported
        fn.restype, fn.argtypes = restype, argtypes
    return lib


lib = load_library()


def load_host_calls():
    """The native host side (``csrc/host_calls.cpp``), built beside the library; missing, the import fails as loudly."""
    path = os.path.join(_CSRC, "bsa_host_calls.so")
    if not os.path.exists(path):
        raise ImportError(f"{path} is missing: build it with `python {os.path.join(_CSRC, 'build.py')}`")
    spec = importlib.util.spec_from_file_location("bsa_host_calls", path,
                                                  loader=importlib.machinery.ExtensionFileLoader("bsa_host_calls", path))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    if module.torch_version != torch.__version__:        # it uses torch's C++ interface, which no two versions share
        raise ImportError(f"{path} was built for torch {module.torch_version}, this is {torch.__version__}: build it again")
    return module


host_calls = load_host_calls()


def dds_panel_limits():
    """Dense rows of a workgroup of the panel walk, block rows of the contraction and blocks it is built for."""
    limits = (ctypes.c_int32 * 3)()
    lib.bsa_matmul_dds_panels_limits(limits)
    return tuple(limits)


def check(status: int) -> None:
    if status != 0:
        raise BsaError(f"bsa status {status}: {lib.bsa_last_error().decode()}")


# The stream and device queries every call makes, as torch's own generated code makes them: 0.1 us each against 3.1 us
# for torch.cuda.current_stream() (which builds a Stream object) and 1.5 us for entering torch.cuda.device.
_current_device = torch._C._cuda_getDevice if hasattr(torch._C, "_cuda_getDevice") else torch.cuda.current_device
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def current_stream() -> int:
    """Handle of the current stream of the current device."""
    if _raw_stream is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_current_device())


_SAME_DEVICE = contextlib.nullcontext()


def on_device(device: torch.device):
    """``torch.cuda.device(device)``, or nothing to enter when that is the current device already."""
    return _SAME_DEVICE if device.index == _current_device() else torch.cuda.device(device)


from . import _ops as sparse_ops  # noqa: E402  (module with the reference's sparse_matmul signature)
