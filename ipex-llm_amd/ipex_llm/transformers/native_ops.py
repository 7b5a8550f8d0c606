"""The native host path (csrc/torch_ops.cpp): from torch tensors to a launch of the C ABI in one call.

Loaded from the same directory as liblowbit_hip.so and bound to the functions of the library that the ctypes binding
has loaded.  Like the library it has no substitute: a build without it raises here."""
import ctypes
import importlib.machinery
import importlib.util

import torch  # noqa: F401  (its shared libraries have to be there before the module's)

import ipex_llm.ggml.model.llama.llama_cpp as ggml
from ipex_llm.utils.common import invalidInputError
from ipex_llm.utils.utils import get_shared_lib_info

_BOUND = ("last_error", "blob_bytes", "tileable", "linear_scratch_bytes", "linear", "gated_mlp", "dequantize_rows", "dequantize", "backward_ws", "backward_workspace_bytes", "backward_ws_applies",
          "experts_workspace_bytes", "experts_forward")


def _load():
    path = get_shared_lib_info("lowbit_hip")[0] / "lowbit_torch.so"
    invalidInputError(path.exists(), f"{path} not found; build it with `make -C ipex-llm_amd/csrc`.")
    loader = importlib.machinery.ExtensionFileLoader("lowbit_torch", str(path))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("lowbit_torch", loader))
    loader.exec_module(module)
    module.bind({f"lowbit_{name}": ctypes.cast(getattr(ggml._lib, f"lowbit_{name}"), ctypes.c_void_p).value
                 for name in _BOUND})
    return module


ops = _load()
