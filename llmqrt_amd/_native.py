"""Loads lib/_llmq_host.so (csrc/host_ops.cpp): the native forward passes of the quantized modules.

Every function returns None for an input outside its layout; the caller then takes its general path.  There is no
fallback for a library that has not been built: loading it raises.
"""
from __future__ import annotations

import importlib.machinery
import importlib.util
import pathlib

import torch  # the extension's torch and HIP libraries must be in the process first

from . import _abi

_PATH = pathlib.Path(__file__).resolve().parent / "lib" / "_llmq_host.so"


def _load():
    _abi.lib()
    if not _PATH.exists():
        raise RuntimeError(f"{_PATH} is missing: build it with `python -m llmqrt_amd.csrc.build` "
                           "(there is no CPU or PyTorch fallback for these ops)")
    loader = importlib.machinery.ExtensionFileLoader("_llmq_host", str(_PATH))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_llmq_host", loader))
    loader.exec_module(module)
    if module.torch_version != torch.__version__:
        raise RuntimeError(f"{_PATH} was built against torch {module.torch_version} and this is torch {torch.__version__}: "
                           "build it again with `python -m llmqrt_amd.csrc.build`")
    return module


_host = None


def host():
    global _host
    if _host is None:
        _host = _load()
    return _host
