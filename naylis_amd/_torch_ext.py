"""Loader for the torch extension of the fused layer node
(``naylis_amd/_lib/ext/naylis_torch.so``, built from csrc/torch_layer.cpp by
naylis_amd/build.py).  The extension makes the library's C-ABI calls itself,
so libnaylis_mom.so is loaded first (with global visibility, _lib.load) and
the extension binds to that instance."""
from __future__ import annotations

import importlib.util
import os
import threading

import torch

from . import _lib

EXT_PATH = os.path.join(_lib.LIB_DIR, "ext", "naylis_torch.so")

_mod = None
_lock = threading.Lock()


class _TracedCall(torch.autograd.Function):
    """An extension call as one node of a torch.jit.trace graph.  The tracer
    sees neither C++ autograd functions nor kernel launches and would keep the
    outputs as constants; a Python function it records and runs again.  The
    last argument, the stream, is the one current at each run."""

    @staticmethod
    def forward(ctx, name, spec, *tensors):
        leaves = [t.detach().requires_grad_(t.requires_grad) for t in tensors]
        it = iter(leaves)
        args = [[next(it) for _ in c] if k == "list" else next(it) if k == "tensor" else c for k, c in spec]
        args[-1] = _lib.stream_of(leaves[0].device)
        with torch.enable_grad():
            outs = getattr(_mod, name)(*args)
        ctx.single = isinstance(outs, torch.Tensor)
        ctx.leaves, ctx.outs = leaves, (outs,) if ctx.single else tuple(outs)
        ctx.set_materialize_grads(False)
        res = tuple(o.detach() for o in ctx.outs)
        return res[0] if ctx.single else res

    @staticmethod
    def backward(ctx, *grads):
        pairs = [(o, g) for o, g in zip(ctx.outs, grads) if g is not None and o.requires_grad]
        ins = [t for t in ctx.leaves if t.requires_grad]
        got = iter(torch.autograd.grad([o for o, _ in pairs], ins, [g for _, g in pairs], retain_graph=True,
                                       allow_unused=True) if pairs else [None] * len(ins))
        return (None, None, *(next(got) if t.requires_grad else None for t in ctx.leaves))


class _Traced:
    """The extension's functions while torch.jit.trace runs."""

    def __getattr__(self, name):
        def call(*args):
            spec, tensors = [], []
            for a in args:
                if isinstance(a, torch.Tensor):
                    spec.append(("tensor", None))
                    tensors.append(a)
                elif isinstance(a, list):
                    spec.append(("list", [None] * len(a)))
                    tensors.extend(a)
                else:
                    spec.append(("value", a))
            return _TracedCall.apply(name, spec, *tensors)
        return call


def load():
    """Load (once) and return the extension module; raises if it is not built.
    Under torch.jit.trace its functions come wrapped for the tracer."""
    if torch._C._get_tracing_state() is not None:
        _load()
        return _Traced()
    return _mod if _mod is not None else _load()


def _load():
    global _mod
    if _mod is not None:
        return _mod
    with _lock:
        if _mod is not None:
            return _mod
        _lib.load()
        if not os.path.exists(EXT_PATH):
            raise RuntimeError(
                f"naylis_amd: torch extension not built ({EXT_PATH} missing). "
                "Run `python -c 'import __graft_entry__ as g; g.build()'` or `python -m naylis_amd.build` first.")
        spec = importlib.util.spec_from_file_location("naylis_torch", EXT_PATH)
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        _mod = mod
        return mod
