"""The Python entry points' short way into the library (sentinel_amd/csrc/torch_calls.cpp), built for host tensors and bound to
functions that only count their calls: what it must decline, what it must not swallow."""
import ctypes
import importlib.machinery
import importlib.util
import os
import subprocess
import sys

import pytest
import torch

from sentinel_amd import build, flash_attention

HERE = os.path.dirname(os.path.abspath(__file__))
MODULE = os.path.join(HERE, "cpp", "_torch_calls.so")
INT, FLOAT, POINTER, SIZE = ctypes.c_int, ctypes.c_float, ctypes.c_void_p, ctypes.c_size_t


def built():
    source = os.path.join(build.CSRC, "torch_calls.cpp")
    if not os.path.exists(MODULE) or os.path.getmtime(MODULE) < os.path.getmtime(source):
        build.compile_calls(MODULE, ["-DSENTINEL_CALLS_HOST_TENSORS", "-O0"])
    loader = importlib.machinery.ExtensionFileLoader("_torch_calls", MODULE)
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_torch_calls", loader))
    loader.exec_module(module)
    return module


class Library:
    """Stands for the library: every call returns `code` and is counted under its name."""
    SIGNATURES = {
        "flash_fwd": [POINTER] * 5 + [INT] * 10 + [FLOAT, INT, POINTER, SIZE, POINTER],
        "flash_bwd": [POINTER] * 10 + [INT] * 10 + [FLOAT, INT, POINTER, SIZE, POINTER],
        "flash_fwd_rope": [POINTER] * 7 + [INT] * 12 + [FLOAT, INT, POINTER, SIZE, POINTER],
        "flash_bwd_rope": [POINTER] * 12 + [INT] * 12 + [FLOAT, INT, POINTER, SIZE, POINTER],
        "flash_fwd_sparse": [POINTER] * 7 + [INT] * 14 + [FLOAT, INT, POINTER, SIZE, POINTER],
        "flash_bwd_sparse": [POINTER] * 12 + [INT] * 14 + [FLOAT, INT, POINTER, SIZE, POINTER],
        "decode_attention": [POINTER] * 4 + [INT] * 5 + [FLOAT, INT, INT, POINTER, SIZE, POINTER],
        "dense_softmax_fwd": [POINTER, INT, ctypes.c_longlong] + [INT] * 6 + [FLOAT, POINTER],
        "dense_softmax_bwd": [POINTER, ctypes.c_longlong, POINTER, ctypes.c_longlong] + [INT] * 7 + [FLOAT, POINTER],
        "rope_rotate": [POINTER] + [INT] * 7 + [POINTER, POINTER, INT, INT, POINTER],
    }

    def __init__(self):
        self.code, self.calls, self.workspace_bytes, self.functions = 0, [], 0, {}
        for name, arguments in self.SIGNATURES.items():
            self._add(name, INT, arguments, lambda *_, name=name: (self.calls.append(name), self.code)[1])
        self._add("flash_workspace_bytes", SIZE, [INT] * 9, lambda *_: self.workspace_bytes)
        self._add("decode_workspace_bytes", SIZE, [INT] * 3, lambda *_: self.workspace_bytes)
        self.message = ctypes.create_string_buffer(b"what went wrong")
        self._add("last_error", POINTER, [], lambda: ctypes.addressof(self.message))

    def _add(self, name, result, arguments, function):
        self.functions["sentinel_hip_" + name] = ctypes.CFUNCTYPE(result, *arguments)(function)

    def addresses(self):
        return {name: ctypes.cast(f, POINTER).value for name, f in self.functions.items()}


@pytest.fixture(scope="module")
def module():
    return built()


@pytest.fixture
def library(module):
    lib = Library()
    module.bind(lib.addresses())
    return lib


def native(**replaced):
    """arguments of a native_forward call"""
    args = dict(q=torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16), k=torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16),
                v=torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16), out=torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16),
                lse=torch.zeros(1, 4, 8), scale=0.125, causal=True, window=0, global_tokens=0)
    args.update(replaced)
    return tuple(args.values())


def decode(**replaced):
    args = dict(q=torch.zeros(64, 1), k=torch.zeros(32, 16), v=torch.zeros(32, 16), out=torch.zeros(64, 1), length=10, heads=4, head_dim=16,
                kv_heads=2, scale=0.25, window=0, global_tokens=0, workspace=None)
    args.update(replaced)
    return tuple(args.values())


def test_expected_calls_are_made(module, library):
    assert module.native_forward(*native()) is True
    assert module.native_forward(*native(window=3)) is True
    assert module.decode(*decode()) is True
    assert library.calls == ["flash_fwd", "flash_fwd_sparse", "decode_attention"]


class Subclass(torch.Tensor):
    pass


@pytest.mark.parametrize("replaced", [
    dict(q=torch.zeros(1, 4, 8, 64)),                                                         # another type than the others
    dict(k=torch.zeros(1, 2, 9, 64, dtype=torch.bfloat16)),                                   # another length
    dict(out=torch.zeros(1, 4, 64, 8, dtype=torch.bfloat16).transpose(2, 3)),                 # not contiguous
    dict(q=torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16).as_subclass(Subclass)),
    dict(out=torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16, device="meta")),                  # another device
    dict(lse=torch.zeros(1, 4, 9)),
    dict(out=None),
    dict(q=torch.zeros(1, 4, 8, 64, dtype=torch.bfloat16).to_sparse()),
    dict(scale=1),
    dict(causal=1),
    dict(window=2 ** 40),
    dict(global_tokens=None),
])
def test_anything_else_is_declined(module, library, replaced):
    assert module.native_forward(*native(**replaced)) is False
    assert library.calls == []


def test_a_short_workspace_is_declined(module, library):
    library.workspace_bytes = 64
    assert module.decode(*decode()) is False
    assert module.decode(*decode(workspace=torch.zeros(63, dtype=torch.uint8))) is False
    assert library.calls == []
    assert module.decode(*decode(workspace=torch.zeros(64, dtype=torch.uint8))) is True


@pytest.mark.parametrize("code", [flash_attention.INVALID_ARGUMENT, flash_attention.UNSUPPORTED])
def test_refused_arguments_go_back_to_python(module, library, code):
    library.code = code
    assert module.decode(*decode()) is False
    assert module.native_forward(*native()) is False


def in_place_calls(module):
    scores, gradient, tables = torch.zeros(8, 8), torch.zeros(8, 8), torch.zeros(8, 4)
    return {"dense_softmax_fwd": lambda: module.softmax_forward(scores, 1.0, 0, 0, 0, 0),
            "dense_softmax_bwd": lambda: module.softmax_backward(scores, gradient, 1.0, 0, 0, 0, 0),
            "rope_rotate": lambda: module.rotate(scores, 1, 8, 4, tables, tables, 0, 0, False),
            "decode_attention": lambda: module.decode(*decode()),
            "flash_fwd": lambda: module.native_forward(*native())}


@pytest.mark.parametrize("name", ["dense_softmax_fwd", "dense_softmax_bwd", "rope_rotate", "decode_attention", "flash_fwd"])
def test_a_runtime_error_is_raised_and_not_tried_again(module, library, name):
    # the launch may have gone through: a second one would work on the first one's result
    call = in_place_calls(module)[name]
    assert call() is True
    library.calls.clear()
    library.code = flash_attention.RUNTIME
    with pytest.raises(RuntimeError, match="what went wrong"):
        call()
    assert library.calls == [name]


def test_tensors_without_storage_are_declined():
    """In a process of its own: an exception that leaves the extension ends it."""
    script = """
import sys
sys.path.insert(0, %r)
import torch
import test_torch_calls as t
module, library = t.built(), t.Library()
module.bind(library.addresses())
answers = []
def call(q):
    answers.append(module.decode(*t.decode(q=q)))
    return q
torch.func.vmap(call)(torch.zeros(3, 64, 1))
def scores(x):
    answers.append(module.softmax_forward(x, 1.0, 0, 0, 0, 0))
    return x.sum()
torch.func.vmap(scores)(torch.zeros(3, 4, 4))
torch.func.grad(scores)(torch.zeros(4, 4))
print("answers", answers, library.calls)
""" % HERE
    built()
    run = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=300, cwd=os.path.dirname(HERE),
                         env={**os.environ, "PYTHONPATH": os.path.dirname(HERE)})
    assert run.returncode == 0, run.stderr
    assert "answers [False, False, False] []" in run.stdout
