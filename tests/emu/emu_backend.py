"""Test-only: the package's operators bound to the CPU build of the kernel sources (libgdn_emu.so).

This exists so that kernel indexing, LDS use and barriers can be checked on a machine without a GPU, with
guard pages instead of GPU faults.  The shipped package never imports this module."""
import contextlib
import ctypes
import os
import shutil
import sys

import torch

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
for p in (ROOT, os.path.join(ROOT, "mindspeed-mm_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

from mindspeed_mm_amd._lib import DTYPE_CODE, GdnLibrary  # noqa: E402
from mindspeed_mm_amd.ops import GdnOps  # noqa: E402

_ops = {}


def emu_ops(compute_units=None) -> GdnOps:
    """The operators on the CPU build.  compute_units: on a copy of the library whose device has that many (the launchers
    ask once per library); results are the same, the choice of launches is that of a device of this size."""
    if compute_units not in _ops:
        from . import build_emu
        path = build_emu.build()
        if compute_units is not None:
            copy = f"{path[:-3]}_{compute_units}.so"
            shutil.copyfile(path, copy)
            path = copy
        ops = GdnOps(GdnLibrary(path, "cpu"))
        ops.lib.cdll.emu_guard_alloc.restype = ctypes.c_void_p
        ops.lib.cdll.emu_guard_alloc.argtypes = [ctypes.c_size_t, ctypes.c_int]
        if compute_units is not None:
            os.environ["GDN_EMU_COMPUTE_UNITS"] = str(compute_units)
            try:
                ops.lib.gdn_chunk_workspace_bytes(1, 64, 1, 1, 1, 128, 128, DTYPE_CODE[torch.bfloat16], 0)
            finally:
                del os.environ["GDN_EMU_COMPUTE_UNITS"]
        _ops[compute_units] = ops
    return _ops[compute_units]


_keep = []


def guarded(t: torch.Tensor, at_end: bool = True) -> torch.Tensor:
    """Copy of `t` whose storage ends (or starts) flush against an inaccessible page."""
    lib = emu_ops().lib.cdll
    t = t.contiguous()
    nbytes = max(t.numel() * t.element_size(), 1)
    p = lib.emu_guard_alloc(nbytes, 1 if at_end else 0)
    buf = (ctypes.c_uint8 * nbytes).from_address(p)
    _keep.append(buf)
    raw = torch.frombuffer(buf, dtype=torch.uint8, count=nbytes)
    out = raw[: t.numel() * t.element_size()].view(t.dtype).view(t.shape)
    out.copy_(t)
    return out


@contextlib.contextmanager
def guarded_outputs():
    """While active, every CPU tensor made by torch.empty (the operators allocate their outputs, gradients and
    workspaces with it) ends flush against an inaccessible page, so that a kernel reading or writing past the end of
    an output is a SIGSEGV here."""
    real = torch.empty

    def empty(*size, **kw):
        t = real(*size, **kw)
        return guarded(t) if t.device.type == "cpu" and t.numel() > 0 and not kw.get("pin_memory") else t
    torch.empty = empty
    try:
        yield
    finally:
        torch.empty = real
