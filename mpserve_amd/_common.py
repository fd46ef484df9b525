"""Helpers shared by the op modules: the current stream's handle, the reference's
contiguity check (decode_huffman.cu:59-63) and the device integrity word."""
from __future__ import annotations

import ctypes
import os
from typing import Dict, Optional

import torch

from . import _native


def _stream_handle(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _check_cuda_contig(t: torch.Tensor, name: str, device: torch.device | None) -> None:
    # decode_huffman.cu:59-63
    if t is None:
        raise ValueError(f"{name} must be defined")
    if not t.is_cuda:
        raise ValueError(f"{name} must be a CUDA tensor")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")
    if device is not None and t.device != device:
        raise ValueError(f"{name} must be on {device}, got {t.device}")


def read_status(device: torch.device | None = None) -> int:
    """MPS_STATUS_* flags recorded by decodes on ``device`` since the last read (synchronises)."""
    device = torch.device("cuda", torch.cuda.current_device()) if device is None else device
    v = ctypes.c_uint32(0)
    _native.check(_native.lib().mps_fp8_read_status(device.index or 0, ctypes.c_void_p(_stream_handle(device)),
                                                    ctypes.byref(v)))
    return int(v.value)


def _maybe_check_status(device: torch.device, op: str = "huffman_decode_fp8") -> None:
    """With MPSERVE_DECODE_CHECK=1: synchronise and raise if the decode flagged the sidecar."""
    if os.environ.get("MPSERVE_DECODE_CHECK", "0") == "1":
        st = read_status(device)
        if st:
            raise RuntimeError(f"{op}: sidecar integrity flags 0x{st:x} "
                               "(1=bucket range, 2=row index, 4=table id, 8=lane bit desync)")


class BuilderOutputs:
    """A sidecar builder's device memory, from torch's allocator: the outputs it asks for by
    slot and its workspaces, all on ``device`` and of the current stream (whose order makes
    it safe to drop the workspaces when the call returns)."""

    def __init__(self, device: torch.device, dtypes: Dict[int, torch.dtype]):
        self._device, self._dtypes = device, dtypes
        self._out: Dict[int, torch.Tensor] = {}
        self._work: list = []
        self._error: Optional[BaseException] = None

    def _alloc(self, _ctx, slot: int, nbytes: int):
        try:
            dtype = self._dtypes.get(slot, torch.uint8)
            t = torch.empty(nbytes // dtype.itemsize, dtype=dtype, device=self._device)
            if slot >= 0:
                self._out[slot] = t
            else:
                self._work.append(t)
            return t.data_ptr()
        except BaseException as e:  # raised again once the native call has returned
            self._error = e
            return None

    def build(self, entry, args, stream: int):
        """Runs ``entry`` (mps_*_encode_alloc); (sizes, stats) of its outputs."""
        sizes, stats = (ctypes.c_int64 * 17)(), (ctypes.c_int64 * 4)()
        rc = entry(ctypes.byref(args), ctypes.c_void_p(stream), _native.ENCODE_ALLOC(self._alloc), None, sizes, stats)
        error, self._error = self._error, None
        if error is not None or rc != 0:
            # The stream is idle. The error's traceback holds _alloc's frame and so this object:
            # it must hold neither the error (a cycle) nor the build's memory, which a caller
            # that tries again would find still taken.
            self._out.clear()
            self._work.clear()
        if error is not None:
            try:
                raise error
            finally:
                del error
        _native.check(rc)
        return sizes, stats

    def complete(self) -> None:
        """Waits for the build's last passes: its outputs and inputs may then be used, rewritten
        or freed on any stream (as after the reference's host builders). Called with the result
        made up, so that the passes run beside that work (14336 x 4096: 547 us a build; waiting in the
        native call 565; not waiting, which raced with work on other streams, 515)."""
        torch.cuda.current_stream(self._device).synchronize()

    def tensor(self, slot: int, shape, on_host: bool) -> torch.Tensor:
        t = self._out.get(slot)
        if t is None:
            t = torch.empty(0, dtype=self._dtypes[slot], device=self._device)
        return t.view(shape).cpu() if on_host else t.view(shape)
