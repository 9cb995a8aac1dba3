"""The library's host side with a recording stand-in for the HIP runtime (tests/native/launch_record.cpp): which kernels a
call launches, on the CPU and for operands that no memory could hold.  Nothing runs on a GPU and no operand is read."""
from __future__ import annotations

import ctypes
from pathlib import Path
from typing import NamedTuple

import emel_hip as eh
from emel_hip.abi import SIGNATURES

LIB = Path(__file__).resolve().parent / "native" / "libemel_record.so"


class Launch(NamedTuple):
    name: str
    grid: int
    block: int
    lds: int


class Recorder:
    def __init__(self):
        if not LIB.exists():
            raise RuntimeError(f"{LIB} missing: run __graft_entry__.build()")
        self.lib = ctypes.CDLL(str(LIB))
        for name, argtypes in SIGNATURES.items():
            getattr(self.lib, name).argtypes = argtypes
            getattr(self.lib, name).restype = ctypes.c_int
        for name in ("count", "grid", "block", "lds"):
            getattr(self.lib, "record_" + name).restype = ctypes.c_uint64
            getattr(self.lib, "record_" + name).argtypes = [] if name == "count" else [ctypes.c_uint64]
        self.lib.record_name.restype = ctypes.c_char_p
        self.lib.record_name.argtypes = [ctypes.c_uint64]
        self.lib.emel_last_error.restype = ctypes.c_char_p

    def launches(self, event) -> list:
        """What an accepted event launches; a refused one raises."""
        self.lib.record_clear()
        status = eh.Status(event._call(self.lib, None))
        if status != eh.Status.OK:
            raise RuntimeError(f"{status.name}: {self.lib.emel_last_error().decode()}")
        get = self.lib
        return [Launch(get.record_name(i).decode(), get.record_grid(i), get.record_block(i), get.record_lds(i))
                for i in range(get.record_count())]


def view(slot: int, ne, nb=None, dtype=eh.DType.F32, mut=False, offset=0):
    """A view at an address of its own (`slot`, 8 TiB apart), `offset` bytes past a 16-byte boundary."""
    lay = eh.Layout.dense(dtype, ne) if nb is None else eh.Layout(dtype, ne, nb)
    return (eh.TensorViewMut if mut else eh.TensorView)((slot + 1) * (1 << 43) + offset, lay, 1 << 43)
