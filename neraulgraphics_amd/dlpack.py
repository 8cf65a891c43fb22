"""Zero-copy views of the backend's device buffers as DLPack capsules, for torch.from_dlpack.

The capsule's manager keeps its owner (the renderer) alive until the consumer releases the tensor, which
is how the reference's Python edge hands out its buffers (python/bindings.cpp:192-202)."""
import ctypes
import functools

import numpy as np

kDLROCM = 10
_CODES = {np.float32: (2, 32), np.int32: (0, 32), np.uint8: (1, 8)}


class DLDevice(ctypes.Structure):
    _fields_ = [("device_type", ctypes.c_int32), ("device_id", ctypes.c_int32)]


class DLDataType(ctypes.Structure):
    _fields_ = [("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16)]


class DLTensor(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("device", DLDevice), ("ndim", ctypes.c_int32), ("dtype", DLDataType),
                ("shape", ctypes.POINTER(ctypes.c_int64)), ("strides", ctypes.POINTER(ctypes.c_int64)),
                ("byte_offset", ctypes.c_uint64)]


_DELETER = ctypes.CFUNCTYPE(None, ctypes.c_void_p)


class DLManagedTensor(ctypes.Structure):
    _fields_ = [("dl_tensor", DLTensor), ("manager_ctx", ctypes.c_void_p), ("deleter", _DELETER)]


_live = {}  # address of a DLManagedTensor -> (struct, shape array, owner)


@_DELETER
def _release(address):
    _live.pop(address, None)


_PyCapsule_New = ctypes.pythonapi.PyCapsule_New
_PyCapsule_New.restype = ctypes.py_object
_PyCapsule_New.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]


_SHAPE = [ctypes.c_int64 * n for n in range(6)]


def capsule(pointer, shape, dtype, device_id, owner):
    """A 'dltensor' capsule viewing `pointer` (device memory) as a C-contiguous array."""
    code, bits = _CODES.get(dtype) or _CODES[np.dtype(dtype).type]
    n = len(shape)
    shp = _SHAPE[n](*shape) if n < len(_SHAPE) else (ctypes.c_int64 * n)(*shape)
    mt = DLManagedTensor((pointer, (kDLROCM, device_id), n, (code, bits, 1), shp, None, 0), None, _release)
    address = ctypes.addressof(mt)
    _live[address] = (mt, shp, owner)
    return _PyCapsule_New(address, b"dltensor", None)


@functools.lru_cache(maxsize=None)
def _from_dlpack():
    from torch.utils.dlpack import from_dlpack
    return from_dlpack


def to_torch(pointer, shape, dtype, device_id, owner):
    return _from_dlpack()(capsule(pointer, shape, dtype, device_id, owner))
