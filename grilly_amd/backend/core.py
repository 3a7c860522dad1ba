"""Device context and buffers: the part of the reference's VulkanCore that the hot path uses
(backend/core.py:304-421: create / upload / download buffer, dispatch + wait), on HIP.

One HipCore = one gfx950 device + one HIP stream + one caching buffer pool, all inside
libgrilly_hip.so.  numpy arrays are copied in and out; nothing here computes.
"""
import ctypes
import functools

import numpy as np

from .. import _lib as L

_DT = {"fp32": L.GRL_F32, "float32": L.GRL_F32, "f32": L.GRL_F32, "bf16": L.GRL_BF16, "bfloat16": L.GRL_BF16}


def dtype_code(dtype):
    try:
        return _DT[dtype]
    except KeyError:
        raise ValueError(f"dtype must be 'fp32' or 'bf16', got {dtype!r}") from None


def dtype_size(code):
    return 2 if code == L.GRL_BF16 else 4


def host_f32(a):
    """a C-contiguous float32 array of a's values (a itself where it is one)"""
    return np.ascontiguousarray(a, dtype=np.float32)


RECYCLED_MIN = 32 << 20         # smaller results: the C library recycles their memory itself


@functools.lru_cache(maxsize=None)
def _result_allocator(lib):
    """(numpy's PyDataMem_SetHandler, the library's allocator as numpy takes one), or None where numpy has no such interface
    (before 1.22)"""
    api = getattr(getattr(np, "_core", None) or np.core, "_multiarray_umath")._ARRAY_API
    pointer, new = ctypes.pythonapi.PyCapsule_GetPointer, ctypes.pythonapi.PyCapsule_New
    pointer.restype, pointer.argtypes = ctypes.c_void_p, [ctypes.py_object, ctypes.c_char_p]
    new.restype, new.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
    table = ctypes.cast(pointer(api, None), ctypes.POINTER(ctypes.c_void_p))
    # slots of numpy's C interface (numpy/__multiarray_api.h): PyArray_GetNDArrayCFeatureVersion, PyDataMem_SetHandler
    if ctypes.PYFUNCTYPE(ctypes.c_uint)(table[211])() < 0x0F:
        return None
    set_handler = ctypes.PYFUNCTYPE(ctypes.py_object, ctypes.py_object)(table[304])
    return set_handler, new(lib.grl_numpy_handler(), b"mem_handler", None)


def result_array(lib, shape):
    """uninitialised float32 array for a result, numpy's own in every respect; a large one stands in recycled memory, whose
    pages the process has already.  numpy keeps its allocator in a context variable, so no other thread or task sees it."""
    nbytes = 4
    for n in shape:
        nbytes *= int(n)
    recycled = _result_allocator(lib) if nbytes >= RECYCLED_MIN else None
    if recycled is None:
        return np.empty(shape, dtype=np.float32)
    set_handler, handler = recycled
    usual = set_handler(handler)
    try:
        return np.empty(shape, dtype=np.float32)
    finally:
        set_handler(usual)


class DeviceBuffer:
    """A pool-owned device allocation; returned to the pool by free() or when collected."""
    __slots__ = ("core", "ptr", "nbytes", "__weakref__")

    def __init__(self, core, nbytes):
        self.core = core
        self.nbytes = int(nbytes)
        self.ptr = core.lib.grl_malloc(core.ctx, max(self.nbytes, 1))
        if not self.ptr:
            raise MemoryError(L.last_error())

    def free(self):
        if self.ptr and self.core.ctx:
            self.core.lib.grl_free(self.core.ctx, self.ptr)
        self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.free()


class HipCore:
    def __init__(self, device=0):
        self.lib = L.load()
        self.ctx = self.lib.grl_create(int(device))
        if not self.ctx:
            # same exception type as the reference when its device layer is absent (backend/core.py:18-19)
            raise RuntimeError(f"HIP device not available: {L.last_error()}")
        self.device = int(device)

    # ---- lifetime
    def cleanup(self):
        if self.ctx:
            self.lib.grl_destroy(self.ctx)
            self.ctx = None

    def __del__(self):
        try:
            self.cleanup()
        except Exception:
            pass

    # ---- info
    def device_info(self):
        d = L.DevInfo()
        L.check(self.lib.grl_device_info(self.ctx, ctypes.byref(d)), "device_info")
        return {"name": d.name.decode(), "arch": d.arch.decode(), "compute_units": d.compute_units,
                "clock_khz": d.clock_khz, "lds_bytes_per_block": d.lds_bytes_per_block,
                "wavefront": d.wavefront, "hbm_bytes": d.hbm_bytes}

    def pool_stats(self):
        s = L.PoolStats()
        L.check(self.lib.grl_pool_get_stats(self.ctx, ctypes.byref(s)), "pool_stats")
        total = s.hits + s.misses
        return {"allocations": s.allocations, "hits": s.hits, "misses": s.misses, "bytes_in_use": s.bytes_in_use,
                "bytes_cached": s.bytes_cached, "bytes_peak": s.bytes_peak,
                "hit_rate": (s.hits / total) if total else 0.0}

    # ---- buffers
    def alloc(self, nbytes):
        return DeviceBuffer(self, nbytes)

    def upload(self, arr, code=L.GRL_F32):
        """numpy (any dtype, any strides) -> fresh device buffer holding fp32 or bf16 values.
        bf16 is rounded (to nearest even) on the way."""
        a = np.ascontiguousarray(arr, dtype=np.float32)
        buf = self.alloc(a.size * dtype_size(code))
        L.check(self.lib.grl_upload(self.ctx, code, a.size, a.ctypes.data, buf.ptr), "upload")
        return buf

    def upload_raw(self, arr):
        """numpy array copied byte-for-byte (int32 ids, fp32 vectors, pre-packed bf16 bits)."""
        a = np.ascontiguousarray(arr)
        buf = self.alloc(a.nbytes)
        L.check(self.lib.grl_h2d(self.ctx, buf.ptr, a.ctypes.data, a.nbytes), "upload")
        return buf

    def download(self, buf, shape, code=L.GRL_F32):
        """device buffer of fp32 or bf16 values -> fresh C-contiguous float32 numpy array."""
        n = int(np.prod(shape)) if len(shape) else 1
        out = result_array(self.lib, shape)
        L.check(self.lib.grl_download(self.ctx, code, n, buf.ptr, out.ctypes.data), "download")
        return out

    def sync(self):
        L.check(self.lib.grl_sync(self.ctx), "sync")

    def timer_start(self):
        L.check(self.lib.grl_timer_start(self.ctx), "timer_start")

    def timer_stop(self):
        ms = ctypes.c_float()
        L.check(self.lib.grl_timer_stop(self.ctx, ctypes.byref(ms)), "timer_stop")
        return float(ms.value)

    def clock_probe_begin(self, millis):
        """start the shader-clock probe: it runs for `millis` (held within the library's (0, 500] ms range) beside
        whatever is enqueued next"""
        L.check(self.lib.grl_clock_probe_begin(self.ctx, min(max(float(millis), 0.05), 500.0)), "clock_probe_begin")

    def clock_probe_end(self):
        """wait for the probe; average shader clock in GHz while it ran"""
        ghz = ctypes.c_float()
        L.check(self.lib.grl_clock_probe_end(self.ctx, ctypes.byref(ghz)), "clock_probe_end")
        return float(ghz.value)
