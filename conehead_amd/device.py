"""Device buffers, streams and events on top of the C-ABI.

The library allocates HBM itself (ch_malloc); numpy arrays are the host side.
"""
import collections
import ctypes
import threading
import weakref

import numpy as np

from . import _lib


_POOLS = weakref.WeakSet()   # the pools alive, for trim_pools


def register_pool(pool):
    _POOLS.add(pool)


def trim_pools():
    """Frees what every pool of this process holds idle; returns its size."""
    freed = 0
    for pool in list(_POOLS):
        freed += pool._bytes
        pool.clear()
    return freed


def allocate(call):
    """Checks the status of `call`, which allocates; where memory is short it
    is called again without the idle buffers of the pools."""
    st = call()
    if st == _lib.CH_ERR_NOMEM and trim_pools() > 0:
        st = call()
    return _lib.check(st)


class Stream:
    """A HIP stream (default priority)."""

    def __init__(self, handle=None):
        self._own = handle is None
        if handle is None:
            h = ctypes.c_void_p()
            _lib.check(_lib.lib().ch_stream_create(ctypes.byref(h)))
            handle = h.value
        self.handle = handle

    def sync(self):
        _lib.check(_lib.lib().ch_stream_sync(self.handle))

    def wait(self, event):
        """Later work on this stream waits for `event`."""
        _lib.check(_lib.lib().ch_stream_wait(self.handle, event.handle))

    def close(self):
        if self._own and self.handle:
            _lib.lib().ch_stream_destroy(self.handle)
        self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


NULL_STREAM = None


def _h(stream):
    return stream.handle if isinstance(stream, Stream) else stream


def arm_launch_events(start, stop):
    """The calling thread's next gather or scatter launch records `start`
    and `stop` (Events) right around its kernel (ch_set_launch_events)."""
    _lib.check(_lib.lib().ch_set_launch_events(start.handle, stop.handle))


class Event:
    def __init__(self):
        h = ctypes.c_void_p()
        _lib.check(_lib.lib().ch_event_create(ctypes.byref(h)))
        self.handle = h.value

    def record(self, stream=None):
        _lib.check(_lib.lib().ch_event_record(self.handle, _h(stream)))
        return self

    def sync(self):
        _lib.check(_lib.lib().ch_event_sync(self.handle))

    def done(self):
        d = ctypes.c_int32()
        _lib.check(_lib.lib().ch_event_query(self.handle, ctypes.byref(d)))
        return bool(d.value)

    def elapsed_ms(self, later):
        ms = ctypes.c_float()
        _lib.check(_lib.lib().ch_event_elapsed(ctypes.byref(ms), self.handle,
                                               later.handle))
        return float(ms.value)

    def __del__(self):
        try:
            if self.handle:
                _lib.lib().ch_event_destroy(self.handle)
        except Exception:
            pass


class DeviceArray:
    """An HBM allocation with a numpy-like shape and dtype."""

    def __init__(self, shape, dtype=np.float32, zero=False, stream=None):
        self.shape = tuple(int(s) for s in np.atleast_1d(shape)) \
            if not isinstance(shape, tuple) else tuple(int(s) for s in shape)
        self.dtype = np.dtype(dtype)
        self.nbytes = int(np.prod(self.shape, dtype=np.int64)) * \
            self.dtype.itemsize
        p = ctypes.c_void_p()
        L = _lib.lib()
        allocate(lambda: L.ch_malloc(ctypes.byref(p), self.nbytes))
        self.ptr = p.value
        if zero:
            self.zero(stream)

    @classmethod
    def from_host(cls, arr, dtype=None, stream=None):
        a = np.ascontiguousarray(arr, dtype=dtype or np.asarray(arr).dtype)
        d = cls(a.shape, a.dtype)
        d.upload(a, stream)
        return d

    @property
    def size(self):
        return int(np.prod(self.shape, dtype=np.int64))

    def upload(self, arr, stream=None):
        a = np.ascontiguousarray(arr, dtype=self.dtype)
        if a.nbytes != self.nbytes:
            raise ValueError("upload of %d bytes into %d" %
                             (a.nbytes, self.nbytes))
        _lib.check(_lib.lib().ch_memcpy_h2d(self.ptr, a.ctypes.data,
                                            self.nbytes, _h(stream)))
        if stream is not None:
            # pageable source: make sure the copy has consumed it
            _lib.check(_lib.lib().ch_stream_sync(_h(stream)))
        return self

    def download(self, out=None, stream=None):
        if out is None:
            out = np.empty(self.shape, self.dtype)
        if not out.flags.c_contiguous or out.nbytes != self.nbytes or \
                out.dtype != self.dtype:
            raise ValueError("download target must be a contiguous %s %s" %
                             (self.dtype, self.shape))
        _lib.check(_lib.lib().ch_memcpy_d2h(out.ctypes.data, self.ptr,
                                            self.nbytes, _h(stream)))
        return out

    def download_async(self, host, offset=0, stream=None):
        """Queues a copy into the pinned HostBuffer `host` at byte `offset`;
        the data is there once an event recorded after it has completed."""
        if offset < 0 or offset + self.nbytes > host.nbytes:
            raise ValueError("download_async: %d bytes at %d into %d" %
                             (self.nbytes, offset, host.nbytes))
        _lib.check(_lib.lib().ch_memcpy_d2h_async(host.ptr + offset,
                                                  self.ptr, self.nbytes,
                                                  _h(stream)))

    def zero(self, stream=None):
        _lib.check(_lib.lib().ch_zero(self.ptr, self.nbytes, _h(stream)))
        return self

    def free(self):
        if self.ptr:
            _lib.lib().ch_free(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass

    def __repr__(self):
        return "DeviceArray(%s, %s, 0x%x)" % (self.shape, self.dtype,
                                             self.ptr or 0)


def mem_info():
    f = ctypes.c_size_t()
    t = ctypes.c_size_t()
    _lib.check(_lib.lib().ch_mem_info(ctypes.byref(f), ctypes.byref(t)))
    return f.value, t.value


def device_sync():
    _lib.check(_lib.lib().ch_device_sync())


class HostBuffer:
    """Pinned host memory (ch_host_alloc): the target of asynchronous
    device-to-host copies."""

    def __init__(self, nbytes):
        self.nbytes = int(nbytes)
        p = ctypes.c_void_p()
        L = _lib.lib()
        allocate(lambda: L.ch_host_alloc(ctypes.byref(p), self.nbytes))
        self.ptr = p.value

    def free(self):
        if self.ptr:
            _lib.lib().ch_host_free(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


# The idle buffers of a pool (_free: key -> list, least recently used key
# first; _bytes: what they hold; _max: what they may), its lock held.

def take_idle(pool, key):
    lst = pool._free.get(key)
    if not lst:
        return None
    buf = lst.pop()
    pool._bytes -= buf.nbytes
    if not lst:
        del pool._free[key]
    return buf


def drop_idle(pool, limit):
    """Frees idle buffers until they hold at most `limit` bytes."""
    while pool._free and pool._bytes > limit:
        key = next(iter(pool._free))
        take_idle(pool, key).free()


def keep_idle(pool, key, buf):
    """Adds a buffer, making room for it: with the newest refused instead, a
    pool full of earlier shapes would allocate every later one anew."""
    if buf.nbytes > pool._max:
        buf.free()
        return
    drop_idle(pool, pool._max - buf.nbytes)
    pool._free.setdefault(key, []).append(buf)
    pool._free.move_to_end(key)
    pool._bytes += buf.nbytes


class _PinnedView:
    """Owner of a HostBuffer while numpy arrays view it; gives the buffer
    back to its pool when the last array is dropped."""

    def __init__(self, buf, pool, shape, dtype):
        self._buf = buf
        self._pool = pool
        dt = np.dtype(dtype)
        self.__array_interface__ = {
            "shape": tuple(shape), "typestr": dt.str,
            "data": (buf.ptr, False), "version": 3}

    def __del__(self):
        try:
            self._pool.put(self._buf)
        except Exception:
            pass


class HostPool:
    """Reusable pinned host buffers keyed by size.  as_array() hands a buffer
    out as a numpy array that owns it: the buffer returns to the pool when
    that array (and every view of it) is gone, so results are delivered
    without a host-side copy.

    Idle buffers hold at most max_free_bytes; those of the size least
    recently used go first.  max_bytes bounds all buffers of the pool, handed
    out or idle, for try_get."""

    def __init__(self, max_free_bytes=4 << 30, max_bytes=None):
        self._free = collections.OrderedDict()
        self._bytes = 0
        self._max = max_free_bytes
        self._max_alive = max_bytes
        self._alive = weakref.WeakSet()
        self._lock = threading.RLock()
        register_pool(self)

    def get(self, nbytes):
        with self._lock:
            b = take_idle(self, int(nbytes))
        if b is None:
            b = HostBuffer(nbytes)
            with self._lock:
                self._alive.add(b)
        return b

    def try_get(self, nbytes):
        """A buffer, or None where it would take the pool past max_bytes
        (idle buffers make room) or no pinned memory is to be had."""
        with self._lock:
            if self._max_alive is not None and int(nbytes) not in self._free:
                out = sum(b.nbytes for b in self._alive if b.ptr) - \
                    self._bytes
                if out + nbytes > self._max_alive:
                    return None
                drop_idle(self, self._max_alive - out - nbytes)
        try:
            return self.get(nbytes)
        except _lib.CHError:
            return None

    def put(self, buf):
        with self._lock:
            keep_idle(self, buf.nbytes, buf)

    def as_array(self, buf, shape, dtype=np.float32):
        if int(np.prod(shape)) * np.dtype(dtype).itemsize > buf.nbytes:
            raise ValueError("as_array: %s %s does not fit %d bytes" %
                             (shape, dtype, buf.nbytes))
        return np.asarray(_PinnedView(buf, self, shape, dtype))

    def clear(self):
        with self._lock:
            drop_idle(self, -1)

    def close(self):
        """Frees the idle buffers, and those given back later."""
        self._max = -1
        self.clear()
