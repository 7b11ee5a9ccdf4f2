"""Pinned host arrays that earlier work on the device is still about to write: what a caller has in hand
who computes a call's inputs on the default stream (or on a stream that waits for it) and copies them
back without waiting. The calls that take host arrays read them after that work."""

import ctypes

import box2d_amd

COPY_BYTES = 1 << 30
COPIES = 40  # about 16 ms


def _check(rc):
    assert rc == 0, f"HIP error {rc}"


class EarlierWork:
    def __init__(self, blocking):
        """blocking: on a stream of its own that waits for the default stream, instead of the default one."""
        self.hip = box2d_amd.library()  # its runtime's functions (torch brings a second runtime)
        self.stream = ctypes.c_void_p()
        self.blocking = blocking
        self.memory = []

    def __enter__(self):
        if self.blocking:
            _check(self.hip.hipStreamCreate(ctypes.byref(self.stream)))
        self.source = self._allocate(self.hip.hipMalloc, COPY_BYTES)
        self.target = self._allocate(self.hip.hipMalloc, COPY_BYTES)
        return self

    def _allocate(self, allocate, size, *flags):
        p = ctypes.c_void_p()
        _check(allocate(ctypes.byref(p), ctypes.c_size_t(size), *flags))
        self.memory.append((self.hip.hipHostFree if flags else self.hip.hipFree, p))
        return p

    def writes(self, records):
        """A pinned array of zeros that receives the records (a ctypes array) after COPIES copies."""
        size = ctypes.sizeof(records)
        pinned = self._allocate(self.hip.hipHostMalloc, size, 0)
        device = self._allocate(self.hip.hipMalloc, size)
        ctypes.memset(pinned, 0, size)
        _check(self.hip.hipMemcpy(device, records, ctypes.c_size_t(size), 1))
        for _ in range(COPIES):
            _check(self.hip.hipMemcpyAsync(self.target, self.source, ctypes.c_size_t(COPY_BYTES), 3, self.stream))
        _check(self.hip.hipMemcpyAsync(pinned, device, ctypes.c_size_t(size), 2, self.stream))
        return pinned

    def __exit__(self, *error):
        _check(self.hip.hipDeviceSynchronize())
        for free, p in self.memory:
            _check(free(p))
        if self.blocking:
            _check(self.hip.hipStreamDestroy(self.stream))
