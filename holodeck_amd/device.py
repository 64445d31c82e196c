"""Device buffers and streams (PyTorch-ROCm tensors used only as HBM buffers)."""
import collections
import threading

import numpy as np

try:
    import torch
except ImportError:   # pragma: no cover
    torch = None

from . import _lib


def require_device():
    """Return the HIP device, or raise: this package has no CPU path."""
    if torch is None or not torch.cuda.is_available():
        raise _lib.HoloHipError("holodeck_amd needs a HIP (ROCm) GPU; none is available")
    _lib.load()
    return torch.device("cuda", torch.cuda.current_device())


def stream_ptr():
    return torch.cuda.current_stream().cuda_stream


def ptr(t):
    """Device pointer of a tensor (None -> NULL)."""
    if t is None:
        return None
    if not t.is_contiguous():
        raise ValueError("tensor must be contiguous")
    return t.data_ptr()


def to_dev(a, dtype=None, slots=False):
    """numpy array / scalar sequence / tensor -> contiguous device tensor (float64 default).

    Host arrays up to STAGE_MAX_BYTES are copied into a pinned staging ring and uploaded
    asynchronously on the current stream, so the host does not wait for the stream's earlier
    work; larger arrays are copied by the runtime, or with ``slots`` through two pinned slots (_Slots):
    faster for a caller that waits for the stream next, as the surrogate does, but the host then waits for
    the stream's earlier kernels (a library with samples in flight on three streams, whose geometry is
    uploaded between them: 222 samples/s against 135 through the slots).  A tensor returned here is ready for work
    on the current stream; another stream must wait for it (an event).
    """
    dev = require_device()
    if isinstance(a, torch.Tensor):
        t = a.to(dev)
        if dtype is not None:
            t = t.to(dtype)
        return t.contiguous()
    arr = np.ascontiguousarray(a)
    if dtype is None:
        dtype = torch.int64 if np.issubdtype(arr.dtype, np.integer) else torch.float64
    host = torch.as_tensor(arr).to(dtype)
    if host.numel() == 0:
        return torch.empty(host.shape, dtype=dtype, device=dev)
    staged = _staging().put(host) if host.numel() * host.element_size() <= STAGE_MAX_BYTES else None
    if staged is None:                          # large
        if not slots:
            return host.to(dev)
        out = torch.empty(host.shape, dtype=dtype, device=dev)
        if not _SLOTS.push(host.contiguous().view(-1).view(torch.uint8), out.view(-1).view(torch.uint8)):
            out.copy_(host)
        return out
    out = torch.empty(host.shape, dtype=dtype, device=dev)
    out.copy_(staged, non_blocking=True)
    _staging().done()
    return out


STAGE_MAX_BYTES = 256 << 10


class _Staging:
    """A pinned host ring (allocated once) for asynchronous uploads.  Each upload copies its
    data into the next free region and records an event after the device copy on the current
    stream; a region is rewritten only after the event of the copy that last used it."""

    def __init__(self, nbytes=64 << 20):
        self.buf = torch.empty(nbytes, dtype=torch.uint8, pin_memory=True)
        self.n = nbytes
        self.head = 0
        self.lap = 0
        self.pending = collections.deque()      # (lap, start, end, event) in allocation order
        self._last = None

    def put(self, host):
        nb = host.numel() * host.element_size()
        size = (nb + 255) & ~255
        if size > self.n // 4:
            return None
        if self.head + size > self.n:
            self.head = 0
            self.lap += 1
        start, end = self.head, self.head + size
        while self.pending and (self.pending[0][0] < self.lap - 1 or
                                (self.pending[0][0] < self.lap and self.pending[0][1] < end)):
            self.pending.popleft()[3].synchronize()
        view = self.buf[start:start + nb].view(host.dtype).view(host.shape)
        view.copy_(host)
        self.head = end
        self._last = (self.lap, start, end)
        return view

    def done(self):
        ev = torch.cuda.Event()
        ev.record()
        self.pending.append(self._last + (ev,))


_STAGING = {}


def _staging():
    dev = torch.cuda.current_device()
    st = _STAGING.get(dev)
    if st is None:
        st = _STAGING[dev] = _Staging()
    return st


def empty(shape, dtype=None):
    dev = require_device()
    return torch.empty(shape, dtype=dtype or torch.float64, device=dev)


def workspace(nbytes):
    dev = require_device()
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=dev)


DOWNLOAD_MIN_BYTES = 64 << 10     # smaller results: the runtime's own copy
SLOT_BYTES = 4 << 20


class _Slots:
    """Two pinned slots through which larger arrays pass between host and device: one is in flight by DMA
    (56 GB/s measured; the runtime's pageable copies reach 4) while the host's threads copy the other
    from or to its place.  One caller at a time; others meanwhile take the runtime's own copy.  After an
    exception (an interrupted wait) a copy may still be in flight in a slot: the slots are given up, and
    torch's host allocator hands their memory out again only when those copies are done."""

    def __init__(self):
        self.lock = threading.Lock()
        self.slots = None

    def _take(self):
        if not self.lock.acquire(blocking=False):
            return False
        if self.slots is None:
            try:
                self.slots = [torch.empty(SLOT_BYTES, dtype=torch.uint8, pin_memory=True) for _ in range(2)]
            except RuntimeError:    # no pinned memory: the runtime's own copy needs none
                self.lock.release()
                return False
            except BaseException:
                self.lock.release()
                raise
        return True

    def fetch(self, src, dst):
        """src: 1-D uint8 device tensor, as its device's current stream leaves it (where the copies run, so
        where their events belong); dst: host tensor of its size.  False (nothing done) when another
        caller holds the slots or none can be had."""
        stream = torch.cuda.current_stream(src.device)
        if not self._take():
            return False
        flying = None
        try:
            for k, s0 in enumerate(range(0, src.numel(), SLOT_BYTES)):
                part = src[s0:s0 + SLOT_BYTES]
                slot = self.slots[k & 1][:part.numel()]
                slot.copy_(part, non_blocking=True)
                ev = torch.cuda.Event()
                ev.record(stream)
                if flying is not None:
                    self._land(*flying)
                flying = (dst[s0:s0 + SLOT_BYTES], slot, ev)
            if flying is not None:
                self._land(*flying)
        except BaseException:
            self.slots = None
            raise
        finally:
            self.lock.release()
        return True

    @staticmethod
    def _land(dst, slot, ev):
        ev.synchronize()
        dst.copy_(slot)

    def push(self, src, dst):
        """src: 1-D uint8 host tensor; dst: device tensor of its size, written on its device's current
        stream before this returns.  False (nothing done) when another caller holds the slots or none can be had."""
        stream = torch.cuda.current_stream(dst.device)
        if not self._take():
            return False
        busy = [None, None]
        try:
            for k, s0 in enumerate(range(0, src.numel(), SLOT_BYTES)):
                part = src[s0:s0 + SLOT_BYTES]
                if busy[k & 1] is not None:
                    busy[k & 1].synchronize()
                slot = self.slots[k & 1][:part.numel()]
                slot.copy_(part)
                dst[s0:s0 + SLOT_BYTES].copy_(slot, non_blocking=True)
                busy[k & 1] = torch.cuda.Event()
                busy[k & 1].record(stream)
            for ev in busy:
                if ev is not None:
                    ev.synchronize()
        except BaseException:
            self.slots = None
            raise
        finally:
            self.lock.release()
        return True


_SLOTS = _Slots()


def to_host(t, out=None):
    """Host numpy copy of a tensor (waits for its device's current stream); into the contiguous array
    ``out`` if given."""
    t = t.detach()
    if not t.is_cuda or t.numel() * t.element_size() < DOWNLOAD_MIN_BYTES:
        if out is None:
            return t.cpu().numpy()
        torch.from_numpy(out).copy_(t)
        return out
    t = t.contiguous()
    host = torch.empty(t.shape, dtype=t.dtype) if out is None else torch.from_numpy(out)
    if not _SLOTS.fetch(t.view(-1).view(torch.uint8), host.view(-1).view(torch.uint8)):
        host.copy_(t)
    return host.numpy()
