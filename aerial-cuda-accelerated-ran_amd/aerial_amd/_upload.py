"""Upload of a call's small host structures (parameters, descriptors, pointer
arrays) as one block: packed in page-locked host memory, copied to the device
by one asynchronous copy on the launching stream.  Separate copies from
pageable memory each wait for the stream's earlier work before the call can
go on, so that a call's host time and its kernels never overlap.  Both blocks
come from torch's caching allocators, which hand the host block out again
only after the copy has run and the device block in the stream's order."""
import contextlib
import ctypes as C

import torch

_ALIGN = 64


class UploadBlock:
    """Space for parts of the given sizes; part i at host(i) / dev(i).

    in_graph: may be used while the stream is being captured.  The graph's copy
    then reads the host block at every replay, so the block is pageable memory of
    its own, and whoever gets it keeps it (`captured`) as long as the graph may run."""

    def __init__(self, sizes, in_graph=False):
        self.captured = torch.cuda.is_current_stream_capturing()
        if self.captured and not in_graph:
            raise RuntimeError("host parameters cannot be uploaded while the stream is being captured")
        self._off, n = [], 0
        for s in sizes:
            self._off.append(n)
            n += (s + _ALIGN - 1) // _ALIGN * _ALIGN
        self._host = torch.empty(max(n, 1), dtype=torch.uint8, device="cpu", pin_memory=not self.captured)
        self._dev = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
        self._hptr, self._dptr = self._host.data_ptr(), self._dev.data_ptr()

    def host(self, i):
        return self._hptr + self._off[i]

    def dev(self, i):
        return C.c_void_p(self._dptr + self._off[i])

    def send(self):
        self._dev.copy_(self._host, non_blocking=True)


class _OnStream:
    def __init__(self, stream):
        self._stream = stream if isinstance(stream, torch.cuda.Stream) else torch.cuda.ExternalStream(stream.cuda_stream)
        self._ctx = torch.cuda.stream(self._stream)

    def __enter__(self):
        capturing, before = torch.cuda.is_current_stream_capturing(), torch.cuda.current_stream()
        self._ctx.__enter__()
        if before != self._stream and not capturing and not torch.cuda.is_current_stream_capturing():
            self._stream.wait_stream(before)
        return self

    def __exit__(self, *exc):
        return self._ctx.__exit__(*exc)


def on_stream(stream):
    """Context in which blocks belong to the launching stream.  What was queued
    on the caller's current stream so far (the inputs' producers, the fill of an
    output) comes before what is launched in it."""
    return _OnStream(stream) if stream is not None else contextlib.nullcontext()


def written_here(stream, tensor):
    """Within on_stream(stream): `tensor`, allocated for the caller's current stream,
    is written by the launching one; its memory is not handed out again before
    that has run."""
    if stream is not None and not torch.cuda.is_current_stream_capturing():
        tensor.record_stream(torch.cuda.current_stream())
