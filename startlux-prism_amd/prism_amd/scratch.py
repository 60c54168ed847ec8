"""Scratch memory of the kernels that need some: one buffer per device and stream, so that calls in flight on different
streams never share one (two launches of a call write it and read it back: another stream's call between them, or a
replayed graph's, would be read instead).

  * Eager calls get their stream's buffer, made at the first call on that stream (at most STREAMS per device; beyond
    that the oldest is given back to the stream it was allocated on, whose order makes that safe).
  * Under graph capture no stream's buffer is handed out.  Scratch with no initial contents is a new tensor, from the
    graph's own pool, for each call.  Scratch that has to start zeroed (a fill would be a node of the graph, run at every
    replay) is the device's own for captured calls, made with its first eager one: graphs holding such calls must not
    be replayed at the same time.  On a device with no eager call yet there is none (None).

Calls of several threads on one stream share its buffer: a call that launches more than one kernel on it holds a lock
(locked_call), so that its launches stay together.
"""
import threading

import torch

from . import _lib as L

STREAMS = 8
_LOCK = threading.Lock()
_capturing = torch._C._cuda_isCurrentStreamCapturing      # (in the path of every decode-size call)


def locked_call(name, *args):
    """_lib.call of an entry point whose launches hand scratch from one to the next."""
    with _LOCK:
        return L.call(name, *args)


class Scratch:
    """`nbytes` of scratch, the first `zeroed` of which every launch finds zero and leaves zero."""

    def __init__(self, nbytes, zeroed=0):
        self.nbytes, self.zeroed = nbytes, zeroed
        self._eager = {}                 # (device index, stream) -> buffer, in the order made
        self._captured = {}              # device index -> the zeroed bytes for captured calls, or None

    def get(self, dev, zeroed=True, need=None, stream=None):
        """The buffer for a call on dev's current stream (stream: its handle, if the caller has it).  zeroed: the call uses
        the zeroed bytes (and no others); need: the bytes the call has a use for, where they are known (all that a captured
        one gets, whose graph's pool keeps them)."""
        idx = dev.index
        if idx is None:
            idx = torch.cuda.current_device()
        if _capturing():
            if idx not in self._captured:
                return None
            if zeroed and self.zeroed:
                return self._captured[idx]
            return self._empty(idx, self.nbytes if need is None else min(need, self.nbytes))
        key = (idx, L.raw_stream(idx) if stream is None else stream)
        buf = self._eager.get(key)
        return self._make(key) if buf is None else buf

    def _make(self, key):
        idx = key[0]
        with _LOCK:
            if key in self._eager:
                return self._eager[key]
            if idx not in self._captured:
                w = None
                if self.zeroed:
                    w = self._empty(idx, self.zeroed).zero_()
                    torch.cuda.current_stream(idx).synchronize()         # replays run on any stream
                self._captured[idx] = w
            mine = [k for k in self._eager if k[0] == idx]
            if len(mine) >= STREAMS:
                del self._eager[mine[0]]
            buf = self._empty(idx, self.nbytes)
            if self.zeroed:
                buf[:self.zeroed].zero_()
            self._eager[key] = buf
        return buf

    @staticmethod
    def _empty(idx, n):
        return torch.empty(n, dtype=torch.uint8, device=torch.device("cuda", idx))
