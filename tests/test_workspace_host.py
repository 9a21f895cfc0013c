"""Workspaces of the mat-vec calls belong to one call: a call that starts while another is
between its launches (the library is entered without the GIL), or a larger call after a graph was
captured, must not be handed, or free, the memory an earlier call's kernels use (CPU, with the
native library replaced)."""
import threading

import pytest
import torch

from brainstate_amd import _native as N
from brainstate_amd import ops


class _Lib:
    """Records (address, bytes) of the workspace of every call; the first call waits inside
    the library until a second one has been through."""

    def __init__(self, size):
        self.size, self.seen = size, []
        self.entered, self.second = threading.Event(), threading.Event()

    def bs_matvec_workspace_size(self, *a):
        return self.size

    bs_event_bucket_batch_workspace_size = bs_matvec_workspace_size

    def _call(self, ws, nbytes):
        self.seen.append((ws.value, nbytes))
        if len(self.seen) == 1:
            self.entered.set()
            assert self.second.wait(20)
        return 0

    def bs_matvec_ws_f32(self, *a):
        return self._call(a[-3], a[-2])

    def bs_event_bucket_batch_f32(self, *a):
        return self._call(a[-3], a[-2])


@pytest.mark.parametrize('call', ['event', 'value', 'bucket_batch'])
@pytest.mark.parametrize('grow', [0, 4096])
def test_calls_on_one_stream_have_workspaces_of_their_own(monkeypatch, call, grow):
    lib = _Lib(4096)
    monkeypatch.setattr(N, 'lib', lambda: lib)
    monkeypatch.setattr(N, 'raw_stream', lambda device=None: 7)
    monkeypatch.setattr(ops, '_WS_CACHE', {})
    idx = torch.zeros(3, 2, dtype=torch.int32)
    L = dict(seg=idx, n_pre=3, n_post=4, nb=1)
    monkeypatch.setattr(ops, '_bucket_call_args', lambda L: ((),))

    def run():
        if call == 'bucket_batch':
            ops.event_bucket_batch(torch.ones(2, 3), L)
        else:
            f = ops.event_matvec if call == 'event' else ops.value_matvec
            f(torch.ones(3), idx, 0.5, 4)

    first = threading.Thread(target=run)
    first.start()
    assert lib.entered.wait(20)
    lib.size += grow
    try:
        run()                                 # while the first call is inside the library
    finally:
        lib.second.set()
        first.join()
    (a, na), (b, nb) = lib.seen
    assert a + na <= b or b + nb <= a, 'two calls in flight share a workspace'
    assert not ops._WS_CACHE                  # nothing that a later, larger call could replace
