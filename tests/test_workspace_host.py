"""Workspaces of the mat-vec calls belong to one call: a call that starts while another is
between its launches (the library is entered without the GIL), or a larger call after a graph was
captured, must not be handed, or free, the memory an earlier call's kernels use (CPU, with the
native library replaced)."""
import ctypes
import threading

import pytest
import torch

from brainstate_amd import _native as N
from brainstate_amd import ops


@pytest.fixture(autouse=True)
def _sizes_asked_anew():
    ops._ws_bytes.cache_clear()
    yield
    ops._ws_bytes.cache_clear()


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
    ops._ws_bytes.cache_clear()
    try:
        run()                                 # while the first call is inside the library
    finally:
        lib.second.set()
        first.join()
    (a, na), (b, nb) = lib.seen
    assert a + na <= b or b + nb <= a, 'two calls in flight share a workspace'
    assert not ops._WS_CACHE                  # nothing that a later, larger call could replace


class _Kept:
    """bs_event_bucket_f32 replaced: notes the workspaces, and a call that starts while another
    is inside."""

    def __init__(self):
        self.seen, self.inside, self.overlap = [], 0, False
        self.entered, self.go = threading.Event(), threading.Event()

    def bs_event_bucket_f32(self, *a):
        self.overlap |= self.inside > 0
        self.inside += 1
        self.seen.append((a[-5].value, a[-4]))
        if len(self.seen) == 1:
            self.entered.set()
            self.go.wait(20)
        self.inside -= 1
        return 0

    def bs_spike_compact_workspace_size(self, n):
        return 8 * n


def test_kept_workspaces_stay_and_calls_do_not_interleave(monkeypatch):
    lib = _Kept()
    monkeypatch.setattr(N, 'lib', lambda: lib)
    monkeypatch.setattr(N, 'raw_stream', lambda device=None: 7)
    monkeypatch.setattr(ops, '_WS_CACHE', {})
    monkeypatch.setattr(ops, '_WS_OUTGROWN', [], raising=False)
    monkeypatch.setattr(ops, '_bucket_hint', lambda L: (None, [1], None))
    monkeypatch.setattr(ops, 'bucket_auto_mode', lambda L: 'split')
    t = torch.zeros(3, 2, dtype=torch.int32)

    def call(nbytes):
        L = dict(seg=t, lidx=t, w=None, qexp=None, n_pre=3, n_post=4)
        L['_call'] = ((), nbytes, (t, t, None, None), 1)
        ops.event_bucket(torch.ones(3, dtype=torch.uint8), L)

    first = threading.Thread(target=call, args=(4096,))
    second = threading.Thread(target=call, args=(4096,))
    first.start()
    assert lib.entered.wait(20)
    second.start()
    second.join(0.2)
    lib.go.set()
    first.join(20)
    second.join(20)
    assert not lib.overlap and len(lib.seen) == 2
    call(5000)                                # outgrows the first: both stay allocated
    call(100_000)
    kept = [lib.seen[0], lib.seen[2], lib.seen[3]]
    alive = {w.data_ptr(): w.numel() for w in [*ops._WS_OUTGROWN, *ops._WS_CACHE.values()]}
    assert all(alive.get(p, 0) >= n for p, n in kept) and len({p for p, _ in kept}) == 3
    sizes = sorted(alive.values())
    assert all(b >= 2 * a for a, b in zip(sizes, sizes[1:]))
    small, large = (ops.compact_workspace(n, torch.device('cpu')) for n in (10, 10_000))
    assert small is ops._WS_OUTGROWN[-1] and large.numel() >= 80_000


def test_dense_counters_are_never_under_partial_sums(monkeypatch):
    """bs_event_dense_f32 finds its leading ticket counters zero, whatever ran before: a call with
    fewer counters writes its partial sums into other memory, and outgrown workspaces stay."""
    class Lib:
        seen = []

        def bs_event_dense_workspace_size(self, B, n_in, n_out):
            return self.bs_event_dense_ticket_bytes(B, n_in, n_out) + 4 * B * n_out

        def bs_event_dense_ticket_bytes(self, B, n_in, n_out):
            return 256 * -(-n_out // 64)

        def bs_event_dense_f32(self, spk, dt, B, n_in, W, n_out, fae, out, ws, nbytes, stream):
            tick = self.bs_event_dense_ticket_bytes(B, n_in, n_out)
            view = (ctypes.c_uint8 * nbytes).from_address(ws.value)
            assert not any(view[:tick])
            for i in range(tick, nbytes):            # partial sums; the counters are left zero
                view[i] = 1
            self.seen.append((ws.value, nbytes))
            return 0

    lib = Lib()
    monkeypatch.setattr(N, 'lib', lambda: lib)
    monkeypatch.setattr(N, 'raw_stream', lambda device=None: 7)
    monkeypatch.setattr(ops, '_WS_CACHE', {})
    monkeypatch.setattr(ops, '_WS_OUTGROWN', [])

    def call(B, n_out):
        ops.event_dense(torch.ones(B, 5), torch.ones(5, n_out))
        return lib.seen[-1]

    ptr, nbytes = call(4, 200)                   # four blocks of counters; captured, say
    call(4, 10)                                  # one
    call(8000, 200)                              # outgrows the first
    call(4, 300)
    alive = {w.data_ptr(): w.numel() for w in [*ops._WS_OUTGROWN, *ops._WS_CACHE.values()]}
    assert alive.get(ptr, 0) >= nbytes
    assert not any((ctypes.c_uint8 * 1024).from_address(ptr))
