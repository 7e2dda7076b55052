"""Argument checks on device tensors, fetched with one host synchronization.

The reference validates cache lengths, page tables and cu_seqlens with a
chain of ``torch.any(...)`` / ``.item()`` calls, each of which waits for the
stream to drain (flash_attn_interface.py:433-470, :583-627).  ``Deferred``
queues those checks and reads them all with one synchronization.  Range
checks on device tensors (an array, an array plus an elementwise addend, or
the differences of adjacent elements) reduce in one native launch per eight
distinct arrays (``fa_check_bounds``), which writes min and max straight into
pinned host memory, where the host polls for them; other device scalars (flags,
values) are packed by reinterpreting them as 32-bit words and copied with one
device-to-host copy.  A call whose launch is safe on unchecked arguments
(``side=True``, the decode path) queues range checks only; they reduce on a
second stream, so the launch does not queue behind them.  A launch that is not
can be guarded instead (``flush(launch, guarded=True)``): it takes the checks'
device flags and does nothing when one is set.  Exceptions keep the reference's order: a check
that fails on the host first raises the first failing device check queued
before it, exactly as the reference's sequential checks would have.
"""
from __future__ import annotations

import struct
from typing import List, Optional

import torch

from . import _native

_I64_MIN, _I64_MAX = -(1 << 63), (1 << 63) - 1
_WORDS = {torch.int32: 1, torch.float32: 1, torch.int64: 2, torch.float64: 2}


def _decode(words: List[int], dtype: torch.dtype):
    if dtype == torch.int32:
        return words[0]
    if dtype == torch.int64:
        return (words[1] << 32) | (words[0] & 0xFFFFFFFF)
    raw = struct.pack("<" + "i" * len(words), *words)
    return struct.unpack("<f" if dtype == torch.float32 else "<d", raw)[0]


_SIDE_STREAMS: dict = {}


def _side_stream(device: torch.device):
    """A second stream per device (default priority) for argument checks, and
    an event to mark their end with (nothing waits for it)."""
    key = device.index if device.index is not None else torch.cuda.current_device()
    pair = _SIDE_STREAMS.get(key)
    if pair is None:
        pair = _SIDE_STREAMS[key] = (torch.cuda.Stream(device=key), torch.cuda.Event())
    return pair


def _as_int(t: torch.Tensor) -> torch.Tensor:
    t = t.reshape(-1)
    if t.dtype not in (torch.int32, torch.int64):
        t = t.long()
    return t.contiguous()


def _host_minmax(a: torch.Tensor, b: Optional[torch.Tensor], diff: bool):
    """min and max of a (+ b) or of a's adjacent differences, on the host
    (for tensors that are not on a GPU)."""
    x = a.long()
    if diff:
        x = x[1:] - x[:-1]
    elif b is not None:
        x = x + b.long()
    return int(x.min()), int(x.max())


def _outside(item, got) -> bool:
    """Whether the (min, max) of a queued range check leaves its bounds."""
    _, _, lo, hi, _ = item
    return (lo is not None and got[0] < lo) or (hi is not None and got[1] > hi)


class Deferred:
    def __init__(self, side: bool = False) -> None:
        # (kind, exception or None, lo, hi, payload), in queue order:
        #   "range":  payload (a, b, diff); raise exc unless the min and max of
        #             a (+ b), or of a's adjacent differences, lie in [lo, hi]
        #   "minmax": payload as "range"; (min, max) is returned as a value
        #   "flag":   payload [bad]; raise exc if the device boolean is true
        #   "value":  payload [t]; the device scalar is returned as a value
        #
        # side=True: range checks only, reduced at flush time on a second
        # stream that first waits for the current one, so a launch passed to
        # flush() starts on the current stream without queueing behind them.
        self._items: list = []
        self._nvalues = 0
        self._side = side

    def check(self, bad: torch.Tensor, exc: BaseException) -> None:
        """Queue ``raise exc`` if the device boolean ``bad`` is true."""
        if self._side:
            raise RuntimeError("Deferred(side=True) queues range checks only")
        self._items.append(("flag", exc, None, None, [bad.reshape(())]))

    def check_range(self, t: torch.Tensor, lo: Optional[int], hi: Optional[int],
                    exc: BaseException, plus: Optional[torch.Tensor] = None,
                    diff: bool = False) -> None:
        """Queue ``raise exc`` unless every element of the integer tensor ``t``
        (plus ``plus`` elementwise, when given; or every difference of
        adjacent elements, with ``diff``) lies in ``[lo, hi]`` (``None``:
        unbounded on that side)."""
        if t.numel() - (1 if diff else 0) <= 0:
            return
        self._items.append(("range", exc, lo, hi,
                            (_as_int(t), None if plus is None else _as_int(plus), diff)))

    def value_range(self, t: torch.Tensor, diff: bool = False) -> int:
        """Queue the (min, max) of an integer tensor as one value; returns its
        index in ``flush()``'s result."""
        if self._side:
            raise RuntimeError("Deferred(side=True) queues range checks only")
        self._items.append(("minmax", None, None, None, (_as_int(t), None, diff)))
        self._nvalues += 1
        return self._nvalues - 1

    def value(self, t: torch.Tensor) -> int:
        """Queue a device scalar to fetch; returns its index in ``flush()``'s result."""
        if self._side:
            raise RuntimeError("Deferred(side=True) queues range checks only")
        self._items.append(("value", None, None, None, [t.reshape(())]))
        self._nvalues += 1
        return self._nvalues - 1

    def fail(self, exc: BaseException) -> None:
        """A host-side check failed: device checks queued earlier win."""
        self.flush()
        raise exc

    def ranges_only(self) -> bool:
        """Whether only range checks of device arrays are queued (what a
        guarded launch can be guarded with)."""
        return all(it[0] == "range" and it[4][0].is_cuda for it in self._items)

    def flush(self, launch=None, guarded: bool = False) -> list:
        """Raise the first failing queued check; return the queued values.

        With ``launch`` (a callable that enqueues kernels on the current
        stream), the checks' results go to pinned host memory first,
        ``launch()`` runs, and only then does the host wait, for the checks
        alone: the launched work runs while the host reads them, and a
        failing check still raises before this call returns.  With
        ``side=True`` the range checks reduce on a second stream, so the
        launch does not queue behind them.  Only kernels that stay inside
        their buffers whatever the checked arrays hold may be launched this
        way, or, with ``guarded`` (range checks only), kernels that return at
        once when one of the int32 device flags ``launch(flags)`` gets is set
        (None: nothing was checked on the device).  Checks of host tensors have
        no flag: when one of them fails, a guarded launch is not made."""
        items, self._items = self._items, []
        self._nvalues = 0
        if not items:
            if launch is not None:
                launch(None) if guarded else launch()
            return []
        # Range reductions: one launch per eight distinct device arrays (an
        # array checked against several bounds reduces once), results in pinned
        # host memory; host tensors on the host.
        ranged = [i for i, it in enumerate(items) if it[0] in ("range", "minmax")]
        on_dev = [i for i in ranged if items[i][4][0].is_cuda]
        results = {i: _host_minmax(*items[i][4]) for i in ranged if not items[i][4][0].is_cuda}
        done = host_rng = guard = handle = marker = None
        jobs, job_of = [], {}
        if on_dev:
            seen = {}
            for i in on_dev:
                a, b, diff = items[i][4]
                lo = _I64_MIN if items[i][2] is None else max(items[i][2], _I64_MIN)
                hi = _I64_MAX if items[i][3] is None else min(items[i][3], _I64_MAX)
                key = (a.data_ptr(), a.numel(), a.dtype, diff,
                       None if b is None else (b.data_ptr(), b.dtype))
                j = seen.get(key)
                if j is None:
                    seen[key] = j = len(jobs)
                    jobs.append([a, b, diff, lo, hi])
                else:
                    jobs[j][3] = max(jobs[j][3], lo)
                    jobs[j][4] = min(jobs[j][4], hi)
                job_of[i] = j
            device = jobs[0][0].device
            stream = torch.cuda.current_stream(device)
            if self._side:
                side, marker = _side_stream(device)
                side.wait_stream(stream)
                stream = side
            handle = stream.cuda_stream
            host_rng = torch.empty(3 * len(jobs), dtype=torch.int64, pin_memory=True)
            if guarded:
                guard = torch.empty(len(jobs), dtype=torch.int32, device=device)
            step = _native.MAX_RANGE_CHECKS
            for s0 in range(0, len(jobs), step):
                chunk = jobs[s0:s0 + step]
                _native.check_bounds(chunk, host_rng[3 * s0:3 * (s0 + len(chunk))],
                                     None if guard is None else guard[s0:s0 + len(chunk)], handle)
        # Flags and values: packed into 32-bit words, one copy.
        scal = [i for i, it in enumerate(items) if it[0] in ("flag", "value")]
        words, dtypes, host_sc = [], [], None
        if scal:
            scalars = []
            for i in scal:
                s = items[i][4][0].reshape(1)
                if s.dtype not in _WORDS:
                    s = s.to(torch.int32 if s.dtype == torch.bool else torch.int64)
                scalars.append(s.view(torch.int32))
                dtypes.append(s.dtype)
            packed = torch.cat(scalars) if len(scalars) > 1 else scalars[0]
            if packed.is_cuda:
                host_sc = torch.empty(packed.shape, dtype=packed.dtype, pin_memory=True)
                host_sc.copy_(packed, non_blocking=True)
                done = torch.cuda.Event()
                done.record()
            else:
                words = packed.tolist()
        failed = None
        # (`results` holds the host tensors' ranges so far, mostly none.)
        if guarded and results and any(_outside(items[i], r) for i, r in results.items()):
            launch = None
        if launch is not None:
            try:
                launch(guard) if guarded else launch()
            except Exception as exc:   # a failing check goes first
                failed = exc
        if marker is not None:
            # Without a marker behind the checks the attention kernel beside them
            # runs 1-3 % slower: one token of 32 (64) sequences of 7000 keys, 8 KV
            # heads of 128, bf16, MI355X: 157.9 (294.5) us a call, 153.4 (289.5)
            # with it.  Recorded here, its 3 us of host time pass while the
            # checks run.
            marker.record(stream)
        # Every tensor checked on the device is referenced by `items` until this
        # wait: none returns to the caching allocator (whose next user could
        # overwrite it on the current stream) while a check reads it, and the
        # pinned results outlive the writes to them.
        if host_rng is not None:
            _native.check_wait(host_rng, len(jobs), handle)
        if done is not None:
            done.synchronize()
        if host_rng is not None:
            got = host_rng.tolist()
            for i in on_dev:
                j = job_of[i]
                results[i] = (got[3 * j], got[3 * j + 1])
        if host_sc is not None:
            words = host_sc.tolist()
        scalars_dec, pos = [], 0
        for dt in dtypes:
            n = _WORDS[dt]
            scalars_dec.append(_decode(words[pos:pos + n], dt))
            pos += n
        values, k = [], 0
        for i, (kind, exc, lo, hi, _) in enumerate(items):
            if kind == "range":
                mn, mx = results[i]
                if (lo is not None and mn < lo) or (hi is not None and mx > hi):
                    raise exc
            elif kind == "minmax":
                values.append(results[i])
            else:
                got = scalars_dec[k]
                k += 1
                if kind == "flag" and got:
                    raise exc
                if kind == "value":
                    values.append(got)
        if failed is not None:
            raise failed
        return values
