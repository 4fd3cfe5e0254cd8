"""Autotuner of the assignment's first pass.

The MFMA assignment exists in a few variants (emma_assign_variants): a coarse
fp16 pass with the fine pass on the frames it leaves, or the fine pass over
every frame.  Which one is faster depends on the dimension, the number of
centers and the data (how many frames the coarse bound leaves).  The
first call for a (dimension, center count) bucket times both on a
sample of the caller's own frames (up to 2^21 frames: smaller samples fill
the device for only a few rounds, where the variants tie and the full-size
winner is not visible) with HIP events on the current stream,
selects the fastest through emma_assign_select, and remembers the choice for
the rest of the process (a lock guards the table; the library's own table is
mutex-guarded).  Variants differ only in speed: labels are identical.
"""
import threading

from . import _native

__all__ = ["tune_assign", "tuned"]

_lock = threading.Lock()
_tuned = {}  # (ks, k bucket) -> (variant, [ms of the coarse, of the fine pipeline])


def _bucket(d, k):
    ks = -(-d // 16)
    for s in (2, 4, 8, 12, 16, 19, 24, 32):
        if ks <= s:
            ks = s
            break
    kp = -(-k // 32) * 32
    b = 0
    while (32 << b) < kp and b < 15:
        b += 1
    return ks, b


def tuned():
    with _lock:
        return dict(_tuned)


def tune_assign(Xt, Ct, mode=_native.EMMA_ASSIGN_BF16X3_RECHECK, sample=2097152, reps=2):
    """Select the fastest assignment variant for these sizes (once per bucket)."""
    if mode != _native.EMMA_ASSIGN_BF16X3_RECHECK:
        return None
    t = _native.torch()
    L = _native.lib()
    n, d = Xt.shape
    k = Ct.shape[0]
    nv = L.emma_assign_variants(d)
    if nv <= 1:
        return 0
    key = _bucket(d, k)
    with _lock:
        if key in _tuned:
            return _tuned[key][0]
        Xs = Xt[: min(n, sample)]
        lab = t.empty(Xs.shape[0], dtype=t.int32, device=Xt.device)
        times = []
        variants = (0, nv // 2)  # the first number of each pipeline
        for v in variants:
            _native.check(L.emma_assign_select(d, k, v), "emma_assign_select")
            _native.assign(Xs, Ct, mode=mode, labels=lab)  # warm-up
            e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(reps):
                _native.assign(Xs, Ct, mode=mode, labels=lab)
            e1.record()
            e1.synchronize()
            times.append(e0.elapsed_time(e1) / reps)
        best = variants[times.index(min(times))]
        _native.check(L.emma_assign_select(d, k, best), "emma_assign_select")
        _tuned[key] = (best, times)
        return best
