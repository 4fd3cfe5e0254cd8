"""Calls on several streams and host threads at once: each uses scratch buffers of its own
and gives the results it gives alone."""
import threading

import pytest

from pyemma_amd import _native

pytestmark = pytest.mark.gpu


def _inputs(i):
    t = _native.torch()
    g = t.Generator(device="cuda").manual_seed(i)
    X = t.randn((20_000 + 501 * i, 24), generator=g, device="cuda")
    return X, X[:: 20 + i][:300].contiguous(), t.tensor([0, len(X)], device="cuda")


def _calls(X, C, off):
    lab = _native.assign(X, C)
    m = _native.moments_lagged(X, off, 3, precision=_native.EMMA_PREC_BF16X4_ACC)
    Ck, idx = _native.kmeanspp(X, 12, 5)
    return lab, m[1], m[3], m[4], Ck, idx


def test_streams():
    t = _native.torch()
    data = [_inputs(i) for i in range(4)]
    ref = [_calls(*d) for d in data]
    t.cuda.synchronize()
    streams = [t.cuda.Stream() for _ in data]
    got = []
    for _ in range(5):
        got.append([])
        for s, d in zip(streams, data):
            with t.cuda.stream(s):
                got[-1].append(_calls(*d))
    t.cuda.synchronize()
    for pas in got:
        for a, b in zip(pas, ref):
            assert all(t.equal(x, y) for x, y in zip(a, b))


def test_threads_on_one_stream():
    t = _native.torch()
    data = [_inputs(i) for i in range(4)]
    ref = [_calls(*d) for d in data]
    t.cuda.synchronize()
    got = [None] * len(data)

    def work(i):
        got[i] = [_calls(*data[i]) for _ in range(5)]
        t.cuda.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(data))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for g, b in zip(got, ref):
        assert g is not None
        for a in g:
            assert all(t.equal(x, y) for x, y in zip(a, b))
