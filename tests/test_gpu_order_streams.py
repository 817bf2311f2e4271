"""Order statistics on several streams (needs an MI355X): the order numbers on
the device belong to the stream whose kernels read them, and a call that names
a stream returns what that stream computed."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _photons(gpu, n=20000):
    import torch
    rng = np.random.default_rng(4)
    t = lambda x: torch.as_tensor(x, device=gpu)  # noqa: E731
    order = rng.integers(-3, 4, n).astype(np.int32)
    return t(order), t(rng.random(n)), t(rng.normal(0, 1, n)), order


def test_order_numbers_of_each_stream(gpu, monkeypatch):
    import torch
    from marxs_amd import _lib, analysis
    order, prob, value, host = _photons(gpu)
    seen = []

    class Noting:
        def __getattr__(self, name):
            return getattr(lib, name)

        def mx_order_stats(self, a, stream):
            seen.append(a.orders)
            return lib.mx_order_stats(a, stream)
    lib = _lib.lib
    monkeypatch.setattr(_lib, 'lib', Noting())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in (*streams, *streams):
        with torch.cuda.stream(s):
            r = analysis.order_stats(order, prob, np.arange(-3, 4), value=value)
        assert r['count'].tolist() == [int((host == k).sum()) for k in range(-3, 4)]
    # one copy a stream, used again
    assert seen[:2] == seen[2:] and seen[0] != seen[1]


@pytest.mark.parametrize('wrap', [int, ctypes.c_void_p])
def test_named_stream(gpu, wrap):
    """The named stream is busy for a while; the results are its results, and
    it starts after what the current stream still does to the inputs."""
    import torch
    from marxs_amd import analysis
    order, prob, value, host = _photons(gpu)
    want = analysis.order_stats(order, prob, np.arange(-3, 4), value=value)
    for busy in (False, True):
        s = torch.cuda.Stream()
        late = torch.zeros_like(value)
        torch.cuda.synchronize()
        if busy:
            with torch.cuda.stream(s):
                torch.cuda._sleep(20_000_000)
        else:
            torch.cuda._sleep(20_000_000)
        late.copy_(value)
        got = analysis.order_stats(order, prob, np.arange(-3, 4), value=late, stream=wrap(s.cuda_stream))
        for k in want:
            assert np.array_equal(got[k], want[k]), k
