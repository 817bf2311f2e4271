"""Limits of turning photon table rows on the device: more rows than a launch
has work-items are refused before anything is launched, and tables beyond the
number that the table call turns there go through numpy with the same columns."""
import numpy as np
import pytest


@pytest.mark.parametrize('n', [-1, 2 ** 32 - 255, 2 ** 32, 2 ** 38])
def test_row_count_out_of_range(n):
    # (no pointer is followed: the count is checked first)
    from marxs_amd import _lib
    for rc in (_lib.lib.mx_pack_rows(16, 16, 16, 1., 16, n, None), _lib.lib.mx_unpack_rows(16, 4, 16, 16, 16, n, None)):
        assert rc == 1 and b'out of range' in _lib.lib.mx_last_error()


@pytest.mark.gpu
def test_long_tables_by_numpy(gpu, monkeypatch):
    import marxs_amd as mx
    import torch
    from marxs_amd import tracer
    rng = np.random.default_rng(3)
    n = 9000
    table = mx.PhotonTable({'pos': rng.normal(size=(n, 4)), 'dir': rng.normal(size=(n, 4)),
                            'polarization': rng.normal(size=(n, 4)), 'energy': np.ones(n), 'probability': np.ones(n)})
    calls = []

    class Noting:
        def __getattr__(self, name):
            if name in ('mx_pack_rows', 'mx_unpack_rows'):
                calls.append(name)
            return getattr(lib, name)
    lib = tracer._lib.lib
    monkeypatch.setattr(tracer._lib, 'lib', Noting())
    out = []
    for most, used in ((2 ** 31, 4), (9001, 4), (9000, 0)):
        monkeypatch.setattr(tracer, 'ROWS_MAX', most)
        calls.clear()
        dp = tracer.DevicePhotons.from_table(table, device=gpu)
        rows = tracer._rows_of(dp.pos, 1.)
        assert len(calls) == used
        out.append((dp, rows))
    for dp, rows in out[1:]:
        assert np.array_equal(rows, out[0][1]) and np.array_equal(rows[:, :3], table['pos'][:, :3])
        for k in ('pos', 'dir', 'pol'):
            assert torch.equal(getattr(dp, k), getattr(out[0][0], k))
