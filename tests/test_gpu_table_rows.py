"""Table rows turned into columns and back on the device (needs an MI355X): the
same values as numpy's, for widths and lengths around a workgroup's, and rows
that are not plain C-ordered float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n', [1, 2, 255, 256, 257, 100003])
@pytest.mark.parametrize('width', [3, 4, 6])
def test_columns_and_back(gpu, n, width, monkeypatch):
    from marxs_amd import tracer
    from marxs_amd.tracer import _columns_of, _rows_of
    monkeypatch.setattr(tracer, 'ROWS_ON_DEVICE', 0)
    rows = np.random.default_rng(n).normal(size=(n, width))
    rows[0, :2] = [np.nan, -0.]
    cols = _columns_of(rows, gpu)
    assert cols.cpu().numpy().tobytes() == np.ascontiguousarray(rows[:, :3].T).tobytes()
    back = _rows_of(cols, 1.)
    assert back.shape == (n, 4) and np.all(back[:, 3] == 1.)
    assert np.array_equal(back[:, :3], rows[:, :3], equal_nan=True)


@pytest.mark.parametrize('kind', ['fortran', 'readonly', 'float32', 'reversed', 'empty'])
@pytest.mark.parametrize('rows', [77, 8191, 8192])
def test_table_forms(gpu, kind, rows):
    import warnings
    import marxs_amd as mx
    from marxs_amd.tracer import DevicePhotons
    n = 0 if kind == 'empty' else rows
    rng = np.random.default_rng(5)
    d = rng.normal(size=(n, 4))
    if kind == 'fortran':
        d = np.asfortranarray(d)
    elif kind == 'float32':
        d = d.astype(np.float32)
    elif kind == 'reversed':
        d = d[::-1]
    elif kind == 'readonly':
        d.flags.writeable = False
    t = mx.PhotonTable({'dir': d, 'polarization': d, 'pos': d, 'energy': np.ones(n), 'probability': np.ones(n)})
    with warnings.catch_warnings():
        warnings.simplefilter('error')
        dp = DevicePhotons.from_table(t, device=gpu)
    want = np.asarray(d, dtype=float)[:, :3].T
    for c in (dp.dir, dp.pol, dp.pos):
        assert np.array_equal(c.cpu().numpy(), want)
    # each column its own memory, and none of it the table's
    assert n == 0 or len({dp.dir.data_ptr(), dp.pol.data_ptr(), dp.pos.data_ptr()}) == 3
