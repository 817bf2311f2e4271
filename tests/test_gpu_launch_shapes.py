"""How the photons of a launch are spread over workgroups, and where a stage's
records are read from, does not show in the results: lists from one photon to
more than the work-items of one workgroup per CU, tables with and without an
LDS image, a detector alone and the same detector as one of two."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 256 * 1024 + 65


def _columns(dp):
    import torch
    cols = {'pos': dp.pos, 'dir': dp.dir, 'pol': dp.pol, 'prob': dp.prob, **dp.fcols, **dp.icols}
    return {k: (v.view(torch.int64) if v.dtype == torch.float64 else v) for k, v in cols.items()}


def _source(n, seed=3):
    import torch
    from marxs_amd.tracer import DevicePhotons
    g = torch.Generator(device='cuda')
    g.manual_seed(seed)
    u = torch.rand((2, n), dtype=torch.float64, device='cuda', generator=g)
    d = torch.zeros((3, n), dtype=torch.float64, device='cuda')
    d[0] = -1.
    phi = 2 * np.pi * u[0]
    pol = torch.stack([torch.zeros_like(phi), torch.sin(phi), torch.cos(phi)])
    return DevicePhotons(d, pol, 0.4 + 1.4 * u[1], torch.ones(n, dtype=torch.float64, device='cuda'))


def _head(src, n):
    from marxs_amd.tracer import DevicePhotons
    return DevicePhotons(src.dir[:, :n], src.pol[:, :n], src.energy[:n], src.prob[:n])


def _launch(ci, src, u, prec):
    import torch
    from marxs_amd.batch import outputs_like
    out = outputs_like(src)
    st = ci.launch(out, u, prec, src=src)
    torch.cuda.synchronize()
    return _columns(out), st.cpu()


def _same(a, b, skip=()):
    import torch
    assert a.keys() == b.keys()
    for k in a:
        if k not in skip:
            assert torch.equal(a[k], b[k]), k


@pytest.fixture(scope='module')
def cat():
    from marxs_amd import configs
    from marxs_amd.tracer import CompiledInstrument
    return CompiledInstrument(configs.cat_rowland_instrument(150)[0])


@pytest.mark.parametrize('prec', [64, 32])
def test_short_lists_are_the_head_of_a_long_one(cat, prec):
    # 64: one chunk; 256 * 64: one chunk per CU; 256 * 768 and 256 * 1024: one
    # workgroup per CU full
    src = _source(N)
    u = cat.draw_uniforms(N)
    full, _ = _launch(cat, src, u, prec)
    for n in (1, 63, 64, 65, 769, 256 * 64 - 1, 256 * 64 + 1, 256 * 768, 256 * 768 + 1, 256 * 1024, N - 1):
        got, _ = _launch(cat, _head(src, n), u[:, :n].contiguous(), prec)
        _same({k: v[..., :n] for k, v in full.items()}, got)


@pytest.mark.parametrize('prec', [64, 32])
def test_tables_in_lds_or_not(cat, prec):
    import torch
    from marxs_amd.batch import _tables_with_budget
    n = 30011
    src = _source(n)
    u = cat.draw_uniforms(n)
    ref, st = _launch(cat, src, u, prec)
    was = cat.dev_tables
    sizes = set()
    try:
        # none; selector tables at most; odd numbers of 16-byte words around
        # multiples of what a workgroup loads at a time; all
        for budget in (0, 4096, 8 * 768 * 16 + 16, 8 * 1024 * 16 - 16, 150000):
            cat.dev_tables = _tables_with_budget(cat, budget)
            sizes.add(int(cat.dev_tables.struct.lds_bytes64 if prec == 64 else cat.dev_tables.struct.lds_bytes32))
            got, st2 = _launch(cat, src, u, prec)
            _same(ref, got, skip=('blaze',) if prec == 32 else ())
            # FP32: the cosine of the blaze angle is rounded in steps of 2^-24
            # below 1, and code that reads its tables from elsewhere may fuse
            # the products in it differently: 4 such steps, times 1 / sine
            x, y = ref['blaze'].view(torch.float64), got['blaze'].view(torch.float64)
            ok = ~torch.isnan(x)
            assert torch.equal(ok, ~torch.isnan(y))
            assert float(((x - y).abs() * torch.sin(x))[ok].max()) <= (4 * 2. ** -24 if prec == 32 else 0.)
            assert (st == st2).all()
    finally:
        cat.dev_tables = was
    assert len(sizes) >= 3


@pytest.mark.parametrize('prec', [64, 32])
def test_detector_alone_and_beside_another(prec):
    # the second detector of the pair lies off the beam
    import marxs_amd as mx
    from marxs_amd import configs
    from marxs_amd.tracer import CompiledInstrument
    n = 20001
    src = _source(n)
    one = configs.flat_grid_instrument(0.008)
    elems = list(one.elements)
    args = {'pixsize': 0.024, 'zoom': [1, 98.304, 98.304]}
    pair = mx.Parallel(elem_class=mx.FlatDetector, elem_args=args, id_col='CCD',
                       elem_pos={'position': [[0, 0.008, 0.008], [0, 5000., 5000.]]})
    single = mx.Parallel(elem_class=mx.FlatDetector, elem_args=args, id_col='CCD',
                         elem_pos={'position': [[0, 0.008, 0.008]]})
    cols = []
    for det in (single, pair):
        ci = CompiledInstrument(mx.Sequence(elements=elems[:-1] + [det]))
        u = ci.draw_uniforms(n) if not cols else u
        cols.append(_launch(ci, src, u, prec)[0])
    assert int((cols[0]['CCD'] == 0).sum()) > n // 2
    if prec == 64:
        _same(*cols)
        return
    # FP32: distances of 5000 mm carry a few 2^-24 of themselves, which the
    # slopes of up to 0.12 turn into 2e-4 mm or 0.01 pixel at most; 0.03 allowed
    import torch
    assert torch.equal(cols[0]['CCD'], cols[1]['CCD'])
    for k in ('detpix_x', 'detpix_y'):
        a, b = (c[k].view(torch.float64) for c in cols)
        ok = ~torch.isnan(a)
        assert torch.equal(ok, ~torch.isnan(b))
        assert float((a[ok] - b[ok]).abs().max()) < 0.03
