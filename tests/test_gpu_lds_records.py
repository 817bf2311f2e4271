"""FP64 test records of 14 words in LDS: the image holds them for the largest
facet arrays, and a trace that reads them gives the bits of one that reads the
records in global memory (needs an MI355X for the traces)."""
import numpy as np
import pytest

from marxs_amd import configs
from marxs_amd.compiler import LDS_BUDGET64, STAGE_DETECTOR, STAGE_GRATING, compile_tree


def _instrument(facets, interp):
    kw = {'efficiency': configs.blaze_interp_efficiency()} if interp else {}
    return configs.cat_rowland_instrument(facets, **kw)[0]


@pytest.mark.parametrize('facets', [50, 121, 800])
@pytest.mark.parametrize('interp', [False, True])
def test_image_holds_the_records(facets, interp):
    t = compile_tree(_instrument(facets, interp))
    assert t.lds_bytes64 <= LDS_BUDGET64
    for s, st in enumerate(t.stages):
        if st.kind not in (STAGE_GRATING, STAGE_DETECTOR):
            continue
        o, n = int(t.stage_i[s, 21]), len(st.elements)
        assert o >= 0 and o % 16 == 0
        rec = t.lds_image64[o:o + 8 * 14 * n].view(np.float64).reshape(n, 14)
        assert np.array_equal(rec, t.elem_t[st.elem0:st.elem0 + n, :14])
        assert np.all(t.elem_t[st.elem0:st.elem0 + n, 14:] == 0.)


@pytest.mark.gpu
@pytest.mark.parametrize('facets', [50, 800])
@pytest.mark.parametrize('interp', [False, True])
def test_lds_and_global_records_agree(gpu, facets, interp):
    import torch
    from marxs_amd.batch import _tables_with_budget
    from marxs_amd.tracer import CompiledInstrument
    from tests.test_gpu_launch_shapes import _launch, _same, _source
    ci = CompiledInstrument(_instrument(facets, interp))
    n = 10007
    src = _source(n)
    u = ci.draw_uniforms(n, torch.Generator(device='cuda').manual_seed(4))
    ref, st = _launch(ci, src, u, 64)
    ci.dev_tables = _tables_with_budget(ci, 0)
    got, st2 = _launch(ci, src, u, 64)
    _same(ref, got)
    assert torch.equal(st, st2)
