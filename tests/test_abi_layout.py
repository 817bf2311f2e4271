"""The table layout that include/marxs_hip.h states is the one that the
compiler writes, and its version tells it from the one with FP64 test records
of 16 words and no detector records (CPU only)."""
import ctypes
import os
import re
import subprocess

import numpy as np

from marxs_amd import _lib, configs
from marxs_amd.compiler import STAGE_DETECTOR, compile_tree

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = open(os.path.join(ROOT, 'include', 'marxs_hip.h')).read()


def _const(name):
    return int(re.search(rf'#define {name} (\d+)', HEADER).group(1))


def test_version_of_the_layout():
    """21 was the layout of 16 words: a caller with tables of that version has
    to be told apart by the version alone."""
    assert _lib.lib.mx_abi_version() == _lib.MX_ABI_VERSION == _const('MX_ABI_VERSION') >= 22


def test_records_have_the_stated_widths():
    t = compile_tree(configs.cat_rowland_instrument(60)[0])
    words, detector, et = _const('MX_LT64'), _const('MX_DR'), _const('MX_ET')
    seen = 0
    for s, st in enumerate(t.stages):
        n, e0 = len(st.elements), st.elem0
        o64, o32 = int(t.stage_i[s, 21]), int(t.stage_i[s, 20])
        if n < 2:
            continue
        rec = t.lds_image64[o64:o64 + 8 * words * n].view(np.float64).reshape(n, words)
        assert np.array_equal(rec, t.elem_t[e0:e0 + n, :words])
        rec = t.lds_image32[o32:o32 + 4 * et * n].view(np.float32).reshape(n, et)
        assert np.array_equal(rec, t.elem_t32[e0:e0 + n])
        if st.kind != STAGE_DETECTOR:
            continue
        for image, col in ((t.lds_image32, 51), (t.lds_image64, 52)):
            o = int(t.stage_i[s, col])
            assert o > 0
            rec = image[o:o + 8 * detector * n].view(np.float64).reshape(n, detector)
            assert np.array_equal(rec[:, :12], t.elem_t[e0:e0 + n, :12])
            assert np.array_equal(rec[:, 12:16], t.elem_p[e0:e0 + n, 6:10])
            assert np.array_equal(np.ascontiguousarray(rec[:, 16:]).view(np.int32)[:, :3],
                                  t.elem_i[e0:e0 + n][:, [0, 4, 5]])
            seen += 1
    assert seen == 2


def test_adjoint_step_struct(tmp_path):
    src = ['#include <stdio.h>', '#include <stddef.h>', '#include "marxs_hip.h"', 'int main(void) {',
           'printf("%zu\\n", sizeof(MxAdjointStep));']
    names = [f[0] for f in _lib.MxAdjointStep._fields_]
    src += [f'printf("%zu\\n", offsetof(MxAdjointStep, {f}));' for f in names] + ['return 0; }']
    (tmp_path / 'a.c').write_text('\n'.join(src))
    subprocess.run(['gcc', '-I', os.path.join(ROOT, 'include'), str(tmp_path / 'a.c'), '-o', str(tmp_path / 'a')],
                   check=True)
    out = subprocess.run([str(tmp_path / 'a')], capture_output=True, text=True, check=True).stdout.split()
    assert [int(x) for x in out] == [ctypes.sizeof(_lib.MxAdjointStep)] + \
        [getattr(_lib.MxAdjointStep, f).offset for f in names]
