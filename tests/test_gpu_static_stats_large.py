"""Sums of many orders over several 1e8 photons from the static workspace,
which takes the orders in several calls then (needs an MI355X).  Probabilities
of 1 add up to the counts exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,no', [(1000003, 64), (660000011, 64), (660000011, 63)])
def test_sums(gpu, n, no):
    import ctypes
    import torch
    from marxs_amd import _lib
    order = torch.arange(n, dtype=torch.int32, device=gpu).remainder_(no + 3)
    prob = torch.ones(n, dtype=torch.float64, device=gpu)
    orders = torch.arange(no, dtype=torch.int32, device=gpu)
    total = torch.full((no,), -1., dtype=torch.float64, device=gpu)
    count = torch.full((no,), -1, dtype=torch.int64, device=gpu)
    a = _lib.MxOrderStats()
    a.n, a.n_orders = n, no
    a.order, a.prob, a.orders = order.data_ptr(), prob.data_ptr(), orders.data_ptr()
    a.prob_sum, a.count = total.data_ptr(), count.data_ptr()
    _lib.check(_lib.lib.mx_order_stats_static(ctypes.byref(a), torch.cuda.current_stream().cuda_stream))
    want = n // (no + 3) + (np.arange(no) < n % (no + 3))
    assert np.array_equal(count.cpu().numpy(), want)
    assert np.array_equal(total.cpu().numpy(), want.astype(float))
