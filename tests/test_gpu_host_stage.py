"""The host-buffer sparse calls through the pinned staging area: the smallest
sizes, list lengths off a 16-byte unit, no and every neuron active, and a call
above the staging limit (1 MiB, pageable copies) between staged ones, so that
a result never shows an earlier call's bytes."""
import numpy as np
import pytest

import llg
import llg.gguf as gg
from tests.helpers import make_sparse_layer, max_rel_err, normal, ref_sparse_f64

pytestmark = pytest.mark.gpu
TOL = 1e-4  # fp32 sums show about 1e-5 of the largest output


@pytest.fixture(scope="module")
def dev():
    d = llg.Device()
    yield d
    d.close()


@pytest.mark.parametrize("h,ff,n", [(32, 64, 1), (160, 1000, 13), (544, 2001, 2001),
                                    (32, 270000, 5000), (96, 333, 7)])
def test_staged_calls(dev, h, ff, n):
    rng = np.random.default_rng(h + ff)
    t = gg.Q4_0
    up, dn = make_sparse_layer(rng, h, ff, t)
    b = dev.upload_bundle(up, dn, t, h, ff)
    x = normal(rng, h, 1.0)
    active = np.sort(rng.choice(ff, n, replace=False)).astype(np.int32)
    ref = ref_sparse_f64(up, dn, t, h, x, active)
    assert max_rel_err(llg.ffn_sparse_load(dev, b, x, active), ref) <= TOL
    wup, wout = normal(rng, (4, h), 0.05), np.zeros((ff, 4), np.float32)
    bias = np.full(ff, -1.0, np.float32)
    for chosen in (active, np.arange(0), active[::2]):  # logits are the bias
        bias[:] = -1.0
        bias[chosen] = 1.0
        pred = llg.Predictor(dev, wup, wout, bias, 0.0)
        out, act = llg.ffn_predict_sparse(dev, pred, b, x, x)
        assert np.array_equal(act, chosen)
        ref = ref_sparse_f64(up, dn, t, h, x, chosen) if len(chosen) else np.zeros(h)
        assert max_rel_err(out, ref) <= TOL
        pred.w_up.release()
        pred.w_out.release()
    b.release()
