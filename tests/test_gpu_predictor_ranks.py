"""The predictor and the fused step at ranks around the logit tiles' limits
(groups of 4 and 16, 128 and 256 units per row, the scalar loop past them) and
at layer sizes that change the hidden units per predictor workgroup, against
the oracle.

The threshold sits in the middle of the widest gap near the wanted count, far
above the rounding of a logit (a dot of `rank` terms), so the active set has
to be identical; the output's bound is the one of every FFN output."""
import numpy as np
import pytest

import llg
import llg.gguf as gg
from oracle import refcpu as R
from tests.helpers import make_sparse_layer, max_rel_err, normal, ref_sparse_f64

pytestmark = pytest.mark.gpu
TOL = 1e-4  # max |difference| / max |output|; fp32 sums show about 1e-5


@pytest.fixture(scope="module")
def dev():
    d = llg.Device()
    yield d
    d.close()


def gap_threshold(logits, n):
    s = np.sort(logits.astype(np.float64))[::-1]
    lo, hi = max(0, n - 8), min(s.size - 1, n + 8)
    i = lo + int(np.argmax(s[lo:hi] - s[lo + 1:hi + 1]))
    return float(np.float32((s[i] + s[i + 1]) / 2))


def check(dev, t, h, ff, rank, bias=False):
    rng = np.random.default_rng(1000 * rank + h)
    up, dn = make_sparse_layer(rng, h, ff, t)
    wup, wout = normal(rng, (rank, h), 0.05), normal(rng, (ff, rank), 0.05)
    b = normal(rng, ff, 0.1) if bias else None
    x, a = normal(rng, h, 1.0), normal(rng, h, 1.0)
    _, lg = R.predict(wup, wout, b, a, 0.0)
    thr = gap_threshold(lg, max(1, ff // 20))
    ref_act, _ = R.predict(wup, wout, b, a, thr)
    bundle = dev.upload_bundle(up, dn, t, h, ff)
    pred = llg.Predictor(dev, wup, wout, b, thr)
    for _ in range(2):  # the second step reads slots of an older epoch
        out, act = llg.ffn_predict_sparse(dev, pred, bundle, a, x)
        assert np.array_equal(act, ref_act)
        assert max_rel_err(out, ref_sparse_f64(up, dn, t, h, x, ref_act)) <= TOL
    pred.w_up.release()
    pred.w_out.release()
    bundle.release()


@pytest.mark.parametrize("t", [gg.Q4_0, gg.Q8_0, gg.F16])
@pytest.mark.parametrize("rank", [1, 3, 15, 17, 100, 127, 128, 129, 131, 240, 255, 256, 257])
def test_step_at_rank(dev, t, rank):
    check(dev, t, 160, 1000, rank, bias=rank % 2 == 1)


@pytest.mark.parametrize("t,h,ff,rank", [
    (gg.Q8_0, 64, 14336, 33),   # twice the units per predictor workgroup
    (gg.Q8_0, 64, 14336, 100),  # 4 times
    (gg.Q8_0, 96, 14336, 256),  # 8 times
    (gg.Q8_0, 64, 24000, 200),  # more tiles than CUs: the most units
    (gg.Q4_0, 96, 18176, 250),  # twice, of Q4_0's two
    (gg.F16, 96, 12288, 255),
])
def test_step_units_per_workgroup(dev, t, h, ff, rank):
    check(dev, t, h, ff, rank)
