"""MoE batches on the fp32-precision grouped GEMMs (llg_moe_split.hip) against a
float64 reference, at the sizes where they can go wrong: one and two 16-row
groups and several tiles per expert, rows of 1 to 9 blocks past a whole number
of 4-block chunks, widths below and off a workgroup's columns, K slices.

The bound: a sum of n fp32 terms in any order is within n * 2^-24 of
sum |terms|; here n is under 2^10 (chunks, slices and the pieces' products) and
the terms' magnitudes are within about 16 times the result's largest value, so
10 * 2^-24 * 16 ~ 1e-5 of it holds with room for random signs."""
import numpy as np
import pytest

import llg
import llg.gguf as gg
from tests.helpers import deq, max_rel_err, normal, quant

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module")
def dev():
    d = llg.Device()
    yield d
    d.close()


def reference(x, ids, w, gate, up, down, t, d, eff, k):
    g = deq(gate, t, d).astype(np.float64).reshape(-1, eff, d)
    u = deq(up, t, d).astype(np.float64).reshape(-1, eff, d)
    dn = deq(down, t, eff).astype(np.float64).reshape(-1, d, eff)
    out = np.zeros(x.shape)
    for i, row in enumerate(x.astype(np.float64)):
        for s in range(k):
            e = ids[i, s]
            a = g[e] @ row
            out[i] += w[i, s] * (dn[e] @ (a / (1 + np.exp(-a)) * (u[e] @ row)))
    return out


def run(dev, rng, t, d, eff, E, k, x):
    router = normal(rng, (E, d), 0.2)
    gate = quant(normal(rng, (E * eff, d), 0.02), t)
    up = quant(normal(rng, (E * eff, d), 0.02), t)
    down = quant(normal(rng, (E * d, eff), 0.02), t)
    hs = (dev.upload_f32(router), dev.upload_matrix(gate, t, E * eff, d),
          dev.upload_matrix(up, t, E * eff, d), dev.upload_matrix(down, t, E * d, eff))
    out, ids, w = llg.moe_ffn(dev, *hs, E, k, x)
    again = llg.moe_ffn(dev, *hs, E, k, x)[0]
    for h in hs:
        h.release()
    assert np.array_equal(out, again, equal_nan=True)
    return out, reference(x, ids, w, gate, up, down, t, d, eff, k)


@pytest.mark.parametrize("t", [gg.Q4_0, gg.Q8_0, gg.F16])
@pytest.mark.parametrize("d,eff,E,k,n_tok", [
    (32, 32, 1, 1, 16),      # one block, one expert, one full row group
    (96, 544, 4, 2, 17),     # ragged chunks; two row groups
    (160, 96, 2, 1, 65),     # several tiles per expert
    (2080, 1440, 8, 2, 33),  # K slices of odd chunk counts
    (288, 256, 16, 4, 40),   # many experts of few rows
])
def test_batch_matches_float64(dev, t, d, eff, E, k, n_tok):
    rng = np.random.default_rng(d + eff + n_tok)
    out, ref = run(dev, rng, t, d, eff, E, k, normal(rng, (n_tok, d), 1.0))
    for i in range(n_tok):
        assert max_rel_err(out[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("t", [gg.Q4_0, gg.Q8_0, gg.F16])
@pytest.mark.parametrize("mag", [1e-12, 3e4, 1e15])
def test_batch_scales_and_outliers(dev, t, mag):
    """Activations far from 1 (no piece may overflow or vanish; the result, about
    mag^2 / 1e6, stays inside the fp32 range at both ends), each row with
    one element 1e5 times the others (its chunk's power of two is set by it)."""
    rng = np.random.default_rng(5)
    d, eff, n_tok = 288, 416, 32  # not the f16 GEMMs' widths
    x = normal(rng, (n_tok, d), mag * 1e-5)
    x[np.arange(n_tok), rng.integers(0, d, n_tok)] = mag
    out, ref = run(dev, rng, t, d, eff, 4, 2, x)
    for i in range(n_tok):
        if np.all(np.isfinite(ref[i].astype(np.float32))):
            assert max_rel_err(out[i], ref[i]) <= TOL, i


@pytest.mark.parametrize("t", [gg.Q4_0, gg.Q8_0, gg.F16])
def test_batch_non_finite_rows_stay_apart(dev, t):
    """A token with an infinity or a NaN leaves the other tokens' outputs as
    they are without it (they share tiles and chunks)."""
    d, eff, n_tok = 288, 416, 32  # not the f16 GEMMs' widths
    rng = np.random.default_rng(6)
    x = normal(rng, (n_tok, d), 1.0)
    good, _ = run(dev, np.random.default_rng(7), t, d, eff, 4, 2, x)
    bad = x.copy()
    bad[3, 5], bad[20, 287] = np.inf, np.nan
    out, _ = run(dev, np.random.default_rng(7), t, d, eff, 4, 2, bad)
    rest = [i for i in range(n_tok) if i not in (3, 20)]
    assert np.array_equal(out[rest], good[rest])
    assert not np.isfinite(out[3]).any() and not np.isfinite(out[20]).any()


def test_f16_subnormal_weights(dev):
    """F16 weights below 2^-14 keep their value in the products."""
    rng = np.random.default_rng(8)
    d, eff, E, n_tok = 64, 64, 1, 16
    x = normal(rng, (n_tok, d), 1.0)
    gate, up = normal(rng, (eff, d), 2e-6), normal(rng, (eff, d), 2e-6)
    down = normal(rng, (d, eff), 1.0)
    q = [quant(w, gg.F16) for w in (gate, up, down)]
    hs = [dev.upload_f32(normal(rng, (E, d), 0.2))] + [
        dev.upload_matrix(w, gg.F16, r, c) for w, r, c in zip(q, (eff, eff, d), (d, d, eff))]
    out, ids, w = llg.moe_ffn(dev, *hs, E, 1, x)
    ref = reference(x, ids, w, *q, gg.F16, d, eff, 1)
    for i in range(n_tok):
        assert max_rel_err(out[i], ref[i]) <= TOL, i
    for h in hs:
        h.release()
