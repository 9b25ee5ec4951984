"""The per-token MoE combine at its edges: one and eight slots, widths below and
off a workgroup's 128 outputs, and down rows of 9 chunks (one past the batch of
loads a thread holds), against float64 over the exactly dequantized experts."""
import numpy as np
import pytest

import llg
import llg.gguf as gg
from tests.helpers import max_rel_err, normal, quant
from tests.test_gpu_moe_split import reference

pytestmark = pytest.mark.gpu
TOL = 1e-4  # of the largest output; the Q4_0 dots' offset shows about 1e-5


@pytest.mark.parametrize("t", [gg.Q4_0, gg.F16])
@pytest.mark.parametrize("d,eff,E,k,n_tok", [(32, 64, 1, 1, 1), (160, 96, 8, 8, 1), (160, 96, 9, 2, 2),
                                             (32, 16416, 2, 2, 1)])
def test_per_token_combine(t, d, eff, E, k, n_tok):
    rng = np.random.default_rng(d + eff)
    mats = [quant(normal(rng, s, 0.02), t) for s in ((E * eff, d), (E * eff, d), (E * d, eff))]
    x = normal(rng, (n_tok, d), 1.0)
    with llg.Device() as dev:
        hs = [dev.upload_f32(normal(rng, (E, d), 0.2))]
        hs += [dev.upload_matrix(m, t, r, c)
               for m, r, c in zip(mats, (E * eff, E * eff, E * d), (d, d, eff))]
        out, ids, w = llg.moe_ffn(dev, *hs, E, k, x)
    ref = reference(x, ids, w, *mats, t, d, eff, k)
    for i in range(n_tok):
        assert max_rel_err(out[i], ref[i]) <= TOL, i
