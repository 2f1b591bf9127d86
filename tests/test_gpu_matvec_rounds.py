"""Decode steps of models whose K-quant rows take two, three or four units per
wave (hidden 2304: 9 units of 256 columns over 8 waves; ffn 4352 and 6400: 17
and 25), which the matvec requests all at once, and hidden 2048, one unit per
wave. Logits against the oracle's at each step, at test_gpu_model's bar, with
the same argmax.
"""
import numpy as np
import pytest

import oracle
from phonemap_amd import api
from tests.test_gpu_model import TOL, _model_file
from tests.util import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", [10, 11, 12, 13, 14])
@pytest.mark.parametrize("hidden,ffn", [(2304, 4352), (2304, 6400), (2048, 8192)])
def test_decode_steps(qtype, hidden, ffn):
    spec = dict(n_layers=1, hidden=hidden, n_heads=hidden // 64, n_kv_heads=hidden // 256, head_dim=64, ffn=ffn,
                vocab=512, context_length=64, seed=hidden + ffn + qtype, layer_type=qtype, scale_mode=1)
    path = _model_file("rounds_%d_%d_%d" % (qtype, hidden, ffn), **spec)
    print("rounds", qtype, hidden, ffn, flush=True)
    om = oracle.Model(path, 64, "f16")
    with api.Model(path, max_context=64) as m:
        tok = 7
        for pos in range(6):
            lg, am = m.eval_token(tok, pos)
            olg = om.forward(tok, pos)
            assert rel_err(lg, olg) <= TOL, pos
            assert am == oracle.argmax(olg) == int(np.argmax(lg)), pos
            tok = am
    om.close()
