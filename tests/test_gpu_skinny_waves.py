"""Decode steps whose o and proj projections take eight waves (one to 24 k-steps
a wave, rounds with a remainder, row counts that do not fill a tile) and, above
one work-group per CU, four: logits against the oracle's KV-cache forward."""

import numpy as np
import pytest

import oracle.ref_model as R
from attention_nn_amd.config import GPTConfig
from attention_nn_amd.weights import init_params, perturb_lambdas

pytestmark = pytest.mark.gpu

LOGIT_TOL = 2e-2    # the suite's bound: bf16 activations over the layers, logits below 23


@pytest.mark.parametrize("d,H,B", [(256, 2, 5), (256, 4, 100), (512, 8, 5), (512, 4, 33), (768, 6, 7),
                                   (768, 6, 81), (1024, 8, 17), (1280, 10, 6), (1536, 12, 9)])
def test_decode_projections_over_waves(d, H, B):
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=640, num_layers=2, num_heads=H, model_dim=d, seq_len=16, window=5,
                    long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 9, dense=True))
    tok = np.random.default_rng(d + B).integers(0, cfg.vocab_size, (B, 5))
    print(f"case skinny d={d} H={H} B={B}", flush=True)
    eng = Engine(cfg, p, max_batch=B, max_ctx=16, max_tokens=B * 5)
    eng.prefill(tok[:, :3])
    prep, cache = R.Prepared(cfg, p), R.KVCache(cfg.num_layers)
    R.forward(prep, tok[:, :3], cache)
    for i in (3, 4):
        _, lg = eng.decode(tok[:, i], want_logits=True)
        ref = R.forward(prep, tok[:, i:i + 1], cache)[:, -1]
        assert (lg.cpu() - ref).abs().max().item() < LOGIT_TOL
    eng.check_device()
