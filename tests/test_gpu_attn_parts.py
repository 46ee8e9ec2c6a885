"""The prefill attention's key parts: prompts whose grids take four, two and
one part, lengths around the query blocks (32, 64, 128) and key stages (128
keys), window and full-causal layers.  Logits of every position against the
oracle."""

import numpy as np
import pytest

import oracle.ref_model as R
from attention_nn_amd.config import GPTConfig
from attention_nn_amd.weights import init_params, perturb_lambdas

pytestmark = pytest.mark.gpu

LOGIT_TOL = 2e-2    # the suite's bound: bf16 activations over the layers, logits below 23


@pytest.mark.parametrize("H,dh,B,T,window", [
    (2, 128, 1, 130, 1), (2, 128, 1, 161, 33), (2, 128, 3, 257, 128), (2, 128, 1, 700, 384),
    (4, 128, 20, 129, 60), (4, 128, 40, 192, 100), (4, 128, 70, 128, 50),
    (4, 64, 1, 159, 31), (4, 64, 2, 515, 200), (4, 64, 30, 161, 64), (4, 64, 66, 130, 129),
])
def test_prefill_attention_key_parts(H, dh, B, T, window):
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=512, num_layers=2, num_heads=H, model_dim=H * dh, seq_len=T,
                    window=window, long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 8, dense=True))
    tok = np.random.default_rng(B * T).integers(0, cfg.vocab_size, (B, T))
    print(f"case key parts H={H} dh={dh} B={B} T={T} window={window}", flush=True)
    got = Engine(cfg, p, max_batch=B, max_ctx=T, max_tokens=B * T).forward_logits(tok).cpu()
    assert (got - R.logits(cfg, p, tok)).abs().max().item() < LOGIT_TOL
