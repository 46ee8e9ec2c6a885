"""Decode of 4..15 rows with the qkv projection and the attention in one launch
against the separate launches: logits bit for bit, over split and unsplit
attention, windowed and full-causal layers, the smallest and largest width."""

import numpy as np
import pytest
import torch

from attention_nn_amd.config import GPTConfig
from attention_nn_amd.weights import init_params, perturb_lambdas

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,prompt", [(4, 4, 2), (5, 6, 40), (7, 6, 150), (15, 6, 300), (8, 1, 33)])
def test_one_launch_equals_two(B, H, prompt, monkeypatch):
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=1024, num_layers=3, num_heads=H, model_dim=128 * H, seq_len=512,
                    window=128, long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 5, dense=True))
    tok = np.random.default_rng(B).integers(0, 1000, (B, prompt + 8)).astype(np.int32)

    def run(val):
        monkeypatch.setenv("ANN_QKV_ATTN", val)
        eng = Engine(cfg, p, max_batch=B, max_ctx=512, max_tokens=B * prompt)
        eng.prefill(tok[:, :prompt])
        lgs = []
        for i in range(prompt, prompt + 8):
            _, lg = eng.decode(torch.from_numpy(tok[:, i].copy()).cuda(), want_logits=True)
            lgs.append(lg.cpu())
        eng.check_device()
        return torch.stack(lgs)

    assert torch.equal(run("1"), run("0"))
