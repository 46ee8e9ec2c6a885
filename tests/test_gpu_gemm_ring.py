"""The ring GEMM (gemm_ring.hip) at the sizes where its tiles and its K loop
can go wrong: every tile shape, row counts around a tile's edge, and fewer K
tiles than ring stages.  Logits of every position against the oracle."""

import numpy as np
import pytest
import torch

import oracle.ref_model as R
from attention_nn_amd.config import GPTConfig
from attention_nn_amd.weights import init_params, perturb_lambdas

pytestmark = pytest.mark.gpu

LOGIT_TOL = 2e-2    # the suite's bound: bf16 activations over the layers, logits below 23


# (model_dim, heads, vocab, batch, length): K of 64 (one K tile) to 3072; 129,
# 300 and 1027 rows end inside every tile height (32, 64, 128, 192); a
# vocabulary of whole 64-, 128- and 192-column tiles; 65 head-64 columns
@pytest.mark.parametrize("d,H,V,B,T", [
    (64, 1, 320, 1, 129), (128, 2, 384, 3, 100), (192, 3, 576, 1, 300), (320, 5, 1088, 2, 150),
    (256, 2, 1000, 1, 129), (512, 8, 1152, 1, 1027), (768, 6, 1216, 1, 129),
    (768, 6, 1536, 5, 385), (768, 6, 1280, 16, 193), (1536, 12, 1152, 2, 257),
])
def test_ring_gemm_logits_every_position(d, H, V, B, T):
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=V, num_layers=2, num_heads=H, model_dim=d, seq_len=T, window=70,
                    long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 5, dense=True))
    tok = np.random.default_rng(d + T).integers(0, V, (B, T))
    print(f"case ring d={d} H={H} V={V} B={B} T={T}", flush=True)
    got = Engine(cfg, p, max_batch=B, max_ctx=T, max_tokens=B * T).forward_logits(tok).cpu()
    assert (got - R.logits(cfg, p, tok)).abs().max().item() < LOGIT_TOL


@pytest.mark.parametrize("B", [3, 7, 40, 70])
def test_ring_gemm_whole_row_sampling_and_graph(B):
    """top_k 0 keeps z: the decode step's lm_head is the ring kernel on 3 .. 128
    rows, inside the captured step below 16 rows; the logits of replayed
    steps against the oracle's forward over the same ids."""
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=1216, num_layers=2, num_heads=2, model_dim=256, seq_len=32,
                    window=8, long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 6, dense=True))
    tok = np.random.default_rng(B).integers(0, cfg.vocab_size, (B, 6))
    print(f"case ring decode B={B}", flush=True)
    eng = Engine(cfg, p, max_batch=B, max_ctx=32, max_tokens=B * 6)
    nxt, _ = eng.prefill(tok, 0.9, 0, 3, 0)
    ids = [tok, nxt.cpu().numpy()[:, None]]
    lg = torch.empty((B, cfg.vocab_size), device="cuda")
    for i in range(4):
        nxt, lg = eng.decode(nxt, 0.9, 0, 3, i + 1, want_logits=True, out=nxt)
        ref = R.logits(cfg, p, np.concatenate(ids, 1))[:, -1]
        assert (lg.cpu() - ref).abs().max().item() < LOGIT_TOL
        ids.append(nxt.cpu().numpy()[:, None])
    eng.check_device()
