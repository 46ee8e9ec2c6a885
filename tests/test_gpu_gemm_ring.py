"""The ring GEMM (gemm_ring.hip) at the sizes where its tiles and its K loop
can go wrong: every tile of every epilogue that takes it, row counts around a
tile's edge, and fewer K tiles than ring stages.  Logits of every position, row
losses and decode steps against the oracle."""

import ctypes

import numpy as np
import pytest
import torch

import oracle.ref_model as R
from attention_nn_amd import _lib
from attention_nn_amd.config import GPTConfig
from attention_nn_amd.weights import init_params, perturb_lambdas

pytestmark = pytest.mark.gpu

LOGIT_TOL = 2e-2    # the suite's bound: bf16 activations over the layers, logits below 23

# (model_dim, heads, vocab, batch, length): K of 64 (one K tile) to 3072; 129,
# 300, 1027, 5500 and 8245 rows end inside every tile height (32, 64, 128, 192);
# a vocabulary of whole 64-, 128- and 192-column tiles; head-64 widths that are no
# multiple of 128 (the plain store).  tests/test_gemm_ring_tiles.py checks that
# they reach every tile of every epilogue.
CASES = [
    (64, 1, 320, 1, 129), (128, 2, 384, 3, 100), (192, 3, 576, 1, 300), (320, 5, 1088, 2, 150),
    (256, 2, 1000, 1, 129), (512, 8, 1152, 1, 1027), (768, 6, 1216, 1, 129),
    (768, 6, 1536, 5, 385), (768, 6, 1280, 16, 193), (1536, 12, 1152, 2, 257),
    (320, 5, 576, 2, 300), (704, 11, 576, 3, 500), (704, 11, 576, 8, 253), (256, 2, 4224, 5, 499),
    (768, 6, 1152, 8, 513), (768, 6, 1152, 11, 500), (768, 6, 1280, 17, 485),
]


@pytest.mark.parametrize("d,H,V,B,T", CASES)
def test_ring_gemm_logits_every_position(d, H, V, B, T):
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=V, num_layers=2, num_heads=H, model_dim=d, seq_len=T, window=70,
                    long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 5, dense=True))
    tok = np.random.default_rng(d + T).integers(0, V, (B, T))
    print(f"case ring d={d} H={H} V={V} B={B} T={T}", flush=True)
    got = Engine(cfg, p, max_batch=B, max_ctx=T, max_tokens=B * T).forward_logits(tok).cpu()
    assert (got - R.logits(cfg, p, tok)).abs().max().item() < LOGIT_TOL


# 128- and 192-column tiles, the last of them whole, of 64, 65 and 188 columns,
# and the only one (70 columns); ragged last row blocks
@pytest.mark.parametrize("d,H,V,B,T,cols", [(128, 1, 2432, 2, 150, 128), (128, 1, 2112, 2, 150, 128),
                                            (128, 1, 2113, 2, 150, 128), (192, 3, 2304, 5, 386, 192),
                                            (192, 3, 2300, 5, 386, 192), (64, 1, 4608, 1, 33, 128),
                                            (64, 1, 70, 1, 20, 128)])
def test_ring_gemm_loss_tiles(d, H, V, B, T, cols, traced):
    """Row losses and their mean; the suite's bounds of the training forward."""
    from attention_nn_amd.engine import Engine
    cfg = GPTConfig(vocab_size=V, num_layers=2, num_heads=H, model_dim=d, seq_len=T, window=70,
                    long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 7, dense=True))
    rng = np.random.default_rng(V + T)
    tok, tgt = rng.integers(0, V, (B, T)), rng.integers(0, V, (B, T))
    tgt.reshape(-1)[[0, -1]] = V - 1, 0      # the last and the first column
    print(f"case ring loss d={d} V={V} B={B} T={T}", flush=True)
    eng = Engine(cfg, p, max_batch=B, max_ctx=T, max_tokens=B * T)
    mean, rows = eng.forward_loss(tok, tgt, rows=True)
    rm, rr = R.loss(cfg, p, tok, tgt, banded_bf16=True)
    assert (rows.cpu().double() - rr.double()).abs().max().item() < 1e-2
    assert abs(mean.item() - rm.item()) < 5e-4
    names = traced(lambda: eng.forward_loss(tok, tgt))
    assert any(f"k_gemm_ring<6, 128, {cols}," in n for n in names)


@pytest.mark.parametrize("B,H,persist,graph", [(3, 2, "0", True), (7, 2, None, False),
                                               (5, 4, None, True), (12, 4, None, True),
                                               (40, 2, None, False), (70, 2, None, False)])
def test_ring_gemm_whole_row_sampling_and_graph(B, H, persist, graph, monkeypatch, traced):
    """top_k 0 keeps z: the decode step's lm_head is the ring kernel on 3 .. 128
    rows (a vocabulary above eight times the width), inside the captured step
    where the qkv projection and the attention are launches of their own below 16
    rows (head dim 64 here, or 3 rows without the persistent kernel).  One set of
    buffers over the steps, so that the step captured first is replayed; the
    logits of every step against the oracle's forward over the same ids."""
    from attention_nn_amd.engine import Engine, _ptr
    from attention_nn_amd._stream import current_stream
    if persist is not None:
        monkeypatch.setenv("ANN_PERSIST", persist)
    cfg = GPTConfig(vocab_size=2112, num_layers=2, num_heads=H, model_dim=256, seq_len=32,
                    window=8, long_layers=(1,))
    p = perturb_lambdas(init_params(cfg, 6, dense=True))
    tok = np.random.default_rng(B).integers(0, cfg.vocab_size, (B, 6))
    print(f"case ring decode B={B} H={H}", flush=True)
    eng = Engine(cfg, p, max_batch=B, max_ctx=32, max_tokens=B * 6)
    nxt, _ = eng.prefill(tok, 0.9, 0, 3, 0)
    ids = [tok, nxt.cpu().numpy()[:, None]]
    lg = torch.empty((B, cfg.vocab_size), device="cuda")

    def step(i):
        s = eng._sampling(0.9, 0, 3, i)
        _lib.check(_lib.lib().ann_decode_step(eng._ctx, _ptr(nxt), B, ctypes.byref(s), _ptr(nxt),
                                              _ptr(lg), current_stream()))

    names = []
    for i in range(5):
        names.append(traced(lambda: step(i + 1), tries=1))
        ref = R.logits(cfg, p, np.concatenate(ids, 1))[:, -1]
        assert (lg.cpu() - ref).abs().max().item() < LOGIT_TOL
        ids.append(nxt.cpu().numpy()[:, None])
    eng.check_device()
    for i, n in enumerate(names):
        # (a replay's kernels are not always in the trace)
        assert graph or any("k_gemm_ring<4," in k for k in n)
        assert any("hipGraphLaunch" in k for k in n) == graph
        # the first step captures and instantiates, the others replay
        assert any("hipGraphInstantiate" in k for k in n) == (graph and i == 0)
