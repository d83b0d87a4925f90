"""Training where the backward's values of all layers are too many to keep (256 MiB): layers take
turns with them, the chain waiting for the side stream's reads. Gradients of a deep narrow model
against the oracle's, as in test_gpu_train.py, after a second step as well; and what a layer adds to a
trainer's memory at 4096 positions, the longest: its weights' four arenas and its forward values,
nothing of the backward's."""
import ctypes as C
import os

import numpy as np
import pytest

import oracle
import stories_hip as sh
from helpers import tiny_config

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))


def test_layers_taking_turns_match_oracle(gpu):
    dim, hidden, layers, seq = 64, 64, 1901, 64
    assert 4 * seq * layers * (7 * dim + 2 * hidden) > 256 << 20
    cfg = tiny_config(dim=dim, hidden=hidden, n_layers=layers, n_heads=1, n_kv_heads=1, head_dim=64, vocab=96, max_seq=seq,
                      residual_scale=float((2 * layers) ** -0.5))
    w = sh.synth_weights(cfg, seed=401, std=0.1)
    tr = sh.Trainer(cfg, seq=seq, lr=1e-3)
    tr.upload(w)
    toks = sh.synth_tokens(2 * seq + 1, 402, cfg.vocab)
    p = oracle.TrainParams.from_weights(w)
    m, v, g = (oracle.TrainParams.zeros_like(p) for _ in range(3))
    inp, tgt = toks[:seq], toks[1:seq + 1]
    loss = tr.step_window(inp, tgt)
    want = oracle.train_step(oracle.config_from(cfg), p, m, v, g, oracle.hparams(lr=1e-3), 1, inp, tgt, threads=THREADS)
    assert abs(loss - want) <= 1e-4
    worst = 0.0
    for name, t in g.tensors():
        got = tr.read(sh.SH_TRAIN_GRADS, name, t.shape)
        worst = max(worst, float(np.max(np.abs(got - t))) / max(float(np.max(np.abs(t))), 1e-30))
    print(f"gradients: {worst:.1e} of each tensor's largest")
    assert worst <= 1e-3
    # the same step again on the same weights, twice: the same bits
    seen = []
    for _ in range(2):
        tr.upload(w)
        tr.step_window(toks[seq:2 * seq], toks[seq + 1:])
        seen.append([tr.read(sh.SH_TRAIN_GRADS, name, t.shape) for name, t in g.tensors()])
    assert all(np.array_equal(a, b) for a, b in zip(*seen))
    tr.close()


def test_memory_of_a_layer_at_the_longest_window(gpu):
    lib = sh.load()
    lib.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def taken(layers):
        free, total = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        before = free.value
        tr = sh.Trainer(sh.make_config(n_layers=layers, max_seq=S), seq=S)
        assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        tr.close()
        return before - free.value

    S, D, F, H = 4096, 768, 2048, 12
    taken(1)   # the runtime's own pools
    grown = taken(6) - taken(4)
    params = 4 * D * D + 3 * D * F + 2 * D
    forward = S * (8 * D + 3 * F + 2 + 3 * H)
    print(f"two layers: {grown / 2**20:.0f} MiB, arenas and forward values {2 * (16 * params + 4 * forward) / 2**20:.0f}")
    assert grown <= 2 * (16 * params + 4 * forward) + (32 << 20)
