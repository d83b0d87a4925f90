"""The prompt forward's attention over the KV cache it fills (k_attn_cache), where it can go
wrong: segments one off a 64-key block and a 128-query tile, sequences of rows that do not start
on a tile, head dims 64 and 128, fp16 and bf16, one to eight q heads' worth of grid at the line
that its dispatch draws. Batched prompts against the oracle's single-sequence decoder: the first
new token's logits of three sequences, 2-norm of the difference over that of the logits. A key or value
of the cache that is rounded the other way makes up to 4.5e-4 in bf16 and 5.7e-5 in fp16 (an fp32 cache:
8e-6); dropping the lo plane of Q, P or the output makes 8.7e-4 to 2.8e-3 in bf16 and 1.1e-4 to 3.5e-4 in
fp16, leaving out one key of the last row 0.05 to 0.1 (the float64 model with the mistake planted)."""
import numpy as np
import pytest

import oracle
import stories_hip as sh
from helpers import random_gains, tiny_config
from test_gpu_seams import THREADS

pytestmark = pytest.mark.gpu

GQA128 = dict(dim=256, hidden=256, n_layers=2, n_heads=4, n_kv_heads=2, head_dim=128, vocab=512, qk_norm=1,
              rope_theta=1e6, norm_eps=1e-6)
MHA64 = dict(dim=256, hidden=256, n_layers=2, n_heads=4, n_kv_heads=4, head_dim=64, vocab=512)


@pytest.mark.parametrize("shape,dtype,kv,seqs,seg", [
    (GQA128, sh.SH_DTYPE_BF16, sh.SH_KV_BF16, 32, 96),     # the shortest it takes; the grid at its line
    (GQA128, sh.SH_DTYPE_BF16, sh.SH_KV_BF16, 16, 129),    # two query tiles, the second of one row
    (GQA128, sh.SH_DTYPE_F16, sh.SH_KV_F16, 11, 257),
    (GQA128, sh.SH_DTYPE_BF16, sh.SH_KV_BF16, 32, 127),
    (MHA64, sh.SH_DTYPE_F16, sh.SH_KV_F16, 32, 128),
    (MHA64, sh.SH_DTYPE_BF16, sh.SH_KV_BF16, 17, 191),
    (GQA128, sh.SH_DTYPE_BF16, sh.SH_KV_BF16, 31, 95),     # below both lines: the 64-query form
    (MHA64, sh.SH_DTYPE_BF16, sh.SH_KV_F32, 16, 130),      # a cache of another type: not read back
])
def test_prompt_attention(gpu, shape, dtype, kv, seqs, seg):
    cfg = tiny_config(**shape, max_seq=seg + 8, kv_dtype=kv, max_batch=32)
    w = random_gains(sh.synth_weights(cfg, seed=501, std=0.05), 502)
    m = sh.Model(cfg, dtype)
    m.upload(w)
    prompts = sh.synth_tokens(seqs * (seg + 1), 503, cfg.vocab).reshape(seqs, seg + 1)
    rows = [0, seqs // 2, seqs - 1]
    _, got = m.batch_greedy_decode_logits(prompts, 1, rows)
    m.close()
    ref = oracle.Decoder(oracle.config_from(cfg), w.rounded(dtype), threads=THREADS)
    for k, b in enumerate(rows):
        ref.reset()
        for p in range(seg + 1):
            want = ref.forward_one(int(prompts[b, p]), p)
        err = float(np.linalg.norm(got[0, k].astype(np.float64) - want) / np.linalg.norm(want))
        print(f"sequence {b}: {err:.2e}")
        assert err <= {sh.SH_KV_BF16: 8e-4, sh.SH_KV_F16: 1e-4, sh.SH_KV_F32: 3e-5}[kv]
