"""The 16-bit GEMM's tile shapes at their edges (k_linear_few, k_gemm_pipe and k_gemm_ring,
chosen by linear_few and gemm_plan, whose choice each case names): row counts one off a tile, K
ranges of one step, of an odd number of steps and of an uneven split, N that fits only the
narrower tiles, and each epilogue, through the entry points.

ConvEval (fp16 weights, activations as hi/lo pairs of fp16) against float64. Each output's error
is at most (2^-21 + (K + 2) * 2^-23) * sum |w x|, the pair's 22 bits and two fp32 roundings per
element of the sum. And in every block of 16 x 16 results, the least that a wave computes, the root mean
square of the error is at most 4 * (2^-24 * sqrt(K / 16 + 8) + 2^-22) of that of all results: a sum of K / 32
products of each plane, rounded each time, and the pair's rounding. One fp16 plane in the place of the
pair exceeds that in every case (checked on the CPU). The layer seam and EvalLogits against the
oracle keep the bars of their own tests."""
import numpy as np
import pytest

import oracle
import plan
import stories_hip as sh
from helpers import tiny_config, tiny_gqa_config
from test_zz_no_alloc import Hip
from test_gpu_seams import THREADS, build, embed_cf, rel_err

pytestmark = pytest.mark.gpu


def block_rms(e):
    """Root mean squares of the 16 x 16 blocks of e."""
    r, c = np.arange(0, e.shape[0], 16), np.arange(0, e.shape[1], 16)
    n = np.add.reduceat(np.add.reduceat(np.ones_like(e), r, 0), c, 1)
    return np.sqrt(np.add.reduceat(np.add.reduceat(e * e, r, 0), c, 1) / n)


def block_bar(K):
    return 4 * (2.0 ** -24 * np.sqrt(K / 16 + 8) + 2.0 ** -22)


@pytest.mark.parametrize("kernel,s,in_dim,out_dim", [
    ("few", 1, 2048, 4096), ("few", 15, 4096, 64), ("few", 16, 1056, 192), ("few", 17, 1536, 448),   # one launch
    ("few", 31, 224, 4096), ("few", 128, 768, 768), ("few", 127, 32, 1024), ("few", 1, 32, 64), ("few", 3, 64, 64),
    ("few", 65, 96, 192), ("few", 31, 1056, 64), ("few", 33, 1056, 1088), ("few", 64, 416, 448),
    ("few", 65, 192, 768), ("few", 129, 768, 768),
    # K of one to three steps, fewer than the ring's slots
    ("ring32x64/1", 300, 32, 1024), ("ring32x64/1", 299, 96, 1024), ("ring64x64/1", 301, 32, 6144),
    ("ring64x64/1", 193, 96, 4096), ("ring64x128/1", 1501, 32, 4096), ("ring64x128/1", 531, 64, 6144),
    # uneven K ranges, K % 64 == 32
    ("ring32x64/4", 33, 1568, 1088), ("ring32x64/4", 200, 1568, 256), ("ring32x64/4", 33, 2016, 192),
    # the pipelined 32 x 32 tiles, split and unsplit
    ("pipe32/4", 65, 2048, 192), ("pipe32/2", 257, 768, 768), ("pipe32/1", 700, 256, 1024),
    # sums of 512 of K at a time: an uneven last run, none, every kernel that has them
    ("pipe32/1 in runs", 1024, 768, 768), ("ring64x64/1 in runs", 1091, 2048, 768), ("ring128x128/1 in runs", 1091, 768, 2048),
    ("ring64x128/1 in runs", 1501, 1536, 1024), ("ring32x64/2", 1024, 1568, 512),
    ("ring64x64/1 in runs", 300, 2016, 2560), ("ring32x64/1 in runs", 190, 1632, 4096),
    ("ring64x128/1", 513, 512, 4096), ("ring64x128/1", 577, 768, 2304),
    ("ring128x128/1", 127, 768, 32000), ("ring128x128/1", 1023, 1024, 3072), ("ring128x128/1", 641, 1024, 4096),
    ("ring128x128/1", 193, 768, 32000), ("ring128x256/1", 2049, 512, 6144),
])
def test_conv_eval_tile_shapes(gpu, kernel, s, in_dim, out_dim):
    assert plan.conv_kernel(s, in_dim, out_dim) == kernel
    rng = np.random.default_rng(s + in_dim + out_dim)
    w = (rng.standard_normal((out_dim, in_dim), np.float32) * 0.05).astype(np.float32)
    x = rng.standard_normal((s, in_dim), np.float32)
    conv = sh.Conv(w)
    got = conv.eval(x)
    conv.close()
    w16 = w.astype(np.float16).astype(np.float64)
    want = x.astype(np.float64) @ w16.T
    bound = (2.0 ** -21 + (in_dim + 2) * 2.0 ** -23) * (np.abs(x).astype(np.float64) @ np.abs(w16).T)
    worst = float(np.max(np.abs(got - want) / bound))
    rms = float(np.sqrt(np.mean(want * want)))
    block = float(block_rms(got - want).max()) / rms
    bar = block_bar(in_dim)
    n = min(s, 16)
    plane = x[:n].astype(np.float16).astype(np.float64) @ w16.T - want[:n]
    print(f"{s} x {out_dim} x {in_dim}: {worst:.2e} of the bound, blocks {block / bar:.2f} of theirs, "
          f"one plane {block_rms(plane).min() / rms / bar:.1f}")
    assert worst <= 1.0 and block <= bar
    assert block_rms(plane).min() / rms > bar


@pytest.mark.parametrize("kernel,seq,dim,vocab", [
    ("pipe32/1 in runs", 1100, 768, 512), ("ring64x128/1 in runs", 1030, 1056, 1024), ("ring128x128/1 in runs", 1030, 768, 2048),
    ("ring64x64/1 in runs", 2001, 768, 512), ("ring32x64/1 in runs", 190, 1632, 4096)])
def test_channel_first_product_in_runs(gpu, kernel, seq, dim, vocab):
    """The same sums in channel-first logits (MatMulVocabSeq), by blocks as above."""
    p = plan.plans([(seq, vocab, dim, 0)])[0]
    assert "%s/%d in runs" % (p.kind, p.ranges) == kernel and p.run
    rng = np.random.default_rng(seq + dim)
    e = (rng.standard_normal((vocab, dim), np.float32) * 0.05).astype(np.float32)
    x = rng.standard_normal((dim, seq), np.float32)
    got = sh.matmul_vocab_seq(e, x)
    want = e.astype(np.float16).astype(np.float64) @ x.astype(np.float64)
    block = float(block_rms(got - want).max()) / float(np.sqrt(np.mean(want * want)))
    print(f"{block / block_bar(dim):.2f} of the bar")
    assert block <= block_bar(dim)


@pytest.mark.parametrize("s,in_dim,out_dim", [(5, 256, 128), (40, 2048, 192), (700, 512, 1024)])
@pytest.mark.parametrize("off", [0, 4, 12])
def test_conv_eval_noalloc_unaligned_buffers(gpu, s, in_dim, out_dim, off):
    """Caller's buffers that are not 16-byte aligned give the same bits, and nothing around the
    output is written."""
    lib, hip = sh.load(), Hip()
    rng = np.random.default_rng(s + off)
    conv = sh.Conv((rng.standard_normal((out_dim, in_dim)) * 0.05).astype(np.float32))
    x = rng.standard_normal((s, in_dim), np.float32)
    want = conv.eval(x)
    n = s * out_dim
    dx, dy = hip.malloc(4 * s * in_dim + 64), hip.malloc(4 * n + 64)
    try:
        hip.h2d(dx.value + off, x)
        hip.h2d(dy, np.full(n + 16, 3.0, np.float32))
        assert lib.sh_conv_eval_noalloc(conv.h, dx.value + off, s, dy.value + off, None) == 0, sh.last_error()
        hip.sync()
        got = np.empty(n + 16, np.float32)
        hip.d2h(got, dy)
        at = off // 4
        np.testing.assert_array_equal(got[at:at + n].view(np.uint32), want.ravel().view(np.uint32))
        assert np.all(got[:at] == 3.0) and np.all(got[at + n:] == 3.0)
    finally:
        hip.free(dx)
        hip.free(dy)
        conv.close()


# the kernels of q|k|v, Wo (residual), W1|W3 (gate) and W2 (residual)
@pytest.mark.parametrize("make_cfg,dtype,seq,kernels", [
    (lambda: tiny_config(dim=768, hidden=2048, n_heads=12, n_kv_heads=12, head_dim=64, max_seq=1100), sh.SH_DTYPE_F16, 1091,
     "ring128x128 ring64x64 ring64x128 ring64x64"),
    (lambda: tiny_gqa_config(dim=256, hidden=768, n_heads=8, n_kv_heads=4, max_seq=700), sh.SH_DTYPE_BF16, 641,
     "pipe32 pipe32 pipe32 pipe32"),
    (lambda: tiny_gqa_config(dim=512, hidden=3072, n_heads=16, n_kv_heads=8, max_seq=1100), sh.SH_DTYPE_BF16, 1091,
     "ring64x128 pipe32 ring128x256 pipe32"),
])
def test_layer_forward_on_ring_tiles(gpu, make_cfg, dtype, seq, kernels):
    cfg = make_cfg()
    D, F, Q = cfg.dim, cfg.hidden, cfg.qdim
    products = [(seq, Q + 2 * cfg.kvdim, D, 0), (seq, D, Q, 0), (seq, 2 * F, D, 0), (seq, D, F, 0)]
    assert [p.kind for p in plan.plans(products)] == kernels.split()
    m, ocfg, ow = build(cfg, dtype, 71, std=0.03)
    x = embed_cf(ow, sh.synth_tokens(seq, 72, cfg.vocab))
    got = m.layer_forward_cf(0, x)
    want = oracle.layer_forward_cf(ocfg, ow, 0, x, threads=THREADS)
    m.close()
    err = rel_err(got, want)
    print(f"S={seq}: rel {err:.2e}")
    assert err <= 1e-4


@pytest.mark.parametrize("dtype,seq,vocab,kernel", [
    (sh.SH_DTYPE_F16, 47, 32000, "ring64x64"), (sh.SH_DTYPE_F16, 190, 32064, "ring64x64"),
    (sh.SH_DTYPE_F16, 188, 16384, "ring128x128"), (sh.SH_DTYPE_BF16, 189, 16384, "ring64x128")])
def test_eval_logits_on_ring_tiles(gpu, dtype, seq, vocab, kernel):
    """Channel-first logits of row counts that are and are not multiples of four; fp16 in one plane."""
    assert plan.plans([(seq, vocab, 256, dtype == sh.SH_DTYPE_F16)])[0].kind == kernel
    cfg = tiny_config(dim=256, hidden=512, n_heads=4, n_kv_heads=4, head_dim=64, vocab=vocab, max_seq=256)
    m, ocfg, ow = build(cfg, dtype, 81)
    toks = sh.synth_tokens(seq, 82, cfg.vocab)
    got = m.eval_logits(toks)
    want = oracle.eval_logits_cf(ocfg, ow, toks, threads=THREADS)
    m.close()
    err = float(np.max(np.abs(got - want)))
    print(f"S={seq} V={vocab}: max-abs {err:.2e}")
    assert err <= 2e-2


@pytest.mark.parametrize("dim,hidden,vocab,seq", [
    (64, 64, 512, 47), (128, 128, 512, 47), (64, 128, 512, 1100),   # every product
    (192, 64, 16384, 256), (64, 64, 16384, 300),                    # a large classifier
])
def test_eval_logits_of_short_k_keep_the_pair(gpu, dim, hidden, vocab, seq):
    """Products over 64, 128 or (large ones) 192 columns take the activations as a hi/lo pair also in
    EvalLogits' fp16 form: relative error (2-norm) below 1e-5, where one fp16 plane makes 1e-4 or more (an
    11-bit significand: 2^-12 / sqrt(3) of each activation). Wo is zero, so the attention, which takes one plane,
    has no part in it, and so is W2 where W1|W3 take one plane."""
    cfg = tiny_config(dim=dim, hidden=hidden, n_layers=2, n_heads=dim // 32, n_kv_heads=dim // 32, head_dim=32, vocab=vocab,
                      max_seq=seq)
    w = sh.synth_weights(cfg, seed=91 + dim, std=0.08)
    for lw in w.layers:
        lw["wo"] = np.zeros_like(lw["wo"])
        if dim == 192:
            lw["w2"] = np.zeros_like(lw["w2"])
    m = sh.Model(cfg, sh.SH_DTYPE_F16)
    m.upload(w)
    toks = sh.synth_tokens(seq, 92, cfg.vocab).astype(np.uint16)
    got = m.eval_logits(toks)
    m.close()
    want = oracle.eval_logits_cf(oracle.config_from(cfg), w.rounded(sh.SH_DTYPE_F16), toks, threads=THREADS)
    err = float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want.astype(np.float64)))
    print(f"rel {err:.2e}")
    assert err <= 1e-5
