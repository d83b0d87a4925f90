"""Large results copied to host arrays (HostCopier) bit for bit: sizes around its threshold
(512 KiB), of an uneven last chunk and beyond its pinned ring (8 MiB), at unaligned host
addresses, through a trainer's embedding [V, D] read back. The ring and its threads come with the
copies that need them, not with a model, are one for all models, and go with the last that used
them; models on two threads return what each returns alone."""
import ctypes as C
import os
import threading

import numpy as np
import pytest

import stories_hip as sh
from helpers import tiny_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1024, 2044, 2048, 2052, 8188, 9004, 32772, 65532])   # rows of 256 bytes
def test_read_round_trip(gpu, vocab):
    cfg = tiny_config(dim=64, hidden=128, n_layers=1, n_heads=4, n_kv_heads=4, head_dim=16, vocab=vocab, max_seq=32)
    tr = sh.Trainer(cfg, seq=16)
    n = vocab * cfg.dim
    F = C.POINTER(C.c_float)
    rms = np.ones(cfg.dim, np.float32)
    for off in (0, 4, 20):
        src = np.random.default_rng(vocab + off).standard_normal(n + 16, np.float32)
        dst = np.full(n + 16, 7.0, np.float32)
        at = off // 4
        assert sh.load().sh_trainer_upload_globals(tr.h, src[at:].ctypes.data_as(F), rms.ctypes.data_as(F)) == 0
        assert sh.load().sh_trainer_read(tr.h, sh.SH_TRAIN_PARAMS, b"embed", dst[at:].ctypes.data_as(F), n) == 0
        np.testing.assert_array_equal(dst[at:at + n].view(np.uint32), src[at:at + n].view(np.uint32))
        assert np.all(dst[:at] == 7.0) and np.all(dst[at + n:] == 7.0)
    tr.close()


def wide_model():
    cfg = tiny_config(dim=1024, hidden=1024, n_layers=1, n_heads=16, n_kv_heads=16, head_dim=64, vocab=8192, max_seq=128)
    m = sh.Model(cfg, sh.SH_DTYPE_F16)
    m.upload(sh.synth_weights(cfg, seed=3, std=0.02))
    return m, sh.synth_tokens(128, 4, cfg.vocab)


def test_threads_come_with_large_copies(gpu):
    def threads():
        return len(os.listdir("/proc/self/task"))

    m, toks = wide_model()
    for _ in range(9):
        m.eval_logits(toks)           # 4 MiB of logits each: the ring's set-up is behind
    m.close()
    before = threads()
    a, _ = wide_model()
    a.greedy_decode(toks[:9], 4)
    a.eval_logits(toks[:15])          # 480 KiB
    assert threads() == before
    b, _ = wide_model()
    for m in (a, b):
        m.eval_logits(toks)
    assert before <= threads() <= before + 5
    a.close()
    b.close()
    assert threads() == before


def test_two_models_on_two_threads(gpu):
    """Whichever copy finds the ring taken goes the runtime's way."""
    models = [wide_model() for _ in range(2)]
    want = [m.eval_logits(t[:128 - 9 * i]) for i, (m, t) in enumerate(models)]
    wrong = []

    def run(i):
        m, t = models[i]
        for _ in range(40):
            if not np.array_equal(m.eval_logits(t[:128 - 9 * i]), want[i]):
                wrong.append(i)

    both = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in both:
        t.start()
    for t in both:
        t.join()
    for m, _ in models:
        m.close()
    assert not wrong
