"""Large results copied to host arrays (HostCopier) bit for bit: sizes around its threshold
(2 MiB), of an uneven last chunk and beyond its pinned ring (8 MiB), at unaligned host
addresses, through a trainer's embedding [V, D] read back."""
import ctypes as C

import numpy as np
import pytest

import stories_hip as sh
from helpers import tiny_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [2048, 8188, 8192, 8196, 9004, 32772, 65532])   # rows of 256 bytes
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
