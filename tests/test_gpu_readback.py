"""Results on their way from the decoder to ordinary host memory (past 2 MiB
through pinned slots of 2 MiB, at most four of them) against the same results
copied straight into pinned memory: the same bytes. Logits below one slot, of
exactly one and of a few bytes more, and past the four (so that slots are used
again); a token ring past one slot."""
import ctypes as C

import numpy as np
import pytest

from hako_amd import mlf2
from hako_amd.decoder import Decoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,vocab,max_seq", [(1, 1000, 16384), (1, 150001, 64), (2, 262144, 64), (2, 262145, 64),
                                                 (4, 150001, 64), (16, 150001, 64), (16, 1000, 40000)])
def test_logits_and_tokens_reach_ordinary_memory(gpu, tmp_path, n_seq, vocab, max_seq):
    with open("/proc/self/maps") as f:   # the HIP runtime that the library runs on
        hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    pin = C.c_void_p()
    path = str(tmp_path / "m.mlf2")
    mlf2.write_qwen2(path, mlf2.Qwen2Config(n_layers=1, d_model=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn_dim=512,
                                            vocab=vocab), 3)
    dec = Decoder(gpu, path, n_seq, max_seq)
    try:
        start = np.arange(n_seq, dtype=np.int32)
        dec.set_pos(0)
        nxt, lg = dec.step(start, logits=True)
        dec.set_pos(0)
        assert hip.hipHostMalloc(C.byref(pin), C.c_size_t(4 * n_seq * vocab), 0) == 0
        pinned = np.ctypeslib.as_array(C.cast(pin, C.POINTER(C.c_float)), (n_seq, vocab))
        again = np.empty(n_seq, np.int32)
        gpu.check(gpu.lib.hako_gpu_decoder_step(dec.d, start.ctypes.data, pin, again.ctypes.data), "step")
        assert np.array_equal(lg.view(np.uint32), pinned.view(np.uint32))
        assert np.array_equal(nxt, again) and np.array_equal(nxt, lg.argmax(1))
        # the ring: generated tokens as single steps make them
        dec.set_pos(0)
        toks = dec.generate(start, 5)
        dec.set_pos(0)
        t = start
        for i in range(5):
            t = dec.step(t)
            assert np.array_equal(toks[i], t)
        # a prompt's last logits and their first largest
        dec.set_pos(0)
        first, plg = dec.prefill(np.arange(20), logits=True)
        assert first == int(plg.argmax())
    finally:
        dec.close()
        if pin:
            hip.hipHostFree(pin)
