"""Host-pointer calls on both sides of the limits of their pinned staging:
the same bits as the device entry points and as the larger form."""
import numpy as np
import pytest

import hiplm
import hipmoe
from common import SEED, bits, model_case, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt", (hipmoe.Q8_0, hipmoe.Q4_K | hipmoe.Q6_K << 8))
def test_gpu_host_ffn_equals_device_entry(wt):
    E, EI, NE, K = 2048, 1024, 64, 8  # 16 tokens are 128 KB
    lw = hipmoe.synth_layer(SEED, 51, wt, E, EI, NE, 0.02, 0.5)
    M = hipmoe.MoeLayer.from_synth(lw, K, True)
    H = hipmoe.hip()
    bias = hipmoe.synth_normal(SEED, 52, NE)
    d_b = H.upload(bias)
    bufs = [d_b]
    try:
        for T in (1, 16, 17, 2):
            for b in (None, bias):
                print(f"host ffn wt={wt} T={T} bias={b is not None}", flush=True)
                x = hipmoe.synth_input(SEED, 0x9900 + T, T, E)
                out, ids, w = M.ffn(x, b)
                d = [H.upload(x), H.malloc(out.nbytes), H.malloc(ids.nbytes), H.malloc(w.nbytes)]
                bufs += d
                M.ffn_dev(d[0], d[1], T, None if b is None else d_b, d[2], d[3])
                H.sync()
                assert np.array_equal(bits(out), bits(H.download(d[1], out.shape, np.float32)))
                assert np.array_equal(ids, H.download(d[2], ids.shape, np.uint32))
                assert np.array_equal(bits(w), bits(H.download(d[3], w.shape, np.float32)))
    finally:
        for b in bufs:
            H.free(b)
        M.free()


def test_gpu_batch_of_more_sequences_than_one_launch_sets():
    """128 ids fit the launch that sets a step, 130 are copied."""
    md, _, case, _ = model_case("mixtral_small")
    M = hiplm.LmModel(md, case[7])
    try:
        ids = np.random.default_rng(SEED).integers(0, md["V"], (130, 3)).astype(np.int32)
        got = {}
        for S in (128, 130):
            B = hiplm.LmBatch(M, S)
            got[S] = [B.decode(ids[:S, i]) for i in range(3)]
            B.free()
        for (n0, l0), (n1, l1) in zip(got[128], got[130]):
            assert np.array_equal(n0, l0.argmax(1)) and np.array_equal(n1, l1.argmax(1))
            err = rel_l2(l1[:128], l0)
            print(f"batch of 130 against 128: {err:.2e}", flush=True)
            # the same products row by row; their sums may be split otherwise
            assert err <= 1e-5
    finally:
        M.free()


def test_gpu_batch_of_more_logits_than_are_pinned():
    """17 MB of logits a step are copied, 2 MB go through pinned memory:
    the same rows, and each row's pick."""
    md = hiplm.synth_olmoe(SEED, 1, 512, 4, 34000, 8, 2, 256, hipmoe.Q8_0, 0.1)
    M = hiplm.LmModel(md, 32)
    try:
        ids = np.random.default_rng(SEED).integers(0, md["V"], (128, 2)).astype(np.int32)
        got = {}
        for S in (16, 128):
            B = hiplm.LmBatch(M, S)
            got[S] = [B.decode(ids[:S, i]) for i in range(2)]
            B.free()
        for (n0, l0), (n1, l1) in zip(got[16], got[128]):
            assert np.array_equal(n0, l0.argmax(1)) and np.array_equal(n1, l1.argmax(1))
            err = rel_l2(l1[:16], l0)
            print(f"batch of 128 against 16: {err:.2e}", flush=True)
            assert err <= 1e-5  # the same products; their sums may be split otherwise
    finally:
        M.free()
