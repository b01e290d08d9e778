"""The Q8_0/Q4_0 product of many tokens in tiles (32 tokens x 128 rows or 64 x
256, stages of 128 columns) at the edges of its tiles, against float64."""
import numpy as np
import pytest

import hipmoe
import oracle
from common import SEED, rel_l2

pytestmark = pytest.mark.gpu


# rows x columns, token counts: one row, row blocks of 128 and 256 and their
# remainders; the fewest columns; many rows at two tokens; a chip-filling grid
@pytest.mark.parametrize("wt", (hipmoe.Q8_0, hipmoe.Q4_0))
@pytest.mark.parametrize("N,K,Ts", ((1, 256, (65,)), (129, 512, (128, 129)), (257, 4096, (191,)),
                                    (20000, 256, (2, 33, 130)), (2100, 1024, (1025,))))
def test_gpu_qmm_tile_vs_float64(wt, N, K, Ts):
    q = hipmoe.synth_quant_matrix(SEED, 41, 0.02, wt, N, K)
    w = oracle.dequant(np.frombuffer(q, np.uint8), wt, N * K).reshape(N, K).astype(np.float64)
    W = hipmoe.QMat(q, wt, N, K)
    H = hipmoe.hip()
    bufs = []
    try:
        for T in Ts:
            x = hipmoe.synth_normal(SEED, 0x9800 + T, T * K).reshape(T, K).copy()
            x[0] = 0.0
            x[1, :100] *= 1e5    # one 128-column stage with a wide range
            if T > 4:
                x[2] *= 1e30
                x[3] *= 1e-41    # subnormal
                x[4, 7] = np.inf  # no finite output, and no other token's
            for add in (None, hipmoe.synth_normal(SEED, 5, N),
                        hipmoe.synth_normal(SEED, 6, T * N)):
                print(f"qmm tile wt={wt} N={N} K={K} T={T}", flush=True)
                d = [H.upload(x), H.malloc(T * N * 4)] + ([] if add is None else [H.upload(add)])
                bufs += d
                W.mul_dev(d[0], T, d[1], None if add is None else d[2],
                          0 if add is None else add.size)
                H.sync()
                got = H.download(d[1], (T, N), np.float32)
                a = 0.0 if add is None else add.astype(np.float64).reshape(-1, N)
                xd = x.astype(np.float64)
                if T > 4:
                    assert not np.isfinite(got[4]).any()
                    xd[4] = 0.0
                want = xd @ w.T + a
                # roundings: 32 in a block's sum, one a block scale, 4 + K / 128 in
                # the chains, 2 of the end; the split keeps 2^-23 of a value and
                # 2^-38 of its stage's largest; results below 2^-126 round as they are
                top = np.abs(xd).reshape(T, -1, 128).max(-1).repeat(128, -1)
                tol = (2.0**-24 * (39 + K / 128) + 2.0**-23) * (np.abs(xd) @ np.abs(w).T) + \
                    2.0**-38 * (top @ np.abs(w).T) + 2.0**-23 * np.abs(want) + K * 2.0**-149
                ok = np.abs(got - want) <= tol
                if T > 4:
                    ok[4] = True
                assert ok.all(), np.argwhere(~ok)[:4]
    finally:
        for b in bufs:
            H.free(b)
        W.free()


@pytest.mark.parametrize("wt", (hipmoe.Q8_0, hipmoe.Q4_0))
@pytest.mark.parametrize("N,K,T", ((300, 512, 70), (2100, 256, 1025)))  # 32 x 128 and 64 x 256 tiles
def test_gpu_qmm_tile_blocks_of_unequal_range_vs_float64(wt, N, K, T):
    """A block whose weights are zero and whose values are 2^24 times its
    neighbours': it adds nothing, and the neighbours keep their 22 bits (a
    scale shared by more than one block would leave them about 14)."""
    q = np.frombuffer(hipmoe.synth_quant_matrix(SEED, 42, 0.02, wt, N, K), np.uint8).copy()
    q.reshape(N, K // 32, -1)[:, 1::4, :2] = 0  # the blocks' f16 scales
    w = oracle.dequant(q, wt, N * K).reshape(N, K).astype(np.float64)
    x = hipmoe.synth_normal(SEED, 0x9810, T * K).reshape(T, K).copy()
    x.reshape(T, K // 32, 32)[:, 1::4] *= 2.0**24
    W = hipmoe.QMat(q, wt, N, K)
    H = hipmoe.hip()
    bufs = [H.upload(x), H.malloc(T * N * 4)]
    try:
        print(f"qmm tile, unequal blocks wt={wt} N={N} K={K} T={T}", flush=True)
        W.mul_dev(bufs[0], T, bufs[1])
        H.sync()
        got = H.download(bufs[1], (T, N), np.float32)
    finally:
        for b in bufs:
            H.free(b)
        W.free()
    xd = x.astype(np.float64)
    # 32 roundings in a block's sum, 4 + K / 128 in the chains; the split keeps
    # 2^-23 of a value and 2^-38 of its block's largest
    top = np.abs(xd).reshape(T, -1, 32).max(-1).repeat(32, -1)
    tol = (2.0**-24 * (36 + K / 128) + 2.0**-23) * (np.abs(xd) @ np.abs(w).T) + \
        2.0**-38 * (top @ np.abs(w).T)
    err = np.abs(got - xd @ w.T)
    print(f"  largest error {np.max(err / tol):.3g} of its bound", flush=True)
    assert (err <= tol).all()


@pytest.mark.parametrize("wt", (hipmoe.Q8_0, hipmoe.Q4_0))
@pytest.mark.parametrize("T", (128, 1024))  # 32 x 128 and 64 x 256 tiles
def test_gpu_qmm_tile_no_further_off_than_few_tokens(wt, T):
    """Sixteen tokens in tiles, among many, are no further from float64 than
    the same sixteen by themselves, which the few-token form takes (65536
    outputs estimate such an error to 0.3 per cent)."""
    N = K = 4096
    q = hipmoe.synth_quant_matrix(SEED, 43, 0.02, wt, N, K)
    w = oracle.dequant(np.frombuffer(q, np.uint8), wt, N * K).reshape(N, K).astype(np.float64)
    x = hipmoe.synth_normal(SEED, 0x9811, T * K).reshape(T, K)
    want = x[:16].astype(np.float64) @ w.T
    W = hipmoe.QMat(q, wt, N, K)
    H = hipmoe.hip()
    bufs = [H.upload(x), H.malloc(T * N * 4)]
    err = []
    try:
        for n in (16, T):
            W.mul_dev(bufs[0], n, bufs[1])
            H.sync()
            err.append(rel_l2(H.download(bufs[1], (16, N), np.float32), want))
    finally:
        for b in bufs:
            H.free(b)
        W.free()
    print(f"qmm tile wt={wt} T={T}: {err[1]:.3e}, few tokens {err[0]:.3e}", flush=True)
    assert err[1] <= 1.01 * err[0]
