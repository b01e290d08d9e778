"""The Q8_0/Q4_0 product of many tokens in tiles (32 tokens x 128 rows or 64 x
256, stages of 128 columns) at the edges of its tiles, against float64."""
import numpy as np
import pytest

import hipmoe
import oracle
from common import SEED

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
