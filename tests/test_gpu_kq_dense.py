"""The K-quant dense product of several tokens on the matrix cores at the
edges of its tiles (32 tokens, 128 rows, 256 columns): bit for bit the
oracle's product."""
import numpy as np
import pytest

import hipmoe
import oracle
from common import SEED, bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt", (hipmoe.Q4_K, hipmoe.Q6_K))
@pytest.mark.parametrize("N,K,Ts", ((1, 256, (8, 10, 33)), (16384, 256, (6, 7)), (129, 768, (31, 32, 65)),
                                    (300, 2048, (11, 96)), (64, 14336, (17,))))
def test_gpu_kq_dense_vs_oracle(wt, N, K, Ts):
    q = hipmoe.synth_quant_matrix(SEED, 31, 0.02, wt, N, K)
    W = hipmoe.QMat(q, wt, N, K)
    try:
        for T in Ts:
            x = hipmoe.synth_normal(SEED, 0x9700 + T, T * K).reshape(T, K).copy()
            x[0] = 0.0                # every Q8_K scale 0
            x[1, :256] *= 1e-42       # a block scale that overflows: d = 0
            x[2, [200, 40]] = 9, -9   # equal magnitudes: the first one's sign
            x[3, [40, 200]] = 9, -9
            x[4, 255] = -1e20
            for add in (None, hipmoe.synth_normal(SEED, 5, N),
                        hipmoe.synth_normal(SEED, 6, T * N)):
                print(f"kq dense wt={wt} N={N} K={K} T={T}", flush=True)
                got, want = W.mul(x, add), oracle.qmat_mul(x, q, wt, N, K, add)
                assert np.array_equal(bits(got), bits(want))
    finally:
        W.free()
