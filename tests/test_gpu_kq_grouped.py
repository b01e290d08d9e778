"""The grouped products of K-quant experts (more pairs than experts) at the
edges of their tiles: bit for bit the oracle's moe_ffn, and the per-pair
products' (the forced GEMV path)."""
import numpy as np
import pytest

import hipmoe
import oracle
from common import SEED, bits

pytestmark = pytest.mark.gpu

Q4K, Q6K = hipmoe.Q4_K, hipmoe.Q6_K
# types, E, EI, NE, topk, renorm, token counts: one super-block a row; every
# token on every expert (tiles of 32, 32 + 1, 32 + 16 and 32 + 17 rows);
# ragged d_ff; tiles of a few rows each; the OLMoE shape
CASES = {
    "one_block": (Q4K | Q6K << 8, 256, 256, 4, 1, 0, (340,)),
    "all_experts": (Q6K, 768, 256, 3, 3, 1, (32, 33, 48, 49)),
    "ragged_dff": (Q6K | Q4K << 8, 512, 768, 8, 2, 1, (29, 70)),
    "q4k_down": (Q4K, 1024, 512, 16, 4, 0, (17, 130)),
    "olmoe": (Q4K | Q6K << 8, 2048, 1024, 64, 8, 0, (10,)),
}
REREAD = 40 << 20  # bytes the pairs past one per expert re-read where the path starts


@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_kq_grouped_tiles_vs_oracle(name):
    wt, E, EI, NE, K, renorm, Ts = CASES[name]
    lw = hipmoe.synth_layer(SEED, 11, wt, E, EI, NE, 0.02, None)
    gt, dt = hipmoe.wtypes(wt)
    expert = 2 * EI * hipmoe.row_bytes(gt, E) + E * hipmoe.row_bytes(dt, EI)
    M = hipmoe.MoeLayer.from_synth(lw, K, bool(renorm))
    try:
        for T in Ts:
            assert (T * K - NE) * expert >= REREAD
            x = hipmoe.synth_input(SEED, 0x9600 + T, T, E)
            x[T // 2] = 0.0  # an all-zero token: every Q8_K scale 0
            x[0, :256] *= 1e6
            M.set_path(hipmoe.PATH_AUTO)
            assert M.path_for(T) == hipmoe.PATH_GROUPED
            out, ids, w = M.ffn(x)
            assert M.path_for(T) == hipmoe.PATH_GROUPED
            M.set_path(hipmoe.PATH_GEMV)
            out_p, ids_p, w_p = M.ffn(x)
            oout, oids, ow, _, _ = oracle.moe_ffn(x, lw, K, bool(renorm), None)
            print(f"kq grouped {name} T={T}: {int(np.sum(bits(out) != bits(oout)))} of "
                  f"{out.size} outputs differ", flush=True)
            assert np.array_equal(ids, oids) and np.array_equal(bits(w), bits(ow))
            assert np.array_equal(bits(out), bits(oout))
            assert np.array_equal(bits(out), bits(out_p)) and np.array_equal(ids, ids_p)
    finally:
        M.free()


def test_gpu_kq_grouped_after_a_larger_reservation():
    """Scratch reserved past the grouped products' limit: the same bits as
    the oracle on both sides of it, from the one h buffer."""
    wt, E, EI, NE, K = Q4K | Q6K << 8, 256, 256, 16, 8
    lw = hipmoe.synth_layer(SEED, 12, wt, E, EI, NE, 0.02, None)
    M = hipmoe.MoeLayer.from_synth(lw, K, False)
    try:
        assert hipmoe.lib().hip_moe_reserve(M.h, 36000) == 1
        for T in (301, 3, 45):
            x = hipmoe.synth_input(SEED, 0x9620 + T, T, E)
            print(f"kq grouped after a reservation, T={T}", flush=True)
            out, ids, w = M.ffn(x)
            oout, oids, ow, _, _ = oracle.moe_ffn(x, lw, K, False, None)
            assert np.array_equal(ids, oids) and np.array_equal(bits(w), bits(ow))
            assert np.array_equal(bits(out), bits(oout))
    finally:
        M.free()


@pytest.mark.parametrize("wt", (Q4K | Q6K << 8, Q6K | Q4K << 8))
def test_gpu_kq_grouped_extreme_h_vs_oracle(wt):
    """Tokens whose h overflows, is subnormal, or makes subnormal products
    with the down weights: the matrix instructions' chains keep the bits of
    the oracle's FMAs, and have NaN and infinities where it has."""
    E, EI, NE, K, T = 512, 512, 4, 2, 120
    lw = hipmoe.synth_layer(SEED, 13, wt, E, EI, NE, 0.02, None)
    x = hipmoe.synth_input(SEED, 0x9630, T, E)
    scale = np.float32([1, 1e25, 1e-19, 1e-21, 1e-17, 2e19])
    x *= scale[np.arange(T) % scale.size][:, None]
    M = hipmoe.MoeLayer.from_synth(lw, K, False)
    try:
        assert M.path_for(T) == hipmoe.PATH_GROUPED
        out, _, _ = M.ffn(x)
        want, _, _, _, _ = oracle.moe_ffn(x, lw, K, False, None)
        small = np.abs(want[want != 0])
        print(f"kq grouped extremes {wt:#x}: {np.isnan(want).sum()} NaN, {np.isinf(want).sum()} "
              f"infinite, {(small < 2.0**-126).sum()} subnormal of {want.size}", flush=True)
        assert np.isnan(want).any() and (small < 2.0**-126).any()
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(out), nan)
        assert np.array_equal(bits(out)[~nan], bits(want)[~nan])
    finally:
        M.free()
