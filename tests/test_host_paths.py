"""The host side of libhip_moe.so (dispatch, scratch, allocations that fail)
on the CPU: the built library over tests/native/fake_hip.c, which logs kernel
launches instead of running them.  Each case is a process of its own, since
the fake runtime has to be loaded before the library."""
import os
import subprocess
import sys
import textwrap

import pytest

from common import HERE, REPO

PRELUDE = f"""
import ctypes as C, sys
F = C.CDLL({os.path.join(HERE, "native", "libfake_hip.so")!r}, mode=C.RTLD_GLOBAL)
sys.path[:0] = [{os.path.join(REPO, "llm.c_amd")!r}]
import numpy as np
import hiplm, hipmoe
for f in (F.fake_log, F.fake_sizes):
    f.restype = C.c_char_p
for f in (F.fake_fail_size, F.fake_fail_host):
    f.argtypes = [C.c_size_t]
F.fake_host_allocs.restype = C.c_size_t
KQ = hipmoe.Q4_K | hipmoe.Q6_K << 8

def layer(wt, E, EI, NE, K):
    # byte 0 everywhere: valid blocks of any type
    gt, dt = hipmoe.wtypes(wt)
    gate = np.zeros((NE, EI * hipmoe.row_bytes(gt, E)), np.uint8)
    down = np.zeros((NE, E * hipmoe.row_bytes(dt, EI)), np.uint8)
    return hipmoe.MoeLayer(np.zeros((NE, E), np.float32), gate, gate, down, wt, E, EI, NE, K, 0)

def kernels(call):
    F.fake_log()
    call()
    return F.fake_log().decode()

def dev_call(L, T):
    # the pointers are handed on, never read
    return kernels(lambda: L.ffn_dev(4096, 4096, T))
"""


def on_fake(body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body)], cwd=REPO,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("reserve", (2000, 65535))
def test_kq_grouped_whatever_was_reserved(reserve):
    """The grouped K-quant products take a 301-token call on a layer whose
    scratch was grown past the largest call they hold (about 34,800 tokens
    here)."""
    on_fake(f"""
    L = layer(KQ, 256, 256, 16, 8)
    hipmoe.lib().hip_moe_reserve(L.h, {reserve})
    assert "k_kq_mm" in dev_call(L, 301)
    assert "k_kq_mm" in dev_call(L, 34000)
    assert "k_kq_mm" not in dev_call(L, 36000)
    assert "k_kq_mm" in dev_call(L, 300)
    """)


def test_kq_grouped_shares_the_per_pair_scratch():
    """One h buffer serves the per-pair and the grouped products."""
    on_fake("""
    L = layer(KQ, 256, 1024, 16, 8)
    F.fake_sizes()
    hipmoe.lib().hip_moe_reserve(L.h, 2000)
    h = 2000 * 8 * 1024 * 4
    big = [int(n) for n in F.fake_sizes().split() if int(n) >= h]
    assert len(big) == 1 and big[0] < 1.05 * h, big
    """)


@pytest.mark.parametrize("which", ("h", "rows", "tiles", "records"))
def test_kq_call_survives_a_failed_grouped_allocation(which):
    """Without memory for the grouped products a call takes the per-pair
    ones, as it did before there were others; with it again, later growth
    brings them back."""
    on_fake(f"""
    L = layer(KQ, 256, 256, 16, 8)
    T, K = 301, 8
    tiles = (T * K + 31) // 32 + 16
    F.fake_fail_size(dict(h=tiles * 32 * 256 * 4, rows=tiles * 32 * 4, tiles=(tiles + 1) * 4,
                          records=T * 548)[{which!r}])
    for _ in range(2):
        got = dev_call(L, T)
        assert "k_kq_mm" not in got and "k_kq_down" in got, got
    F.fake_fail_size(0)
    assert "k_kq_mm" in dev_call(L, 2 * T) and "k_kq_mm" in dev_call(L, T)
    """)


@pytest.mark.parametrize("wt,E,EI,NE,K", (("KQ", 2048, 1024, 64, 8), ("KQ", 4096, 14336, 8, 2),
                                          ("hipmoe.Q6_K", 1024, 512, 8, 2),
                                          ("hipmoe.Q4_0", 2048, 1024, 64, 8)))
def test_path_for_names_the_kernels_of_the_call(wt, E, EI, NE, K):
    """hip_moe_path_for, asked before and after the scratch holds the call,
    against the kernels the call launches, forced and not."""
    on_fake(f"""
    L = layer({wt}, {E}, {EI}, {NE}, {K})
    of = dict(k_moe_decode=1, k_kq_route_gateup=1, k_gateup=2, k_kq_gateup=2, k_pf_gateup=3,
              k_pf_gateup_v=3, k_kq_mm=3)
    # mangled: the name behind its length
    names = {{f"{{len(n)}}{{n}}": p for n, p in of.items()}}
    seen = set()
    for path in (0, 2):
        L.set_path(path)
        for T in (1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 16, 33, 64, 301, 7, 1):
            said = L.path_for(T)
            got = dev_call(L, T)
            took = {{p for n, p in names.items() if n in got}}
            assert took == {{said}} == {{L.path_for(T)}}, (path, T, said, took, got)
            seen.add(said)
    assert seen == {{1, 2, 3}}, seen
    L.set_path(3)  # K-quants: AUTO alone takes the grouped products
    assert L.path_for(301) == (0 if L.wtype != hipmoe.Q4_0 else 3)
    """)


def test_first_host_call_locks_no_memory():
    """The pinned staging of hip_moe_ffn is made with the layer."""
    on_fake("""
    L = layer(hipmoe.Q8_0, 2048, 1024, 8, 2)
    n = F.fake_host_allocs()
    got = kernels(lambda: L.ffn(np.zeros((1, 2048), np.float32)))
    assert "k_copy_segs" in got and F.fake_host_allocs() == n, (got, n)
    """)


def test_host_call_without_page_locked_memory():
    """A layer that got none takes the copies, every call of it."""
    on_fake("""
    F.fake_fail_host(1)
    L = layer(hipmoe.Q8_0, 2048, 1024, 8, 2)
    for _ in range(2):
        got = kernels(lambda: L.ffn(np.zeros((1, 2048), np.float32)))
        assert "k_copy_segs" not in got and "k_moe_decode" in got, got
    """)


TINY = "hiplm.synth_olmoe(1, 1, 256, 2, 256, 4, 2, 256, hipmoe.Q8_0)"


def test_model_and_batch_without_page_locked_memory():
    """Upload and every host call of a model work from plain host memory."""
    on_fake(f"""
    md = {TINY}
    F.fake_fail_host(1)
    M = hiplm.LmModel(md, 64)
    ids = np.arange(5, dtype=np.int32)
    M.prefill(ids)
    M.decode(3)
    M.reset()
    assert len(M.generate(ids, 3)[0]) == 4
    B = hiplm.LmBatch(M, 3)
    B.decode(ids[:3])
    B.reset()
    B.generate(np.tile(ids, (3, 1)), 2)
    B.free()
    M.free()
    """)


@pytest.mark.parametrize("heads,ok", ((4, True), (6, False)))
def test_model_refuses_head_rows_no_kernel_covers(heads, ok):
    """The one-token products cover rows of 64 columns times a power of two
    up to 64; heads * 128 = 768 would leave two thirds of a row out."""
    on_fake(f"""
    md = hiplm.synth_mixtral(1, 1, 512, {heads}, 2, 256, 4, 2, 256, hipmoe.Q4_0)
    try:
        hiplm.LmModel(md, 64)
        ok = True
    except hipmoe.HipMoeError as e:
        assert "not supported" in str(e)
        ok = False
    assert ok == {ok}
    """)


@pytest.mark.parametrize("N,K", ((300, 256), (2048, 2048), (6144, 2048), (4096, 4096), (32000, 4096)))
def test_split_buffer_holds_what_the_few_token_form_writes(N, K):
    """A matrix's partial sums: enough for every token count that takes the
    form with partial sums, none where no count does; one token has its own
    kernel, larger counts the tiles."""
    on_fake(f"""
    N, K, top = {N}, {K}, 64
    lib = hipmoe.lib()
    for f in (lib.moe_qmm_work_bytes, lib.moe_qmm_work_most):
        f.restype = C.c_size_t
    few = [t > 0 and not lib.moe_qmm_tile_better(N, t) for t in range(2001)]
    for T in (2, 16, 40, 64, 333, 2000):
        need = max(lib.moe_qmm_work_bytes(t, N, K) if few[t] else 0 for t in range(T + 1))
        assert lib.moe_qmm_work_most(T, N, K) == need, T
    F.fake_sizes()
    W = hipmoe.QMat(np.zeros(N * hipmoe.row_bytes(hipmoe.Q4_0, K), np.uint8), hipmoe.Q4_0, N, K)
    sizes = [int(n) for n in F.fake_sizes().split()]
    weights = max(sizes)
    split = [n for n in sizes if n != weights]
    assert sum(split) == lib.moe_qmm_work_most(top, N, K), sizes
    for T in (1, 2, 16, 17, 64, 65, 301):
        got = kernels(lambda: W.mul_dev(4096, T, 4096))
        want = "k_qgemv1" if T == 1 else "5k_qmmI" if few[T] and T <= top else "k_qmm_tile"
        assert [n for n in ("k_qgemv", "5k_qmmI", "k_qmm_tile") if n in got] == \
            [want.removesuffix("1")], (T, got)
    """)
