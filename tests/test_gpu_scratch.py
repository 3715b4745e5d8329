"""What the library's scratch does when memory is short: calls that can do without a buffer do without it, nothing that
was there is given up for a buffer that does not come, and only what a recorded chain holds is kept beside a larger one."""
import ctypes

import numpy as np
import pytest

from conftest import peak_err

pytestmark = pytest.mark.gpu
Q6_K = 14
K = 2048


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _device(pkg, monkeypatch, limit=0):
    monkeypatch.setenv("OJAS_HIP_GEMM_SR", "1")              # K whole: results do not depend on arrival
    monkeypatch.setenv("OJAS_HIP_SCRATCH_MAX", str(limit))
    return pkg.HipGpu(0)


def _weights(pkg, n):
    return np.tile(pkg.synth.q6k_weights(256, K, "scratch", "w"), n // 256)


def _want(pkg, orc, x):
    return orc.matmul_ref(pkg.synth.q6k_weights(256, K, "scratch", "w"), Q6_K, 256, K, x, wmode=1, xmode=1)


def _check(g, yd, n, m, toks, want):
    got = g.read(yd, m * n).reshape(m, n)[toks]
    # f16 operands: exact products, K of them added in f32 — about sqrt(K) 2^-24 of sum |products|, itself some
    # 0.15 sqrt(K) peaks for such inputs: 1.8e-5; K 2^-24 = 1.2e-4 leaves a factor of six
    assert peak_err(got, np.tile(want, (1, n // 256))) <= K * 2.0 ** -24


def test_a_batch_without_room_for_the_decoded_rows_keeps_its_loader(pkg, orc, monkeypatch):
    """Q6_K rows are decoded into scratch from 129 tokens on.  The activations' scratch, which every form of the call needs,
    fits the limit and the decoded rows fit it too, but not both: the call runs on the tile that decodes into LDS."""
    n, m = 8192, 700
    xh, wdeq = m * K * 2, n * K * 2
    g = _device(pkg, monkeypatch, wdeq + xh // 2)
    try:
        x = pkg.synth.normal_f32(m * K, "scratch", "x", m).reshape(m, K)
        toks = np.r_[0:4, m - 4:m]
        yd = g.alloc(m * n)
        g.mm(g.upload(x), g.lin(Q6_K, n, K, _weights(pkg, n)), yd, m, act_mode=pkg.ACT_FLOAT)
        _check(g, yd, n, m, toks, _want(pkg, orc, x[toks]))
    finally:
        g.close()


def test_a_refused_growth_leaves_the_smaller_buffer(pkg, orc, monkeypatch):
    """Two layer sizes by turns beside a recorded chain, the larger beyond the limit: every call succeeds, and neither gives
    the smaller matrix's buffer up (or strands one per turn)."""
    small, large, m = 8192, 65536, 300
    g = _device(pkg, monkeypatch, 160 << 20)
    try:
        x = pkg.synth.normal_f32(m * K, "scratch", "x", m).reshape(m, K)
        want = _want(pkg, orc, x[:8])
        xd, yd = g.upload(x), g.alloc(m * large)
        lins = {n: g.lin(Q6_K, n, K, _weights(pkg, n)) for n in (small, large)}
        g.mm(xd, lins[large], yd, m, act_mode=pkg.ACT_FLOAT)
        g.mm(xd, lins[small], yd, m, act_mode=pkg.ACT_FLOAT)
        g.capture_begin()
        g.mm(xd, lins[small], yd, m, act_mode=pkg.ACT_FLOAT)
        graph = g.capture_end()
        g.submit()
        free = _free_bytes()
        for _ in range(3):
            for n in (large, small):
                g.mm(xd, lins[n], yd, m, act_mode=pkg.ACT_FLOAT)
                _check(g, yd, n, m, slice(0, 8), want)
                assert _free_bytes() == free, n
            g.memset0(yd)
            graph.launch()
            _check(g, yd, small, m, slice(0, 8), want)
        graph.free()
    finally:
        g.close()


def test_a_failed_allocation_leaves_no_error_behind(gpu, pkg):
    """... for whoever asks the runtime next: the failure is the return code's, and a call that goes on without the buffer
    has succeeded."""
    with pytest.raises(pkg.OjasHipError, match="hipMalloc"):
        gpu.alloc_bytes(1 << 50)
    assert ctypes.CDLL("libamdhip64.so").hipGetLastError() == 0


def test_an_outgrown_buffer_no_chain_holds_is_given_back(pkg, orc, monkeypatch):
    """A recorded chain that never touched the decoded rows' scratch (a decode step) does not keep what eager prefill outgrows."""
    m, sizes = 300, (16384, 32768, 65536)
    g = _device(pkg, monkeypatch)
    try:
        x = pkg.synth.normal_f32(m * K, "scratch", "x", m).reshape(m, K)
        want = _want(pkg, orc, x[:8])
        xd, yd = g.upload(x), g.alloc(m * sizes[-1])
        lins = [g.lin(Q6_K, n, K, _weights(pkg, n)) for n in sizes]
        one = g.lin(Q6_K, 256, K, _weights(pkg, 256))
        g.mm(xd, one, yd, m, act_mode=pkg.ACT_FLOAT)                       # code objects loaded, the activations' scratch sized
        g.mm(xd, one, yd, 1, act_mode=pkg.ACT_Q8K)
        g.capture_begin()
        g.mm(xd, one, yd, 1, act_mode=pkg.ACT_Q8K)
        graph = g.capture_end()
        g.submit()
        free = _free_bytes()
        for n, lin in zip(sizes, lins):
            g.mm(xd, lin, yd, m, act_mode=pkg.ACT_FLOAT)
            _check(g, yd, n, m, slice(0, 8), want)
        assert free - _free_bytes() <= sizes[-1] * K * 2 + (16 << 20)      # the largest alone, not the 67 and 134 MB before it
        graph.free()
    finally:
        g.close()


def test_a_chain_keeps_the_decoded_rows_it_was_recorded_with(pkg, orc, monkeypatch):
    """... while one that did replays into its own buffer after eager calls have outgrown it."""
    m, small, large = 130, 512, 16384
    g = _device(pkg, monkeypatch)
    try:
        x = pkg.synth.normal_f32(m * K, "scratch", "x", m).reshape(m, K)
        want = _want(pkg, orc, x[:8])
        xd, yd, yl = g.upload(x), g.alloc(m * small), g.alloc(m * large)
        lins = {n: g.lin(Q6_K, n, K, _weights(pkg, n)) for n in (small, large)}
        g.mm(xd, lins[small], yd, m, act_mode=pkg.ACT_FLOAT)
        eager = g.read(yd, m * small)
        g.capture_begin()
        g.mm(xd, lins[small], yd, m, act_mode=pkg.ACT_FLOAT)
        graph = g.capture_end()
        for _ in range(3):
            g.mm(xd, lins[large], yl, m, act_mode=pkg.ACT_FLOAT)
            g.memset0(yd)
            graph.launch()
            assert np.array_equal(g.read(yd, m * small), eager)
            _check(g, yl, large, m, slice(0, 8), want)
        graph.free()
    finally:
        g.close()


@pytest.mark.parametrize("room", [-4096, 4096])
def test_a_batch_that_cannot_have_all_its_scratch_takes_none(pkg, orc, monkeypatch, room):
    """24 tokens of Q4_K rows run on the 64-row int8 tile where its four scratch buffers are to be had.  Where the limit holds the
    small ones, or the largest, but not all, the call stays with the few-token kernel, and none of them is left to take room from other calls."""
    m, n = 24, 2112
    w = pkg.synth.q4k_weights(n, 4096, "scratch", "w24")
    x = pkg.synth.normal_f32(m * 4096, "scratch", "x24").reshape(m, 4096)
    part = 33 * 4 * 32768                                    # 33 64-row tiles over four slices of K
    g = _device(pkg, monkeypatch, part + room)
    try:
        lin, xd, yd = g.lin(12, n, 4096, w), g.upload(x), g.alloc(m * n)
        xq, xs = g.alloc_bytes(m * 4096), g.alloc(m * 16)
        g.quant_q8k(xd, m, 4096, xq, xs)
        g.ensure_family("gemm_q8k")
        other = g.lin(Q6_K, 256, K, _weights(pkg, 256))
        xo, yo = g.upload(np.zeros(4096 * K, np.float32)), g.alloc(4096 * 256)
        g.mm_q8k(xq, xs, lin, yd, m)
        assert peak_err(g.read(yd, m * n).reshape(m, n), np.stack([orc.matvec_kq(w, 12, n, 4096, x[t]) for t in range(m)])) <= 2e-5
        g.mm(xo, other, yo, (part + room - 4096) // (K * 2), act_mode=pkg.ACT_FLOAT)      # f16 activations that fill the limit but for 4 KB
    finally:
        g.close()


@pytest.mark.parametrize("first", ["decoded", "int8", "few"])
def test_scratch_that_a_call_could_do_without_is_given_back(pkg, orc, monkeypatch, first):
    """A limit that holds what two calls need one after the other: what the first took beside, for speed, does not refuse the second."""
    n, k, m = 1100, 2304, 1900
    w = pkg.synth.q4k_weights(n, k, "scratch", "back")
    x = pkg.synth.normal_f32(m * k, "scratch", "x-back", m)
    need = 2000 * K * 2                                      # f16 activations of the second call
    room = {"decoded": m * k * 5 // 2 + n * k * 2 + 4096, "int8": need + 128 * 1024, "few": need}[first]
    monkeypatch.setenv("OJAS_HIP_SCRATCH_MAX", str(room))
    g = pkg.HipGpu(0)
    try:
        xd, yd = g.upload(x), g.alloc(m * n)
        if first == "decoded":                               # the decoded rows beside the activations
            g.mm(xd, g.lin(12, n, k, w), yd, m, act_mode=pkg.ACT_AUTO)
            assert g.has_kernel("gemm_f16d_128")
            need = room - 1024 * 1024
        elif first == "int8":                                # the side arrays of the 64-row tile
            w4 = pkg.synth.q4k_weights(2112, 4096, "scratch", "back")
            g.mm(xd, g.lin(12, 2112, 4096, w4), yd, 24, act_mode=pkg.ACT_Q8K)
        else:                                                # one token's int8 copy
            g.mm(xd, g.lin(12, n, k, w), yd, 1, act_mode=pkg.ACT_Q8K)
        toks = need // (K * 2)
        xo = pkg.synth.normal_f32(toks * K, "scratch", "x-back2").reshape(toks, K)
        yo = g.alloc(toks * 256)
        g.mm(g.upload(xo), g.lin(Q6_K, 256, K, _weights(pkg, 256)), yo, toks, act_mode=pkg.ACT_FLOAT)
        _check(g, yo, 256, toks, slice(0, 4), _want(pkg, orc, xo[:4]))
    finally:
        g.close()
