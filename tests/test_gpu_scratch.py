"""What the library's scratch does when memory is short: calls that can do without a buffer do without it."""
import numpy as np
import pytest

from conftest import peak_err

pytestmark = pytest.mark.gpu
Q6_K = 14
K = 2048


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
