"""Recorded chains of dispatches replay with the same results as eager submission."""
import numpy as np
import pytest

from conftest import peak_err

pytestmark = pytest.mark.gpu
Q4_K = 12


@pytest.fixture(params=["list", "graph"])
def replay_mode(request, monkeypatch):
    """The two replay engines: the library's own command list (default) and an instantiated hipGraph."""
    if request.param == "graph":
        monkeypatch.setenv("OJAS_HIP_REPLAY", "graph")     # read by capture_begin
    else:
        monkeypatch.delenv("OJAS_HIP_REPLAY", raising=False)
    return request.param


def test_recorded_step_replays_identically(gpu, orc, pkg, replay_mode):
    n, k = 300, 1024
    w = pkg.synth.q4k_weights(n, k, "graph", "w")
    lin = gpu.lin(Q4_K, n, k, w)
    xs = [pkg.synth.normal_f32(k, "graph", "x", i) for i in range(4)]
    xd, yd = gpu.upload(xs[0]), gpu.alloc(n)
    xq, xsc = gpu.alloc_bytes(k), gpu.alloc(k // 256)

    def chain():
        gpu.quant_q8k(xd, 1, k, xq, xsc)
        gpu.mm_q8k(xq, xsc, lin, yd)

    chain()                      # eager once: loads the families, sizes nothing lazily later
    eager = gpu.read(yd, n)
    gpu.capture_begin()
    chain()
    with pytest.raises(pkg.OjasHipError, match="recording"):
        gpu.submit()
    with pytest.raises(pkg.OjasHipError, match="recording"):
        gpu.alloc(16)
    graph = gpu.capture_end()
    # replay several times with eager work and synchronisations in between; every replay is checked
    for i, x in enumerate(xs):
        gpu.write_bytes(xd, 0, x)
        gpu.memset0(yd)
        graph.launch()
        got = gpu.read(yd, n)
        want = orc.matvec_kq(w, Q4_K, n, k, x)
        assert peak_err(got, want) <= 2e-5, i
        if i == 0:
            assert np.array_equal(got, eager)
    graph.free()


def test_replay_survives_a_scratch_buffer_that_grows(gpu, orc, pkg, replay_mode):
    """`ojh_mm` stages quantized activations in the library's scratch; a chain recorded at m = 1 keeps that address.
    A later eager call with more tokens outgrows the buffer: the old one must stay alive for the chain."""
    n, k = 256, 2048
    w = pkg.synth.q4k_weights(n, k, "graph", "w2")
    lin = gpu.lin(Q4_K, n, k, w)
    x1 = pkg.synth.normal_f32(k, "graph", "x1")
    xd, yd = gpu.upload(x1), gpu.alloc(n)
    gpu.mm(xd, lin, yd, 1, act_mode=pkg.ACT_Q8K)     # eager once: families loaded, scratch sized for one token
    want = gpu.read(yd, n)
    gpu.capture_begin()
    gpu.mm(xd, lin, yd, 1, act_mode=pkg.ACT_Q8K)
    graph = gpu.capture_end()
    m_big = 4096                                        # 8 MB of int8 activations: far beyond the recorded buffer
    xb, yb = gpu.upload(pkg.synth.normal_f32(m_big * k, "graph", "xbig")), gpu.alloc(m_big * n)
    gpu.mm(xb, lin, yb, m_big, act_mode=pkg.ACT_Q8K)
    big = [gpu.alloc_bytes(m_big * k) for _ in range(4)]   # allocations that would reuse freed scratch addresses
    for b in big:
        gpu.memset0(b)
    for _ in range(3):
        gpu.memset0(yd)
        graph.launch()
        assert np.array_equal(gpu.read(yd, n), want)
    assert peak_err(want, orc.matvec_kq(w, Q4_K, n, k, x1)) <= 2e-5
    graph.free()


def test_a_failed_call_while_recording_leaves_the_device_usable(gpu, pkg, replay_mode):
    n, k = 64, 512
    lin = gpu.lin(Q4_K, n, k, pkg.synth.q4k_weights(n, k, "graph", "w3"))
    xd, yd, small = gpu.upload(pkg.synth.normal_f32(k, "graph", "x3")), gpu.alloc(n), gpu.alloc(n // 2)
    gpu.mm(xd, lin, yd, 1, act_mode=pkg.ACT_Q8K)
    want = gpu.read(yd, n)
    gpu.capture_begin()
    with pytest.raises(pkg.OjasHipError) as e:
        gpu.mm(xd, lin, small, 1, act_mode=pkg.ACT_Q8K)        # y too small: refused before anything is queued
    assert e.value.code == -5
    try:
        gpu.capture_end().free()
    except pkg.OjasHipError:
        pass                                                     # the recording is over either way
    gpu.memset0(yd)
    gpu.mm(xd, lin, yd, 1, act_mode=pkg.ACT_Q8K)
    assert np.array_equal(gpu.read(yd, n), want)


def test_recorded_batch_needs_no_more_scratch_than_the_calls_before_it(gpu, orc, pkg):
    """A batch of Q6_K rows is decoded into scratch from some token count on.  Recorded after eager calls that left
    everything but that scratch in place, it runs on the tile that decodes on the way into LDS instead of being refused."""
    n, k, few, m = 16448, 256, 256, 300           # (257 tokens is where rows of this many start to be decoded first)
    w = pkg.synth.q6k_weights(n, k, "graph", "w6")
    x = pkg.synth.normal_f32(m * k, "graph", "x6").reshape(m, k)
    g = pkg.HipGpu(0)
    try:
        lin, xd, yd = g.lin(14, n, k, w), g.upload(x), g.alloc(m * n)
        g.mm(xd, lin, yd, few, act_mode=pkg.ACT_FLOAT)
        g.capture_begin()
        g.mm(xd, lin, yd, m, act_mode=pkg.ACT_FLOAT)
        graph = g.capture_end()
        rows = np.r_[0:16, n - 16:n]
        rb = len(w) // n
        want = orc.matmul_ref(np.concatenate([w[r * rb:(r + 1) * rb] for r in rows]), 14, len(rows), k, x, wmode=1, xmode=1)
        for _ in range(3):
            g.memset0(yd)
            graph.launch()
            # f16 operands: exact products, K of them added in f32 — about sqrt(K) 2^-24 of sum |products|, itself some
            # 0.15 sqrt(K) peaks for such inputs: 2.3e-6; K 2^-24 = 1.5e-5 leaves a factor of six
            assert peak_err(g.read(yd, m * n).reshape(m, n)[:, rows], want) <= k * 2.0 ** -24
        graph.free()
    finally:
        g.close()


@pytest.mark.parametrize("ty", [14, 18])
def test_a_smaller_batch_is_recorded_after_eager_long_ones(orc, pkg, ty):
    """Eager calls long enough for the decode pass and the copied tile leave behind what a recorded call of fewer tokens
    needs: the tile that decodes Q6_K rows on the way into LDS, the plain f16 tile behind the decoded rows of IQ3_XXS."""
    n, k, many, few = 256, 512, 300, 100
    w = pkg.synth.weights(ty, n, k, "graph", "w7")
    x = pkg.synth.normal_f32(many * k, "graph", "x7").reshape(many, k)
    g = pkg.HipGpu(0)
    try:
        lin, xd, yd = g.lin(ty, n, k, w), g.upload(x), g.alloc(many * n)
        g.mm(xd, lin, yd, many, act_mode=pkg.ACT_FLOAT)
        g.capture_begin()
        g.mm(xd, lin, yd, few, act_mode=pkg.ACT_FLOAT)
        graph = g.capture_end()
        want = orc.matmul_ref(w, ty, n, k, x[:few], wmode=1, xmode=1)
        for _ in range(3):
            g.memset0(yd)
            graph.launch()
            # f16 operands, K products added in f32: K 2^-24 of the peak (the magnitudes sum to some 0.15 sqrt(K) peaks)
            assert peak_err(g.read(yd, few * n).reshape(few, n), want) <= k * 2.0 ** -24
        graph.free()
    finally:
        g.close()


@pytest.mark.parametrize("n2,few", [(1100, 100), (1180, 1900)])
def test_q4k_batches_are_recorded_after_eager_ones_that_were_decoded_first(orc, pkg, n2, few):
    """1900 tokens of 1100 Q4_K rows are decoded ahead of the copied tile, whose family alone they need.  A recorded batch of fewer
    tokens, and one of more rows than the decoded rows' scratch holds, run on the tiles that read Q4_K rows."""
    n, k, many = 1100, 2304, 1900
    x = pkg.synth.normal_f32(many * k, "graph", "x8").reshape(many, k)
    w, w2 = pkg.synth.q4k_weights(n, k, "graph", "w8"), pkg.synth.q4k_weights(n2, k, "graph", "w9")
    g = pkg.HipGpu(0)
    try:
        lin, lin2, xd, yd = g.lin(Q4_K, n, k, w), g.lin(Q4_K, n2, k, w2), g.upload(x), g.alloc(many * n2)
        g.mm(xd, lin, yd, many, act_mode=pkg.ACT_AUTO)
        assert g.has_kernel("gemm_f16d_128")
        g.capture_begin()
        g.mm(xd, lin2, yd, few, act_mode=pkg.ACT_AUTO)
        graph = g.capture_end()
        rows = np.r_[0:3, n2 // 2, n2 - 2:n2]
        bits = np.asarray(orc.q4l_weights_f16(w2, k, n2)).view(np.float16).astype(np.float64).reshape(n2, k)[rows]
        want = x[:few].astype(np.float16).astype(np.float64) @ bits.T
        for _ in range(3):
            g.memset0(yd)
            graph.launch()
            # f16 operands, K products added in f32: K 2^-24 of the peak (the magnitudes sum to some 0.15 sqrt(K) peaks)
            assert peak_err(g.read(yd, few * n2).reshape(few, n2)[:, rows], want) <= 2 * k * 2.0 ** -24
        graph.free()
    finally:
        g.close()


def test_int8_batch_recorded_after_an_eager_longer_one_has_its_slices_places(orc, pkg):
    """256 int8 tokens of 8192 Q4_K rows fill the chip with whole tiles; 100 need two K slices of them, which meet in scratch.  The
    longer call leaves that scratch behind for a shorter one that is recorded."""
    n, k, many, few = 8192, 8192, 256, 100
    rows = pkg.synth.q4k_weights(256, k, "graph", "w10")
    x = pkg.synth.normal_f32(many * k, "graph", "x10").reshape(many, k)
    g = pkg.HipGpu(0)
    try:
        lin, xd, yd = g.lin(Q4_K, n, k, np.tile(rows, n // 256)), g.upload(x), g.alloc(many * n)
        g.mm(xd, lin, yd, many, act_mode=pkg.ACT_Q8K)
        g.capture_begin()
        g.mm(xd, lin, yd, few, act_mode=pkg.ACT_Q8K)
        graph = g.capture_end()
        toks = [0, 63, few - 1]
        want = np.stack([np.tile(orc.matvec_kq(rows, Q4_K, 256, k, x[t]), n // 256) for t in toks])
        for _ in range(3):
            g.memset0(yd)
            graph.launch()
            assert peak_err(g.read(yd, few * n).reshape(few, n)[toks], want) <= 2e-5
        graph.free()
    finally:
        g.close()


@pytest.mark.parametrize("multi", [False, True])
@pytest.mark.parametrize("ty", [12, 13])
def test_one_token_recorded_after_a_small_matrix_quantized_inside_its_launch(orc, pkg, ty, multi):
    """A small matrix of one token quantizes inside its launch; a larger one of the same K, and the same with a bias, quantize ahead
    of it into scratch, which the small one's eager call leaves behind."""
    k, small, large = 8192, 64, 8192
    rows = pkg.synth.weights(ty, small, k, "graph", "w11")
    x, b = pkg.synth.normal_f32(k, "graph", "x11"), pkg.synth.normal_f32(small, "graph", "b11")
    g = pkg.HipGpu(0)
    try:
        ls, ll = g.lin(ty, small, k, rows), g.lin(ty, large, k, np.tile(rows, large // small))
        xd, bd, ys, yl = g.upload(x), g.upload(b), g.alloc(small), g.alloc(large)
        call = (lambda lin, y: g.mm_multi(xd, [lin], [y])) if multi else (lambda lin, y: g.mm(xd, lin, y, 1, act_mode=pkg.ACT_Q8K))
        call(ls, ys)
        g.capture_begin()
        call(ll, yl)
        g.mm(xd, ls, ys, 1, bias=bd, act_mode=pkg.ACT_Q8K)
        graph = g.capture_end()
        want = orc.matvec_kq(rows, ty, small, k, x)
        for _ in range(3):
            g.memset0(yl)
            g.memset0(ys)
            graph.launch()
            assert peak_err(g.read(yl, large), np.tile(want, large // small)) <= 2e-5
            assert peak_err(g.read(ys, small), want + b) <= 2e-5
        graph.free()
    finally:
        g.close()


def test_a_batch_of_a_few_more_tokens_is_recorded_after_an_eager_one(orc, pkg):
    """Scratch that grows takes a quarter more than was asked for: 36 tokens are recorded after 30, which the few-token kernel reads
    in groups of sixteen."""
    n, k, first, more = 96, 512, 30, 36
    w = pkg.synth.weights(23, n, k, "graph", "w12")
    x = pkg.synth.normal_f32(more * k, "graph", "x12").reshape(more, k)
    g = pkg.HipGpu(0)
    try:
        lin, xd, yd = g.lin(23, n, k, w), g.upload(x), g.alloc(more * n)
        g.mm(xd, lin, yd, first, act_mode=pkg.ACT_FLOAT)
        g.capture_begin()
        g.mm(xd, lin, yd, more, act_mode=pkg.ACT_FLOAT)
        graph = g.capture_end()
        want = orc.matmul_ref(w, 23, n, k, x, wmode=1, xmode=1)
        for _ in range(3):
            g.memset0(yd)
            graph.launch()
            # f16 operands, K products added in f32: K 2^-24 of the peak (the magnitudes sum to some 0.15 sqrt(K) peaks)
            assert peak_err(g.read(yd, more * n).reshape(more, n), want) <= k * 2.0 ** -24
        graph.free()
    finally:
        g.close()


def _layer(g, pkg, E, d, nff, dty, tag):
    """Expert tensors of one layer, a few experts' rows repeated, as what `moe_ffn_routed` takes."""
    lins = []
    for ty, n, k in ((Q4_K, nff, d), (Q4_K, nff, d), (dty, d, nff)):
        few = min(E, 4)
        rows = pkg.synth.weights(ty, few * n, k, "graph-moe", tag, ty, n, k, len(lins))
        lins.append(g.lin(ty, E * n, k, np.tile(rows, -(-E // few))[:len(rows) // few * E]))
    return lins


def _expert_call(g, pkg, lins, T, E, ksel, d, nff):
    x = pkg.synth.normal_f32(T * d, "graph-moe", "x", T, d)
    lg = pkg.synth.normal_f32(T * E, "graph-moe", "lg", T, E)
    bufs = [g.upload(x), g.upload(lg), g.alloc_bytes(T * ksel * 4), g.alloc(T * ksel), g.alloc(T * d)]

    def call():
        g.moe_ffn_routed(bufs[0], T, d, nff, E, ksel, bufs[1], bufs[2], bufs[3], *lins, bufs[4])

    return call, bufs[4], T * d


def _replays(g, calls):
    """The calls recorded one after the other: three replays against the eager results of another time."""
    g.capture_begin()
    try:
        for call, _, _ in calls:
            call()
    finally:
        graph = g.capture_end()
    outs = []
    for _ in range(3):
        for _, y, _ in calls:
            g.memset0(y)
        graph.launch()
        outs.append([g.read(y, n) for _, y, n in calls])
        for call, y, n in calls:
            g.memset0(y)
            call()
            outs[-1].append(g.read(y, n))
    graph.free()
    return outs


def test_expert_layers_are_recorded_after_an_eager_one_of_more_tokens(pkg):
    """300 experts, top 8: 200 tokens find their assignments on the wave tiles, 70 take lists, 40 find theirs on integer dots, 4 take
    the decode form.  What the first leaves behind is enough for the others, whichever way each runs."""
    E, ksel, d, nff = 300, 8, 256, 256
    g = pkg.HipGpu(0)
    try:
        lins = _layer(g, pkg, E, d, nff, Q4_K, "many")
        first, y, n = _expert_call(g, pkg, lins, 200, E, ksel, d, nff)
        first()
        assert np.isfinite(g.read(y, n)).all()
        calls = [_expert_call(g, pkg, lins, T, E, ksel, d, nff) for T in (70, 40, 4)]
        for out in _replays(g, calls):
            for a, b in zip(out[:3], out[3:]):
                assert a.any() and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        g.close()


def test_an_expert_layer_of_larger_experts_is_recorded_after_one_in_the_decode_form(pkg):
    """4 tokens of a layer whose experts are small enough for the decode form leave behind what the next layer's, with a finer down
    tensor, need grouped."""
    T, E, ksel, d, nff = 4, 8, 4, 1024, 512
    g = pkg.HipGpu(0)
    try:
        small, large = (_layer(g, pkg, E, d, nff, ty, "mixed") for ty in (Q4_K, 14))
        eager = _expert_call(g, pkg, small, T, E, ksel, d, nff)
        eager[0]()
        calls = [_expert_call(g, pkg, large, T, E, ksel, d, nff), eager]
        for out in _replays(g, calls):
            for a, b in zip(out[:2], out[2:]):
                assert a.any() and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        g.close()


@pytest.mark.parametrize("limit", [None, 65536])
def test_two_tokens_of_large_experts_without_the_grouped_scratch(pkg, monkeypatch, limit):
    """Two tokens over experts of more than 32 MB in all are grouped where the scratch is to be had.  Recorded after one token of
    another layer, or under a limit that holds the activations alone, they run in the decode form, which needs no more than that."""
    T, E, ksel, d, nff = 2, 16, 8, 2048, 768
    if limit:
        monkeypatch.setenv("OJAS_HIP_SCRATCH_MAX", str(limit))
    g = pkg.HipGpu(0)
    try:
        lins, other = _layer(g, pkg, E, d, nff, Q4_K, "two"), _layer(g, pkg, 8, 256, 2048, Q4_K, "one")
        call, y, n = _expert_call(g, pkg, lins, T, E, ksel, d, nff)
        if limit:
            call()
            got = [g.read(y, n)]
        else:
            _expert_call(g, pkg, other, 1, 8, 8, 256, 2048)[0]()
            got = [out[0] for out in _replays(g, [(call, y, n)])]
    finally:
        g.close()
    monkeypatch.setenv("OJAS_HIP_MOE", "3")
    monkeypatch.setenv("OJAS_HIP_SCRATCH_MAX", "0")
    g = pkg.HipGpu(0)
    try:
        call, y, n = _expert_call(g, pkg, _layer(g, pkg, E, d, nff, Q4_K, "two"), T, E, ksel, d, nff)
        call()
        want = g.read(y, n)
    finally:
        g.close()
    assert want.any()
    for out in got:
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
