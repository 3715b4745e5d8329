"""Q4_K rows against batches of tokens on the int8 matrix cores (`gemm_q8k_q4k_mf`): the CPU
reference's arithmetic at verify and prefill sizes — every token against matvec_kq
(crates/ojas-cpu/src/cpu_math.rs:1145-1189), the same bar as the one-token kernels."""
import numpy as np
import pytest

from conftest import peak_err

pytestmark = pytest.mark.gpu
Q4_K = 12
TOL_SEEN = 2e-5


def _case(pkg, m, n, k, tag):
    w = pkg.synth.q4k_weights(n, k, "gq", tag, n, k)
    x = pkg.synth.normal_f32(m * k, "gq", tag, "x", m, k).reshape(m, k)
    x[0, :256] = 0.0                      # an all-zero segment: scale 1
    return w, x


@pytest.mark.parametrize("m,n,k,accum", [(2, 50, 256, False), (16, 130, 4096, True), (17, 333, 2560, False),
                                         (40, 64, 14336, True), (128, 100, 1024, False), (129, 300, 512, False),
                                         (300, 40, 4096, True), (8, 4099, 4096, False), (64, 17, 8192, False),
                                         (130, 6200, 512, True),
                                         # the 128-token tile in K slices below 128 tokens: from 17 tokens where K >= 2 N, from 33 otherwise
                                         (20, 1030, 4096, True), (33, 2100, 2048, False), (64, 4096, 4096, False)])
def test_router_path_matches_the_cpu_reference(gpu, orc, pkg, m, n, k, accum):
    w, x = _case(pkg, m, n, k, "a")
    lin = gpu.lin(Q4_K, n, k, w)
    y0 = pkg.synth.normal_f32(m * n, "gq", "y0", m, n).reshape(m, n) if accum else np.zeros((m, n), np.float32)
    yd = gpu.upload(np.concatenate([y0.ravel(), np.full(n, 4242.5, np.float32)]))
    gpu.mm(gpu.upload(x), lin, yd, m, accum, act_mode=pkg.ACT_Q8K)
    got = gpu.read(yd, m * n + n)
    assert np.all(got[m * n:] == 4242.5), "wrote past the last token"
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    assert peak_err(got[:m * n].reshape(m, n) - y0, want) <= TOL_SEEN


@pytest.mark.parametrize("m,n,k", [(5, 70, 4096), (33, 200, 2048), (100, 48, 14336), (128, 64, 512)])
def test_every_row_tiling_and_the_integer_dot_kernel_agree(gpu, orc, pkg, m, n, k):
    """By name: RW = 1, 2, 4 row tiles per workgroup (4, 2, 1 waves on K) where the tokens' chunk
    allows it, and `gemv_q8k_q4k_m` on the same quantized activations.  Integer sums are exact in
    all of them; the f32 sums over super-blocks associate differently."""
    w, x = _case(pkg, m, n, k, "b")
    gpu.ensure_family("gemm_q8k")
    gpu.ensure_family("gemv_q8k")
    nsb = k // 256
    xq, xs = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
    gpu.quant_q8k(gpu.upload(x), m, k, xq, xs)
    wd = gpu.upload_bytes(w)
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    y = gpu.alloc(m * n)
    gpu.dispatch(gpu.begin(), "gemv_q8k_q4k_m", [(xq, 0), (xs, 0), (wd, 0), (y, 0)], [k, n, m, 0],
                 [(n + 3) // 4, 1, 1], [256, 1, 1])
    dots = gpu.read(y, m * n).reshape(m, n)
    ran = 0
    for rw in (1, 2, 4):
        grid = [(n + 16 * rw - 1) // (16 * rw), (m + 63) // 64, 1]
        y = gpu.upload(np.full(m * n, 7.0, np.float32))
        try:
            gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (y, 0)], [k, n, m, 0, rw, 1], grid,
                         [256, 1, 1])
        except pkg.OjasHipError as e:
            assert "super-blocks" in str(e)            # the chunk is too short for that many waves on K
            continue
        got = gpu.read(y, m * n).reshape(m, n)
        assert peak_err(got, want) <= TOL_SEEN, rw
        assert peak_err(got, dots) <= 2e-6, rw
        ran += 1
    assert ran >= 1
    with pytest.raises(pkg.OjasHipError, match="RT"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (y, 0)], [k, n, m, 0, 4, 4],
                     [(n + 255) // 256, (m + 63) // 64, 1], [256, 1, 1])
    with pytest.raises(pkg.OjasHipError, match="RW"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (y, 0)], [k, n, m, 0, 3, 1],
                     [(n + 47) // 48, (m + 63) // 64, 1], [256, 1, 1])
    with pytest.raises(pkg.OjasHipError, match="grid"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (y, 0)], [k, n, m, 0, 4, 1], [100000, 1, 1],
                     [256, 1, 1])


@pytest.mark.parametrize("m,n,k,accum,grid_x,block_x", [(2, 50, 256, False, None, 512), (16, 130, 4096, True, 3, 512),
                                                        (9, 301, 4096, False, 2, 256), (16, 1000, 5120, False, 7, 512),
                                                        (1, 17, 512, True, None, 64), (5, 4099, 2560, False, None, 512),
                                                        (8, 77, 1024, True, 1, 128)])
def test_rows_copied_through_lds_by_name(gpu, orc, pkg, m, n, k, accum, grid_x, block_x):
    """`gemm_q8k_q4k_ml`, up to 16 tokens: against matvec_kq per token and, bit for bit, against
    `gemm_q8k_q4k_mf` with four row tiles per workgroup (no wave splits K there either, so the same
    sums in the same order).  Small grids make a wave walk many tiles: its copy ring wraps and runs
    ahead across tile borders; the last row ends exactly at the end of the weight buffer."""
    w, x = _case(pkg, m, n, k, "ml")
    y0 = pkg.synth.normal_f32(m * n, "gq", "ml-y0", m, n).reshape(m, n) if accum else np.zeros((m, n), np.float32)
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    gpu.ensure_family("gemm_q8k")
    nsb = k // 256
    xq, xs = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
    gpu.quant_q8k(gpu.upload(x), m, k, xq, xs)
    wd = gpu.upload_bytes(w)
    grid, block = gpu.launch_shape("gemm_q8k_q4k_ml", k, n, m)
    assert block == [512, 1, 1]
    grid, block = [grid_x or grid[0], 1, 1], [block_x, 1, 1]
    yd = gpu.upload(np.concatenate([y0.ravel(), np.full(8, 4242.5, np.float32)]))
    gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_ml", [(xq, 0), (xs, 0), (wd, 0), (yd, 0)], [k, n, m, int(accum)], grid, block)
    got = gpu.read(yd, m * n + 8)
    assert np.all(got[m * n:] == 4242.5), "wrote past the last token"
    got = got[:m * n].reshape(m, n) - y0
    assert peak_err(got, want) <= TOL_SEEN
    y2 = gpu.upload(y0)
    gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (y2, 0)], [k, n, m, int(accum), 4, 1],
                 [(n + 63) // 64, 1, 1], [256, 1, 1])
    assert np.array_equal(got, gpu.read(y2, m * n).reshape(m, n) - y0)
    for consts, what in (([k, n, 17, 0], "do not fit"), ([8192, n, 4, 0], "do not fit")):
        with pytest.raises(pkg.OjasHipError, match=what):
            gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_ml", [(xq, 0), (xs, 0), (wd, 0), (yd, 0)], consts, [8, 1, 1], [512, 1, 1])


@pytest.mark.parametrize("m,n,k,accum,grid_x", [(2, 50, 256, False, None), (16, 130, 4096, True, 3), (9, 301, 14336, False, None),
                                                (16, 100, 8192, False, 2), (5, 4099, 2560, True, None)])
def test_k_split_over_the_waves_by_name(gpu, orc, pkg, m, n, k, accum, grid_x):
    """`gemm_q8k_q4k_mk`: a workgroup per 16-row tile, super-blocks dealt to its eight waves, partial
    sums added in wave order; token rows past M are a shared block of zeros."""
    w, x = _case(pkg, m, n, k, "mk")
    y0 = pkg.synth.normal_f32(m * n, "gq", "mk-y0", m, n).reshape(m, n) if accum else np.zeros((m, n), np.float32)
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    gpu.ensure_family("gemm_q8k")
    nsb = k // 256
    xq, xs = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
    gpu.quant_q8k(gpu.upload(x), m, k, xq, xs)
    wd = gpu.upload_bytes(w)
    grid, block = gpu.launch_shape("gemm_q8k_q4k_mk", k, n, m)
    grid = [grid_x or grid[0], 1, 1]
    yd = gpu.upload(np.concatenate([y0.ravel(), np.full(8, 4242.5, np.float32)]))
    gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mk", [(xq, 0), (xs, 0), (wd, 0), (yd, 0)], [k, n, m, int(accum)], grid, block)
    got = gpu.read(yd, m * n + 8)
    assert np.all(got[m * n:] == 4242.5), "wrote past the last token"
    assert peak_err(got[:m * n].reshape(m, n) - y0, want) <= TOL_SEEN
    with pytest.raises(pkg.OjasHipError, match="do not fit"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mk", [(xq, 0), (xs, 0), (wd, 0), (yd, 0)], [14336, n, 12, 0], [8, 1, 1], [512, 1, 1])
    with pytest.raises(pkg.OjasHipError, match="block"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mk", [(xq, 0), (xs, 0), (wd, 0), (yd, 0)], [k, n, m, 0], [8, 1, 1], [256, 1, 1])


def test_a_token_does_not_depend_on_its_batch(gpu, pkg):
    """The same tokens rolled by 37 positions: every output bit for bit, moved."""
    m, n, k = 200, 512, 4096
    w, x = _case(pkg, m, n, k, "c")
    lin = gpu.lin(Q4_K, n, k, w)
    y1, y2 = gpu.alloc(m * n), gpu.alloc(m * n)
    gpu.mm(gpu.upload(x), lin, y1, m, act_mode=pkg.ACT_Q8K)
    perm = np.roll(np.arange(m), 37)
    gpu.mm(gpu.upload(x[perm].copy()), lin, y2, m, act_mode=pkg.ACT_Q8K)
    assert np.array_equal(gpu.read(y2, m * n).reshape(m, n), gpu.read(y1, m * n).reshape(m, n)[perm])


@pytest.mark.parametrize("m,n,k", [(130, 200, 512), (128, 128, 256), (300, 77, 2048), (97, 1000, 4096)])
def test_prefill_tiles_by_name(gpu, orc, pkg, m, n, k):
    """`q8k_token_sides` + `gemm_q8k_q4k_xt` / `_xt64` by name: ragged tokens and rows, plain store and accumulate,
    nothing written past row M — against matvec_kq and (a few ulp: the min term is associated per 32-position run
    there, per super-block here) against `gemm_q8k_q4k_mf`; the two tile heights give the same bits."""
    w, x = _case(pkg, m, n, k, "xt")
    gpu.ensure_family("gemm_q8k")
    gpu.ensure_family("gemv_q8k")
    nsb, mp = k // 256, (m + 127) // 128 * 128
    xq, xs = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
    gpu.quant_q8k(gpu.upload(x), m, k, xq, xs)
    wd = gpu.upload_bytes(w)
    xst, sums = gpu.alloc(nsb * mp), gpu.alloc(nsb * mp * 8)
    gpu.dispatch(gpu.begin(), "q8k_token_sides", [(xq, 0), (xs, 0), (xst, 0), (sums, 0)], [k, m, mp], [nsb, (mp + 255) // 256, 1], [256, 1, 1])
    # the side arrays: scales transposed; scale x the sum of every 32-position run, runs in the order 0 4 1 5 2 6 3 7;
    # zeros past row M
    q = gpu.read(xq, m * k, np.int8).reshape(m, nsb, 8, 32).astype(np.int32).sum(3)
    st = gpu.read(xst, nsb * mp).reshape(nsb, mp)
    assert np.array_equal(st[:, :m], gpu.read(xs, m * nsb).reshape(m, nsb).T) and not st[:, m:].any()
    sd = gpu.read(sums, nsb * mp * 8).reshape(nsb, mp, 8)
    scaled = st[:, :m, None] * q.transpose(1, 0, 2)[:, :, [0, 4, 1, 5, 2, 6, 3, 7]].astype(np.float32)
    assert np.array_equal(sd[:, :m].view(np.uint32), scaled.astype(np.float32).view(np.uint32)) and not sd[:, m:].any()
    # the quantizer that leaves the side arrays as well: the same bytes in all four outputs, from f32 and from bf16 tokens
    xb = (x.view(np.uint32) >> 16).astype(np.uint16)
    for name, src in (("quantize_q8k_sides", gpu.upload(x)), ("quantize_q8k_bf16_sides", gpu.upload_bytes(xb))):
        q2, s2 = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
        xst2 = gpu.upload(np.full(nsb * mp, 7.5, np.float32))
        sums2 = gpu.upload(np.full(nsb * mp * 8, 7.5, np.float32))
        gpu.dispatch(gpu.begin(), name, [(src, 0), (q2, 0), (s2, 0), (xst2, 0), (sums2, 0)], [k, m, mp], [nsb * mp // 4, 1, 1], [256, 1, 1])
        if "bf16" in name:
            q1, s1 = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
            gpu.quant_q8k(gpu.upload((xb.astype(np.uint32) << 16).view(np.float32)), m, k, q1, s1)
            xst1, sums1 = gpu.alloc(nsb * mp), gpu.alloc(nsb * mp * 8)
            gpu.dispatch(gpu.begin(), "q8k_token_sides", [(q1, 0), (s1, 0), (xst1, 0), (sums1, 0)], [k, m, mp], [nsb, (mp + 255) // 256, 1], [256, 1, 1])
        else:
            q1, s1, xst1, sums1 = xq, xs, xst, sums
        assert np.array_equal(gpu.read(q2, m * k, np.int8), gpu.read(q1, m * k, np.int8)), name
        assert np.array_equal(gpu.read(s2, m * nsb).view(np.uint32), gpu.read(s1, m * nsb).view(np.uint32)), name
        assert np.array_equal(gpu.read(xst2, nsb * mp).view(np.uint32), gpu.read(xst1, nsb * mp).view(np.uint32)), name
        assert np.array_equal(gpu.read(sums2, nsb * mp * 8).view(np.uint32), gpu.read(sums1, nsb * mp * 8).view(np.uint32)), name
    with pytest.raises(pkg.OjasHipError, match="rounded up to 128"):
        gpu.dispatch(gpu.begin(), "quantize_q8k_sides", [(gpu.upload(x), 0), (xq, 0), (xs, 0), (xst, 0), (sums, 0)], [k, m, mp + 128],
                     [nsb * (mp + 128) // 4, 1, 1], [256, 1, 1])
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    ymf = gpu.alloc(m * n)
    gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (ymf, 0)], [k, n, m, 0, 4, 1],
                 [(n + 63) // 64, (m + 63) // 64, 1], [256, 1, 1])
    ref, bits = gpu.read(ymf, m * n).reshape(m, n), {}
    for name, br in (("gemm_q8k_q4k_xt", 128), ("gemm_q8k_q4k_xt64", 64)):
        for acc in (0, 1):
            y0 = pkg.synth.normal_f32(m * n, "gq", "xt-y0", acc).reshape(m, n)
            yd = gpu.upload(np.concatenate([y0.ravel(), np.full(n, 4242.5, np.float32)]))
            gpu.dispatch(gpu.begin(), name, [(xq, 0), (xst, 0), (sums, 0), (wd, 0), (yd, 0)], [k, n, m, acc, mp],
                         [(n + br - 1) // br, mp // 128, 1], [512, 1, 1])
            got = gpu.read(yd, m * n + n)
            assert np.all(got[m * n:] == 4242.5), "wrote past the last token"
            got = got[:m * n].reshape(m, n)
            if acc:
                assert peak_err(got - y0, want) <= TOL_SEEN
            else:
                assert peak_err(got, want) <= TOL_SEEN and peak_err(got, ref) <= 2e-6
                bits[name] = got.view(np.uint32).copy()
    assert np.array_equal(bits["gemm_q8k_q4k_xt"], bits["gemm_q8k_q4k_xt64"])
    # the 64-row tile over K slices: one slice gives the unsliced bits; more give the slice sums added in slice order
    # (the same bits on every launch, whoever finishes last), and every launch leaves the tile counters at zero
    tiles = (n + 63) // 64 * (mp // 128)
    cnt = gpu.alloc_bytes(tiles * 4)
    gpu.memset0(cnt)
    for nsplit in sorted({min(s, nsb) for s in (1, 2, 3, nsb)}):
        per = (nsb + nsplit - 1) // nsplit
        slices = (nsb + per - 1) // per
        part = gpu.alloc(tiles * slices * 8192)
        seen = []
        for acc in (0, 1, 0):
            y0 = pkg.synth.normal_f32(m * n, "gq", "xt-y0", acc).reshape(m, n)
            yd = gpu.upload(np.concatenate([y0.ravel(), np.full(n, 4242.5, np.float32)]))
            gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_xt64_sr", [(xq, 0), (xst, 0), (sums, 0), (wd, 0), (yd, 0), (part, 0), (cnt, 0)],
                         [k, n, m, acc, mp, nsplit], [(n + 63) // 64, mp // 128, slices], [512, 1, 1])
            got = gpu.read(yd, m * n + n)
            assert np.all(got[m * n:] == 4242.5), "wrote past the last token"
            assert not gpu.read(cnt, tiles, np.uint32).any()
            got = got[:m * n].reshape(m, n)
            if acc:
                assert peak_err(got - y0, want) <= TOL_SEEN
            else:
                assert peak_err(got, want) <= TOL_SEEN and peak_err(got, ref) <= 2e-6
                seen.append(got.view(np.uint32).copy())
        assert np.array_equal(seen[0], seen[1]), nsplit
        if slices == 1:
            assert np.array_equal(seen[0], bits["gemm_q8k_q4k_xt64"])
    with pytest.raises(pkg.OjasHipError, match="grid must be"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_xt64_sr", [(xq, 0), (xst, 0), (sums, 0), (wd, 0), (ymf, 0), (part, 0), (cnt, 0)],
                     [k, n, m, 0, mp, 1], [(n + 63) // 64, mp // 128, 2], [512, 1, 1])
    with pytest.raises(pkg.OjasHipError, match="rounded up to 128"):
        gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_xt", [(xq, 0), (xst, 0), (sums, 0), (wd, 0), (ymf, 0)], [k, n, m, 0, mp + 128],
                     [(n + 127) // 128, mp // 128, 1], [512, 1, 1])


@pytest.mark.parametrize("m,n,k", [(1, 64, 256), (40, 130, 512), (64, 65, 2304), (65, 77, 768), (128, 128, 256), (190, 200, 2048), (300, 1000, 1280)])
def test_tile_with_a_cu_to_itself_by_name(gpu, orc, pkg, m, n, k):
    """`gemm_q8k_q4k_xk64{,_sr}` and the side arrays they read: one super-block, odd counts (the second half of K idle in the
    last step), up to 64 tokens in a tile and just past, ragged rows; the sums are `gemm_q8k_q4k_mf`'s terms, two halves of K
    added once (K / 256 f32 additions: 2e-6 of the peak, as for the other tile)."""
    w, x = _case(pkg, m, n, k, "xk")
    gpu.ensure_family("gemm_q8k")
    gpu.ensure_family("gemv_q8k")
    nsb, mp = k // 256, (m + 127) // 128 * 128
    xq, xs, xst, sums = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb), gpu.alloc(nsb * mp), gpu.alloc(nsb * mp * 8)
    gpu.quant_q8k(gpu.upload(x), m, k, xq, xs)
    gpu.dispatch(gpu.begin(), "q8k_token_sides_h", [(xq, 0), (xs, 0), (xst, 0), (sums, 0)], [k, m, mp], [nsb, (mp + 255) // 256, 1], [256, 1, 1])
    # halved run sums and their last bits as f16, zeros past row M; the quantizer that writes them gives the same bytes
    q = gpu.read(xq, m * k, np.int8).reshape(m, nsb, 8, 32).astype(np.int32).sum(3).transpose(1, 0, 2)
    sd = gpu.read(sums, nsb * mp * 16, np.float16).reshape(nsb, mp, 16)
    assert np.array_equal(sd[:, :m, :8], (q >> 1).astype(np.float16)) and np.array_equal(sd[:, :m, 8:], (q & 1).astype(np.float16))
    assert np.array_equal(2 * sd[:, :m, :8].astype(np.int32) + sd[:, :m, 8:].astype(np.int32), q) and not sd[:, m:].any()
    xb = (x.view(np.uint32) >> 16).astype(np.uint16)
    for name, src in (("quantize_q8k_sides_h", x), ("quantize_q8k_bf16_sides_h", xb)):
        bf = src is xb
        q1, s1, t1, u1 = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb), gpu.alloc(nsb * mp), gpu.alloc(nsb * mp * 8)
        gpu.quant_q8k(gpu.upload((xb.astype(np.uint32) << 16).view(np.float32) if bf else x), m, k, q1, s1)
        gpu.dispatch(gpu.begin(), "q8k_token_sides_h", [(q1, 0), (s1, 0), (t1, 0), (u1, 0)], [k, m, mp], [nsb, (mp + 255) // 256, 1], [256, 1, 1])
        q2, s2 = gpu.alloc_bytes(m * k), gpu.alloc(m * nsb)
        t2, u2 = gpu.upload(np.full(nsb * mp, 7.5, np.float32)), gpu.upload(np.full(nsb * mp * 8, 7.5, np.float32))
        gpu.dispatch(gpu.begin(), name, [(gpu.upload_bytes(xb.view(np.uint8)) if bf else gpu.upload(x), 0), (q2, 0), (s2, 0), (t2, 0), (u2, 0)],
                     [k, m, mp], [nsb * mp // 4, 1, 1], [256, 1, 1])
        for a, b, c in ((q1, q2, m * k // 4), (s1, s2, m * nsb), (t1, t2, nsb * mp), (u1, u2, nsb * mp * 8)):
            assert np.array_equal(gpu.read(a, c, np.uint32), gpu.read(b, c, np.uint32)), name
    wd, ymf = gpu.upload_bytes(w), gpu.alloc(m * n)
    gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_mf", [(xq, 0), (xs, 0), (wd, 0), (ymf, 0)], [k, n, m, 0, 4, 1],
                 [(n + 63) // 64, (m + 63) // 64, 1], [256, 1, 1])
    ref = gpu.read(ymf, m * n).reshape(m, n)
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    tiles = (n + 63) // 64 * (mp // 128)
    cnt = gpu.alloc_bytes(tiles * 4)
    gpu.memset0(cnt)
    for nsplit in [0] + sorted({min(s, nsb) for s in (2, 3, nsb)}):
        per = (nsb + nsplit - 1) // nsplit if nsplit else nsb
        slices = (nsb + per - 1) // per
        part = gpu.alloc(tiles * slices * 8192)
        seen = []
        for acc in (0, 1, 0):
            y0 = pkg.synth.normal_f32(m * n, "gq", "xk-y0", acc).reshape(m, n)
            yd = gpu.upload(np.concatenate([y0.ravel(), np.full(n, 4242.5, np.float32)]))
            bufs = [(xq, 0), (xst, 0), (sums, 0), (wd, 0), (yd, 0)]
            gpu.dispatch(gpu.begin(), "gemm_q8k_q4k_xk64_sr" if nsplit else "gemm_q8k_q4k_xk64", bufs + [(part, 0), (cnt, 0)] if nsplit else bufs,
                         [k, n, m, acc, mp, nsplit] if nsplit else [k, n, m, acc, mp], [(n + 63) // 64, mp // 128, slices], [512, 1, 1])
            got = gpu.read(yd, m * n + n)
            assert np.all(got[m * n:] == 4242.5), "wrote past the last token"
            assert not gpu.read(cnt, tiles, np.uint32).any()
            got = got[:m * n].reshape(m, n)
            if acc:
                assert peak_err(got - y0, want) <= TOL_SEEN
            else:
                assert peak_err(got, want) <= TOL_SEEN and peak_err(got, ref) <= 2e-6
                seen.append(got.view(np.uint32).copy())
        assert np.array_equal(seen[0], seen[1]), nsplit


@pytest.mark.parametrize("m,n,k", [(17, 4096, 1024), (33, 1100, 2304), (128, 2048, 4096), (200, 4100, 1280)])
def test_both_forms_of_the_int8_tile_through_mm(pkg, monkeypatch, m, n, k):
    """What `OJAS_HIP_Q4K_XK` chooses between, for the sizes the rule sends to the new form: the same terms in another order."""
    w, x = _case(pkg, m, n, k, "xk-mm")
    outs = []
    for xk in ("0", "1"):
        monkeypatch.setenv("OJAS_HIP_Q4K_XK", xk)
        g = pkg.HipGpu(0)
        try:
            for xd, dt in ((g.upload(x), pkg.X_F32), (g.upload_bytes((x.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8)), pkg.X_BF16)):
                yd = g.upload(np.full(m * n + 64, 4242.5, np.float32))
                g.mm(xd, g.lin(Q4_K, n, k, w), yd, m, x_dtype=dt, act_mode=pkg.ACT_Q8K)
                got = g.read(yd, m * n + 64)
                assert np.all(got[m * n:] == 4242.5)
                outs.append(got[:m * n])
        finally:
            g.close()
    assert peak_err(outs[2], outs[0]) <= 2e-6 and peak_err(outs[3], outs[1]) <= 2e-6


def test_few_tokens_without_room_for_the_tile_keep_their_kernel(pkg, orc, monkeypatch):
    """24 tokens of Q4_K rows run on the 64-row tile where its scratch is to be had.  A limit that holds the quantized tokens
    alone, and a chain recorded before anything ran at that size, leave them on the few-token kernel: the same terms."""
    m, n, k = 24, 700, 2048
    w, x = _case(pkg, m, n, k, "early")
    want = np.stack([orc.matvec_kq(w, Q4_K, n, k, x[t]) for t in range(m)])
    for limit, first in (("0", m), ("65536", m), ("0", 16)):
        monkeypatch.setenv("OJAS_HIP_SCRATCH_MAX", limit)
        g = pkg.HipGpu(0)
        try:
            xd, lin, yd = g.upload(x), g.lin(Q4_K, n, k, w), g.alloc(m * n)
            g.ensure_family("gemm_q8k")
            xq, xs = g.alloc_bytes(m * k), g.alloc(m * k // 256)
            g.quant_q8k(xd, m, k, xq, xs)
            g.mm_q8k(xq, xs, lin, yd, first)
            if first < m:
                g.submit()
                g.capture_begin()
                g.mm_q8k(xq, xs, lin, yd, m)
                chain = g.capture_end()
                chain.launch()
            assert peak_err(g.read(yd, m * n).reshape(m, n), want) <= TOL_SEEN
        finally:
            g.close()


def _bits_of_both_forms(pkg, monkeypatch, m, n, k):
    """ojh_mm on int8 activations with the form that has a CU to itself switched off and as chosen"""
    w, x = _case(pkg, m, 64, k, "xk-route")
    w = np.tile(w.reshape(64, -1), (n // 64 + 1, 1))[:n].ravel()
    outs = []
    for xk in ("0", "1"):
        monkeypatch.setenv("OJAS_HIP_Q4K_XK", xk)
        g = pkg.HipGpu(0)
        try:
            yd = g.alloc(m * n)
            g.mm(g.upload(x), g.lin(Q4_K, n, k, w), yd, m, act_mode=pkg.ACT_Q8K)
            outs.append(g.read(yd, m * n).view(np.uint32))
        finally:
            g.close()
    return outs


@pytest.mark.parametrize("m,n,k,taken", [(24, 6000, 1024, False), (24, 3500, 2048, False), (24, 2100, 2048, True), (24, 4000, 2304, True), (24, 8300, 1024, True)])
def test_few_tokens_take_the_tile_on_long_or_many_rows(pkg, monkeypatch, m, n, k, taken):
    """On short rows the few-token kernel stays ahead unless it walks two tiles a wave; seen by the order of the sums."""
    old, new = _bits_of_both_forms(pkg, monkeypatch, m, n, k)
    assert np.array_equal(old, new) != taken


@pytest.mark.parametrize("m,n,k,taken", [(70, 8300, 12288, False), (60, 8300, 12288, True), (70, 11000, 12288, True)])
def test_three_slices_of_whole_tiles_stay_with_two_workgroups_a_cu(pkg, monkeypatch, m, n, k, taken):
    """130 tiles of more than 64 tokens over three slices of K keep the form that shares a CU; 64 tokens, and two slices, do not."""
    old, new = _bits_of_both_forms(pkg, monkeypatch, m, n, k)
    assert np.array_equal(old, new) != taken


@pytest.mark.parametrize("m,n,k", [(17, 1, 2304), (33, 65, 1024), (32, 64, 5632), (64, 730, 2560), (129, 63, 4096), (300, 130, 3072), (100, 959, 1280)])
@pytest.mark.parametrize("accum", [False, True])
def test_few_rows_take_the_tile_in_slices(gpu, orc, pkg, monkeypatch, m, n, k, accum):
    """Fewer rows than the slices fill half the CUs with: against matvec_kq, one row, rows past a tile, tokens past one; and where
    there is no room for the tile's scratch the few-token kernel still takes the call (which calls take the tile: test_routes.py)."""
    w, x = _case(pkg, m, n, k, "few-rows")
    y0 = pkg.synth.normal_f32(m * n, "gq", "y0", m, n).reshape(m, n) if accum else np.zeros((m, n), np.float32)
    got = []
    for room in (None, str(m * k * 2)):         # (the codes and scales, and half as much again)
        if room:
            monkeypatch.setenv("OJAS_HIP_SCRATCH_MAX", room)
        g = pkg.HipGpu(0) if room else gpu
        try:
            yd = g.upload(np.concatenate([y0.ravel(), np.full(16, 4242.5, np.float32)]))
            g.mm(g.upload(x), g.lin(Q4_K, n, k, w), yd, m, accum=accum, act_mode=pkg.ACT_Q8K)
            out = g.read(yd, m * n + 16)
            assert np.all(out[m * n:] == 4242.5)
            got.append(out[:m * n].reshape(m, n) - y0)
        finally:
            if room:
                g.close()
    for t in sorted({0, m // 2, m - 1}):
        want = orc.matvec_kq(w, Q4_K, n, k, x[t])
        tol = TOL_SEEN * max(1.0, 4.0 * float(np.max(np.abs(y0))) / max(1e-30, float(np.max(np.abs(want)))))
        for out in got:
            assert peak_err(out[t], want) <= tol, t
