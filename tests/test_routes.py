"""Which launches the op-level calls choose: the host code that decides compiled for the CPU, over a runtime that notes each launch
(after the manifest's own checks of its constants, grid and buffers' alignment) instead of issuing it."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ojas-engine_amd", "csrc")
Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 8, 12, 13, 14, 23
AUTO, Q8K, FLOAT = 0, 1, 2
RUNTIME = r"""
#include "ojh_internal.h"
#include <algorithm>
#include <cstring>
static std::string g_log, g_error;
static std::vector<uint32_t> g_consts;
static uintptr_t g_next = 1ull << 40;
static ojh_buf *fake(size_t bytes) {
    ojh_buf *b = new ojh_buf;
    b->ptr = (void *)g_next;
    b->bytes = bytes;
    g_next += (bytes + 4096) & ~(size_t)4095;
    return b;
}
int ojh_fail(int code, const char *fmt, ...) {
    char s[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(s, sizeof s, fmt, ap);
    va_end(ap);
    g_error = s;
    return code;
}
extern "C" int ojh_alloc(ojh_device *, size_t bytes, ojh_buf **out) { *out = fake(bytes); return OJH_OK; }
extern "C" int ojh_free(ojh_device *, ojh_buf *) { return OJH_OK; }
extern "C" int ojh_upload(ojh_device *, ojh_buf *, size_t, const void *, size_t) { return OJH_OK; }
extern "C" int ojh_ensure_family(ojh_device *dev, const char *family) {
    if (dev->modules.count(family)) return OJH_OK;
    if (dev->capturing) return ojh_fail(OJH_ERR_ARG, "family %s while recording", family);
    dev->modules[family] = nullptr;
    return OJH_OK;
}
extern "C" int ojh_launch_shape(const ojh_device *dev, const char *name, uint32_t K, uint32_t N, uint32_t M, uint32_t grid[3], uint32_t block[3]) {
    const ojh_kernel_spec *s = ojh_find_kernel(name);
    return s ? s->shape(s, dev, K, N, M, grid, block) : ojh_fail(OJH_ERR_UNSUPPORTED, "unknown kernel '%s'", name);
}
int ojh_launch(ojh_device *dev, const char *name, const std::vector<void *> &ptrs, const std::vector<uint32_t> &consts, const uint32_t grid[3],
               const uint32_t block[3]) {
    const ojh_kernel_spec *s = ojh_find_kernel(name);
    if (!s || (int)ptrs.size() != s->n_bufs || (int)consts.size() != s->n_consts) return ojh_fail(-99, "%s: not as in the manifest", name);
    if (!dev->modules.count(s->family)) return ojh_fail(OJH_ERR_NOT_LOADED, "%s: family %s", name, s->family);
    size_t need[16] = {}, align[16];
    for (size_t &a : align) a = 4;
    const uint32_t b[3] = {strstr(name, "fq8k_q4k_x4") ? 256 : block[0], block[1], block[2]};     // (a caller's own dispatch of that one: 256 threads)
    if (int rc = s->check(s, consts.data(), grid, b, need, align)) return rc;
    for (size_t i = 0; i < ptrs.size(); i++)
        if (ptrs[i] && (uintptr_t)ptrs[i] % align[i]) return ojh_fail(-98, "%s: buffer %zu not aligned", name, i);
    g_log += std::string(name) + " ";
    g_consts = consts;
    return OJH_OK;
}
static size_t held(const ojh_device *dev) {
    size_t n = 0;
    for (const auto &s : dev->scratch) n += s.second ? s.second->bytes : 0;
    return n;
}
int ojh_scratch_get(ojh_device *dev, const char *name, size_t bytes, ojh_buf **out) {
    ojh_buf *&b = dev->scratch[name];
    if (!b || b->bytes < bytes) {
        if (dev->capturing) return ojh_fail(OJH_ERR_ARG, "scratch '%s' while recording", name);
        if (dev->scratch_max && held(dev) - (b ? b->bytes : 0) + bytes > dev->scratch_max) return ojh_fail(OJH_ERR_HIP, "scratch '%s' over the limit", name);
        b = fake(bytes);
    }
    *out = b;
    return OJH_OK;
}
int ojh_scratch_get_zeroed(ojh_device *dev, const char *name, size_t bytes, ojh_buf **out) { return ojh_scratch_get(dev, name, bytes, out); }
int ojh_scratch_spare(ojh_device *dev, const char *name, size_t bytes, ojh_buf **out, bool) { return ojh_scratch_get(dev, name, bytes, out); }
bool ojh_scratch_fits(const ojh_device *dev, std::initializer_list<std::pair<const char *, size_t>> wanted) {
    size_t n = held(dev);
    bool grows = false;
    for (const auto &w : wanted) {
        const auto it = dev->scratch.find(w.first);
        const size_t has = it == dev->scratch.end() || !it->second ? 0 : it->second->bytes;
        if (has < w.second) grows = true, n += w.second - has;
    }
    return !grows || (!dev->capturing && (!dev->scratch_max || n <= dev->scratch_max));
}

static ojh_lin *lin(uint32_t type, uint32_t n, uint32_t k) {
    const ojh_block_format *f = ojh_format(type);
    ojh_lin *w = new ojh_lin;
    w->type = type, w->n = n, w->k = k;
    w->row_bytes = (size_t)k / f->weights * f->bytes;
    w->raw = fake(w->row_bytes * n + 16);
    return w;
}
extern "C" ojh_device *dev_new() {
    ojh_device *d = new ojh_device;
    d->prop.multiProcessorCount = 256;
    return d;
}
extern "C" void dev_set(ojh_device *d, const char *key, long v) {
    if (!strcmp(key, "moe")) d->moe_mode = (int)v;
    else if (!strcmp(key, "moe_fuse")) d->moe_fuse = v;
    else if (!strcmp(key, "moe_route_fuse")) d->moe_route_fuse = v;
    else if (!strcmp(key, "moe_dec_tokens")) d->moe_dec_tokens = (int)v;
    else if (!strcmp(key, "capturing")) d->capturing = v;
    else if (!strcmp(key, "scratch_max")) d->scratch_max = (uint64_t)v;
    else abort();
}
extern "C" uint32_t last_const(int i) { return g_consts[i]; }      // of the last launch
static int out(int rc, char *log, size_t room) {
    snprintf(log, room, "%s", rc ? g_error.c_str() : g_log.c_str());
    return rc;
}
extern "C" int route_moe(ojh_device *d, int routed, uint32_t T, uint32_t E, uint32_t ksel, uint32_t dim, uint32_t n_ff, uint32_t down, int act, char *log, size_t room) {
    g_log.clear();
    const uint32_t gu = down == OJH_Q8_0 ? OJH_Q8_0 : OJH_Q4_K;
    ojh_buf *x = fake((size_t)T * dim * 4), *y = fake((size_t)T * dim * 4), *lg = fake((size_t)T * E * 4), *idx = fake((size_t)T * ksel * 4), *wgt = fake((size_t)T * ksel * 4);
    ojh_lin *g = lin(gu, E * n_ff, dim), *u = lin(gu, E * n_ff, dim), *dn = lin(down, E * dim, n_ff);
    return out(routed ? ojh_moe_ffn_routed(d, x, T, dim, n_ff, E, ksel, lg, idx, wgt, g, u, dn, y, 0, act)
                      : ojh_moe_ffn(d, x, T, dim, n_ff, E, ksel, idx, wgt, g, u, dn, y, 0, act), log, room);
}
extern "C" int route_mm(ojh_device *d, uint32_t type, uint32_t n, uint32_t k, uint32_t m, int act, int over, char *log, size_t room) {
    g_log.clear();
    ojh_buf *x = fake((size_t)m * k * 4 + (size_t)m * n * 4);
    return out(ojh_mm(d, x, 0, OJH_X_F32, lin(type, n, k), over ? x : fake((size_t)m * n * 4), 0, nullptr, m, 0, act), log, room);
}
// outputs one behind the other in one buffer, `step` bytes apart
extern "C" int route_multi(ojh_device *d, uint32_t type, uint32_t n, uint32_t k, int count, size_t step, int accum, char *log, size_t room) {
    g_log.clear();
    ojh_buf *y = fake((size_t)4 * n * 4), *ys[4] = {y, y, y, y};
    const ojh_lin *ws[4];
    size_t offs[4];
    for (int i = 0; i < count; i++) ws[i] = lin(type, n, k), offs[i] = step * i;
    return out(ojh_mm_multi(d, fake((size_t)k * 4), 0, count, ws, ys, offs, accum), log, room);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    (d / "runtime.cpp").write_text(RUNTIME)
    srcs = [str(d / "runtime.cpp")] + [os.path.join(CSRC, s) for s in ("ojh_moe.cpp", "ojh_ops.cpp", "ojh_manifest.cpp")]
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I", CSRC, "-o", str(d / "r.so"), *srcs, "-L/opt/rocm/lib", "-lamdhip64"])
    so = ctypes.CDLL(str(d / "r.so"))
    so.dev_new.restype = ctypes.c_void_p
    return so


class Dev:
    def __init__(self, lib, **keys):
        self.lib, self.dev = lib, ctypes.c_void_p(lib.dev_new())
        self.set(**keys)

    def set(self, **keys):
        for k, v in keys.items():
            self.lib.dev_set(self.dev, k.encode(), ctypes.c_long(v))

    def _log(self, fn, *args):
        log = ctypes.create_string_buffer(4096)
        rc = fn(self.dev, *args, log, ctypes.c_size_t(4096))
        text = log.value.decode()
        assert rc == 0, text
        return text.split()

    def moe(self, T, E, ksel, d, nff, down=Q4_K, act=AUTO, routed=True):
        return self._log(self.lib.route_moe, int(routed), T, E, ksel, d, nff, down, act)

    def mm(self, ty, n, k, m, act=AUTO, over=False):
        return self._log(self.lib.route_mm, ty, n, k, m, act, int(over))

    def multi(self, ty, n, k, count, step, accum):
        return self._log(self.lib.route_multi, ty, n, k, count, ctypes.c_size_t(step), int(accum))


def _form(launches):
    """Which form of the expert layer these launches are."""
    names = " ".join(launches)
    return "decode" if "_dec" in names else "tiles" if "_ti" in names else "dots" if "q4k_mi" in names else \
        "lists dense" if "_gs" in names else "lists tiles" if "_mt" in names else "lists"


# (T, E, ksel, d, n_ff, down) of one layer for each form
FORMS = {"decode": (1, 128, 8, 2048, 768, Q4_K), "dots": (4, 128, 8, 2048, 768, Q4_K), "tiles": (64, 128, 8, 2048, 768, Q4_K),
         "lists": (16, 128, 8, 2048, 768, Q4_K)}


@pytest.mark.parametrize("form", sorted(FORMS))
def test_the_router_is_a_launch_of_its_own_where_that_is_asked_for(lib, form):
    """OJAS_HIP_MOE_ROUTE_FUSE=0, in every form of the layer; the rest of the layer's launches stays what it was, but for the
    quantizer that the router shared one with."""
    fused, apart = Dev(lib).moe(*FORMS[form]), Dev(lib, moe_route_fuse=0).moe(*FORMS[form])
    assert apart[0] == "moe_topk_m"
    assert apart[1:] == Dev(lib).moe(*FORMS[form], routed=False)
    if form == "lists":
        assert fused == apart
    elif form == "decode":
        assert fused == ["moe_gu_q4k_decr"] + apart[2:]
    else:
        assert fused == ["moe_topk_quant"] + apart[2:]


@pytest.mark.parametrize("n,k,one", [(4096, 4096, True), (2500, 14336, True), (1024, 14336, False), (7500, 5120, True), (7500, 3840, True), (7500, 3072, False),
                                     (5300, 6144, True), (4608, 9984, True), (6144, 5120, False), (6144, 4096, False), (16000, 4096, True), (24000, 4096, False),
                                     (12000, 5120, True), (30000, 9984, True), (30000, 4096, False), (30000, 3072, True), (50000, 1024, True), (50000, 4096, False)])
def test_one_token_of_q6k_rows_on_either_side_of_the_line(lib, n, k, one):
    """The sizes whose times stand beside the rule take the form that is ahead there."""
    got = Dev(lib).mm(Q6_K, n, k, 1)
    assert (got[0].startswith("gemv_fq8k_q6k_one") and len(got) == 1) == one, got
    assert one or got[0] == "quantize_q8k"


@pytest.mark.parametrize("ty,n,k,want", [(Q4_K, 26000, 9216, 104), (Q4_K, 24000, 9984, 96), (Q4_K, 22000, 10752, 88), (Q4_K, 25500, 9216, 100), (Q4_K, 27000, 9216, 106),
                                         (Q5_K, 38400, 5120, 152), (Q5_K, 42496, 9216, 166), (Q6_K, 23040, 7168, 92), (Q4_K, 4096, 4096, 16), (Q5_K, 128256, 2560, 502)])
def test_workgroups_do_not_lie_where_their_streams_meet(lib, ty, n, k, want):
    """A row count a workgroup that puts them a 128th off 512 KB or 1 MB apart is raised by two; others are dealt evenly over 256 CUs."""
    dev = Dev(lib)
    assert "_one_r" in dev.mm(ty, n, k, 1)[-1] and lib.last_const(2) == want
    if ty == Q4_K and k > 4096:
        assert dev.multi(ty, n, k, 1, 0, False) == ["gemv_fq8k_q4k_x4_r2"] and lib.last_const(5) == want


@pytest.mark.parametrize("ty,tag,k,m,shared", [(Q8_0, "q80", 2080, 2, True), (Q8_0, "q80", 2048, 2, False), (IQ4_XS, "iq4xs", 1280, 3, True),
                                               (IQ4_XS, "iq4xs", 1024, 3, False), (Q8_0, "q80", 4096, 31, True), (Q8_0, "q80", 2080, 300, True),
                                               (Q8_0, "q80", 992, 300, False)])
def test_tokens_from_which_waves_share_rows(lib, ty, tag, k, m, shared):
    """f32 activations: both sides of the row length, two tokens, three, and batches that no tile takes."""
    assert Dev(lib).mm(ty, 2000, k, m, FLOAT) == ["gemv_nat_%s_%s" % (tag, "ms" if shared else "m")]


@pytest.mark.parametrize("T,E,ksel,d,nff,down,form", [
    # the decode form: one token always, two up to 32 MB of experts for their assignments, up to 16 MB more
    (1, 128, 8, 4096, 2048, Q4_K, "decode"), (2, 128, 8, 2048, 512, Q4_K, "decode"), (2, 128, 8, 2048, 768, Q4_K, "dots"),
    (6, 96, 4, 512, 768, Q4_K, "decode"), (4, 8, 4, 1024, 512, Q4_K, "decode"), (4, 8, 4, 1024, 512, Q6_K, "dots"), (3, 96, 8, 1536, 768, Q6_K, "dots"),
    # dots below 3.4 - 0.75 d / 1024 assignments an expert, tiles from there; from 1.1 where a row is more than one step
    (42, 128, 8, 1024, 512, Q4_K, "dots"), (43, 128, 8, 1024, 512, Q4_K, "tiles"), (14, 64, 8, 2048, 768, Q4_K, "dots"), (16, 64, 8, 2048, 768, Q4_K, "tiles"),
    (8, 64, 8, 2304, 768, Q4_K, "dots"), (9, 64, 8, 2304, 768, Q4_K, "tiles"),
    # lists where one-step rows have more than 150 MB, beyond what the kernels find, where the dense tile is ahead
    (8, 128, 8, 2048, 768, Q4_K, "dots"), (16, 128, 8, 2048, 768, Q4_K, "lists"), (64, 300, 8, 256, 256, Q4_K, "dots"), (65, 300, 8, 256, 256, Q4_K, "lists"),
    (512, 128, 8, 1024, 512, Q4_K, "tiles"), (513, 128, 8, 1024, 512, Q4_K, "lists tiles"), (512, 64, 8, 4096, 512, Q4_K, "tiles"),
    (512, 64, 8, 4352, 512, Q4_K, "lists tiles"),
    (30, 12, 4, 1024, 512, Q6_K, "lists dense"), (29, 12, 4, 1024, 512, Q6_K, "tiles"), (33, 13, 4, 1024, 512, Q6_K, "tiles"),
    (512, 16, 6, 1024, 512, Q5_K, "lists dense"), (511, 16, 6, 1024, 512, Q5_K, "tiles"), (512, 16, 6, 1024, 512, Q4_K, "tiles"),
    (8, 128, 8, 2048, 2304, Q4_K, "lists")])
def test_forms_of_the_expert_layer_on_either_side_of_their_lines(lib, T, E, ksel, d, nff, down, form):
    for routed in (True, False):
        assert _form(Dev(lib).moe(T, E, ksel, d, nff, down, routed=routed)) == form


def test_two_tokens_without_the_grouped_scratch_keep_the_decode_form(lib):
    """... while the calls of three tokens that are grouped are refused where it is not to be had."""
    shape = (128, 8, 2048, 768)
    assert _form(Dev(lib, scratch_max=2 * 8 * 768 * 4).moe(2, *shape)) == "decode"
    dev = Dev(lib)
    dev.moe(1, 128, 16, 2048, 768)
    dev.set(capturing=1)
    assert _form(dev.moe(2, *shape)) == "decode"
    with pytest.raises(AssertionError, match="gemv_q8k"):
        dev.moe(3, *shape)
    with pytest.raises(AssertionError, match="limit"):
        Dev(lib, scratch_max=3 * 8 * 768 * 4).moe(3, *shape)


@pytest.mark.parametrize("T,then", [(64, 16), (64, 8), (64, 2), (8, 4), (9, 3)])
def test_an_expert_layer_is_recorded_after_any_of_more_tokens(lib, T, then):
    dev = Dev(lib)
    dev.moe(T, 128, 8, 2048, 768)
    dev.set(capturing=1)
    assert dev.moe(then, 128, 8, 2048, 768) == Dev(lib).moe(then, 128, 8, 2048, 768)


@pytest.mark.parametrize("m,n,k,tile", [(17, 1, 2304, True), (33, 65, 1024, True), (32, 64, 5632, True), (64, 730, 2560, True), (16, 64, 5632, False),
                                        (32, 65, 1024, False), (65, 63, 4096, False), (129, 63, 4096, False), (100, 959, 1280, False)])
def test_few_rows_of_q4k_take_the_tile_up_to_half_a_tile_of_tokens(lib, m, n, k, tile):
    """Matrices of fewer rows than the slices fill half the CUs with: eight slices of the tile from 17 tokens (33 on short rows) to 64,
    and the few-token kernel without room for them."""
    for room, taken in ((0, tile), (m * k + m * k // 64 * 2, False)):
        got = Dev(lib, scratch_max=room).mm(Q4_K, n, k, m, Q8K)
        assert ("gemm_q8k_q4k_xk64_sr" in got) == taken, got


@pytest.mark.parametrize("ty,m,n,k,tile", [(Q6_K, 17, 4100, 512, True), (Q6_K, 17, 4096, 512, False), (Q6_K, 32, 130, 4352, True), (Q6_K, 32, 130, 4096, False),
                                           (Q6_K, 16, 4100, 512, False), (Q6_K, 9, 300, 14336, False), (Q6_K, 16, 4096, 14336, False), (Q6_K, 33, 130, 4096, True),
                                           (Q5_K, 5, 8192, 512, True), (Q5_K, 4, 8192, 512, False), (Q5_K, 9, 300, 512, True), (Q5_K, 8, 300, 512, False)])
def test_tokens_from_which_q6k_and_q5k_rows_take_the_int8_tile(lib, ty, m, n, k, tile):
    got = Dev(lib).mm(ty, n, k, m, Q8K)
    assert any("_gs" in name for name in got) == tile, got
    if tile and ty == Q6_K and m < 33:      # the early tile: not where its slices have no room
        assert not any("_gs_sr" in name for name in Dev(lib, scratch_max=m * k + m * k // 64 * 2).mm(ty, n, k, m, Q8K))


@pytest.mark.parametrize("ty", [Q4_K, Q5_K])
@pytest.mark.parametrize("accum", [False, True])
def test_outputs_over_each_other_take_a_launch_each(lib, ty, accum):
    n, k = 600, 4352
    apart, over = (Dev(lib).multi(ty, n, k, 3, step, accum) for step in (n * 4, n * 4 - 4))
    assert over[0] == "quantize_q8k" and len(over) == 4 and len(set(over[1:])) == 1
    if ty == Q4_K:
        assert apart == ["gemv_fq8k_q4k_x4_r2"]
