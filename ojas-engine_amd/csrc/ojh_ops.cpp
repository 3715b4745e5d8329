// Host side of the op seam: weight handles that keep GGUF block bytes in place, and the matmul
// router that picks a kernel per call — the role `Lin::load` and `CudaSsm::mm` play in the
// reference (crates/ojas-cuda/src/qwen35.rs:174-201, :644-702; Metal twin
// crates/ojas-models/src/decoder/dispatch.rs:288-626).
#include <cstdlib>
#include <cmath>
#include <cstring>

#include "ojh_internal.h"

static int ensure(ojh_device *dev, const char *family) {
    return dev->modules.count(family) ? OJH_OK : ojh_ensure_family(dev, family);
}

static int span_ok(const char *what, const ojh_buf *b, size_t off, size_t bytes, size_t align) {
    if (!b) return ojh_fail(OJH_ERR_ARG, "%s: NULL buffer", what);
    if (off > b->bytes || bytes > b->bytes - off)
        return ojh_fail(OJH_ERR_BOUNDS, "%s needs %zu bytes at offset %zu, buffer has %zu", what, bytes, off,
                        b->bytes);
    if (((uintptr_t)b->ptr + off) % align)
        return ojh_fail(OJH_ERR_ARG, "%s (+%zu) must be %zu-byte aligned", what, off, align);
    return OJH_OK;
}

static inline void *at(const ojh_buf *b, size_t off) { return (char *)b->ptr + off; }

static inline bool overlap(const void *a, size_t a_bytes, const void *b, size_t b_bytes) {
    return (uintptr_t)a < (uintptr_t)b + b_bytes && (uintptr_t)b < (uintptr_t)a + a_bytes;
}

// ---- Lin ---------------------------------------------------------------------------------------
static int lin_check(uint32_t type, uint32_t n, uint32_t k, size_t *row_bytes) {
    const ojh_block_format *f = ojh_format(type);
    if (!f) return ojh_fail(OJH_ERR_UNSUPPORTED, "GGUF type %u has no kernel on this backend", type);
    if (!n || !k || k % f->weights)
        return ojh_fail(OJH_ERR_ARG, "Lin %ux%u: K must be a positive multiple of %u for %s", n, k, f->weights,
                        f->tag);
    *row_bytes = (size_t)(k / f->weights) * f->bytes;
    return OJH_OK;
}

extern "C" int ojh_lin_create(ojh_device *dev, uint32_t type, uint32_t n, uint32_t k, const void *raw,
                              ojh_lin **out) {
    if (!dev || !raw || !out) return ojh_fail(OJH_ERR_ARG, "ojh_lin_create: NULL argument");
    *out = nullptr;
    size_t rb;
    int rc = lin_check(type, n, k, &rb);
    if (rc) return rc;
    ojh_buf *buf = nullptr;
    // up to the next multiple of 16: kernels that copy whole aligned 16-byte pieces may read that far
    if ((rc = ojh_alloc(dev, (rb * n + 15) & ~(size_t)15, &buf))) return rc;
    if ((rc = ojh_upload(dev, buf, 0, raw, rb * n))) {
        ojh_free(dev, buf);
        return rc;
    }
    ojh_lin *l = new ojh_lin();
    l->type = type; l->n = n; l->k = k; l->row_bytes = rb; l->raw = buf; l->off = 0; l->owns_raw = true;
    *out = l;
    return OJH_OK;
}

extern "C" int ojh_lin_wrap(ojh_device *dev, uint32_t type, uint32_t n, uint32_t k, ojh_buf *raw, size_t off,
                            ojh_lin **out) {
    if (!dev || !raw || !out) return ojh_fail(OJH_ERR_ARG, "ojh_lin_wrap: NULL argument");
    *out = nullptr;
    size_t rb;
    int rc = lin_check(type, n, k, &rb);
    if (rc) return rc;
    const ojh_block_format *f = ojh_format(type);
    if ((rc = span_ok("ojh_lin_wrap: raw", raw, off, rb * n, ojh_block_align(f)))) return rc;
    ojh_lin *l = new ojh_lin();
    l->type = type; l->n = n; l->k = k; l->row_bytes = rb; l->raw = raw; l->off = off; l->owns_raw = false;
    *out = l;
    return OJH_OK;
}

extern "C" int ojh_lin_free(ojh_device *dev, ojh_lin *lin) {
    if (!lin) return OJH_OK;
    int rc = OJH_OK;
    if (lin->owns_raw) rc = ojh_free(dev, lin->raw);
    delete lin;
    return rc;
}

// ---- dequant -----------------------------------------------------------------------------------
extern "C" int ojh_dequant_f16(ojh_device *dev, uint32_t type, const ojh_buf *raw, size_t raw_off,
                               size_t n_weights, ojh_buf *out, size_t out_off) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_dequant_f16: NULL device");
    const ojh_block_format *f = ojh_format(type);
    if (!f) return ojh_fail(OJH_ERR_UNSUPPORTED, "GGUF type %u has no decoder on this backend", type);
    if (!n_weights || n_weights % f->weights)
        return ojh_fail(OJH_ERR_ARG, "dequant: %zu weights is not a positive multiple of %u", n_weights, f->weights);
    size_t nb = n_weights / f->weights;
    if (nb > 0x7FFFFFFFu / 64) return ojh_fail(OJH_ERR_ARG, "dequant: too many blocks in one call (%zu)", nb);
    int rc;
    if ((rc = span_ok("dequant: raw", raw, raw_off, nb * f->bytes, ojh_block_align(f)))) return rc;
    if ((rc = span_ok("dequant: out", out, out_off, n_weights * 2, 2))) return rc;
    if ((rc = ensure(dev, ojh_grid_type(type) ? "iq_grid" : "dequant"))) return rc;
    std::string name = std::string("dequant_") + f->tag + "_f16";
    uint32_t grid[3], block[3];
    if ((rc = ojh_launch_shape(dev, name.c_str(), 0, (uint32_t)nb, 0, grid, block))) return rc;
    return ojh_launch(dev, name.c_str(), {at(raw, raw_off), at(out, out_off)}, {(uint32_t)nb}, grid, block);
}

extern "C" int ojh_relayout_q4k_q4l(ojh_device *dev, const ojh_buf *raw, size_t raw_off, uint32_t n, uint32_t k,
                                    ojh_buf *nib, ojh_buf *qa, ojh_buf *qb) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_relayout_q4k_q4l: NULL device");
    if (!n || !k || k % 256) return ojh_fail(OJH_ERR_ARG, "relayout_q4k_q4l: %u rows of %u weights (K must be a multiple of 256)", n, k);
    size_t nb = (size_t)n * (k / 256);
    if (nb > 0x0FFFFFFFu) return ojh_fail(OJH_ERR_ARG, "relayout_q4k_q4l: too many super-blocks (%zu)", nb);
    int rc;
    if ((rc = span_ok("relayout: raw", raw, raw_off, nb * 144, 16))) return rc;
    if ((rc = span_ok("relayout: nib", nib, 0, nb * 128, 16))) return rc;
    if ((rc = span_ok("relayout: qa", qa, 0, nb * 16, 2))) return rc;
    if ((rc = span_ok("relayout: qb", qb, 0, nb * 16, 2))) return rc;
    if ((rc = ensure(dev, "dequant"))) return rc;
    uint32_t grid[3] = {(uint32_t)((nb + 31) / 32), 1, 1}, block[3] = {256, 1, 1};
    return ojh_launch(dev, "relayout_q4k_q4l", {at(raw, raw_off), nib->ptr, qa->ptr, qb->ptr}, {(uint32_t)nb}, grid, block);
}

// ---- activation quantizer ----------------------------------------------------------------------
int ojh_quant_q8k_launch(ojh_device *dev, const void *x, int x_dtype, uint32_t m, uint32_t k, void *q,
                            void *scales) {
    const char *name = x_dtype == OJH_X_BF16 ? "quantize_q8k_bf16" : "quantize_q8k";
    uint32_t grid[3] = {(k + 255) / 256, m, 1}, block[3] = {256, 1, 1};
    // many segments (a batch): a segment per wave, four to a workgroup
    const uint64_t segs = (uint64_t)grid[0] * m;
    if (segs >= 1024) {
        uint32_t gw[3] = {(uint32_t)((segs + 3) / 4), 1, 1};
        return ojh_launch(dev, x_dtype == OJH_X_BF16 ? "quantize_q8k_bf16_w" : "quantize_q8k_w", {(void *)x, q, scales}, {k, m}, gw, block);
    }
    return ojh_launch(dev, name, {(void *)x, q, scales}, {k, m}, grid, block);
}

extern "C" int ojh_quant_q8k(ojh_device *dev, const ojh_buf *x, size_t x_off, int x_dtype, uint32_t m,
                             uint32_t k, ojh_buf *q, ojh_buf *scales) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_quant_q8k: NULL device");
    if (x_dtype != OJH_X_F32 && x_dtype != OJH_X_BF16)
        return ojh_fail(OJH_ERR_UNSUPPORTED, "quant_q8k takes f32 or bf16 activations");
    if (!m || !k || m > 65535) return ojh_fail(OJH_ERR_ARG, "quant_q8k: m=%u k=%u out of range", m, k);
    size_t esz = x_dtype == OJH_X_BF16 ? 2 : 4, nsb = (k + 255) / 256;
    int rc;
    if ((rc = span_ok("quant_q8k: x", x, x_off, (size_t)m * k * esz, esz))) return rc;
    if ((rc = span_ok("quant_q8k: q", q, 0, (size_t)m * nsb * 256, 16))) return rc;
    if ((rc = span_ok("quant_q8k: scales", scales, 0, (size_t)m * nsb * 4, 4))) return rc;
    if ((rc = ensure(dev, "gemv_q8k"))) return rc;
    return ojh_quant_q8k_launch(dev, at(x, x_off), x_dtype, m, k, q->ptr, scales->ptr);
}

// ---- mm ----------------------------------------------------------------------------------------
// Rows per wave for the row-parallel matvecs: enough waves to put several on every SIMD, while
// reusing each activation fragment across as many rows as that allows.
static int pick_rows(const ojh_device *dev, uint32_t n) {
    if (dev->gemv_rows_override == 1 || dev->gemv_rows_override == 2 || dev->gemv_rows_override == 4)
        return dev->gemv_rows_override;
    uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
    // Measured on MI355X (Q4_K, K=4096): two rows per wave streams fastest once N gives every CU
    // several workgroups; four rows per wave loses to it at every size.
    return n >= cus * 32u ? 2 : 1;
}

// y (=,+=,+bias) quantized-x . W^T for K-quant weights: the matvec (m = 1) and its batched form.
// Whether a Q4_K product of m tokens takes the 128-token int8 tile (when its tiles cover at least half of the CUs: a
// 4096-row matrix against 128 tokens stays below).
// K slices the 64-row int8 tile is launched over (measured on 4096 / 14336-wide matrices at 128 .. 2048 tokens): two
// workgroups per CU is the aim, with at most eight slices of at least four super-blocks each (two, where four would
// leave more than half the CUs idle); a grid that already covers more than half the CUs is sliced only when a slice
// keeps sixteen super-blocks.  1 = unsliced; 0 = even sliced, most CUs would idle: another kernel takes the product.
// By default the form that has a CU to itself (q4k_xk_slices) runs these grids but for three slices of more than half the CUs'
// tiles: for the others this says whether the int8 tile is taken at all, and what scratch is left behind for recorded calls.
static uint32_t q4k_xt_slices(const ojh_device *dev, uint32_t K, uint32_t N, uint32_t m) {
    const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount, nsb = K / 256;
    const uint64_t tiles = (uint64_t)((N + 63) / 64) * ((m + 127) / 128);
    const uint32_t whole = tiles * 2 >= cus ? 1u : 0u;
    if (dev->q4k_xt_split == 0 || (tiles > cus && dev->q4k_xt_split == 1)) return whole;
    uint32_t z = (uint32_t)(2 * (uint64_t)cus / tiles);
    if (z > 8) z = 8;
    uint32_t cap = nsb / 4;
    if (tiles * (z < cap ? z : cap) * 2 < cus) cap = nsb / 2;
    if (z > cap) z = cap;
    if (tiles * 2 > cus && z > 1 && nsb / z < 16) z = 1;
    if (dev->q4k_xt_split > 1) z = dev->q4k_xt_split <= nsb ? dev->q4k_xt_split : nsb;
    if (z < 2 || tiles * z * 2 < cus) return whole;
    return ojh_gemm_sr_slices(K, z);
}
// Slices of the form that has a CU to itself (1: whole; 0: not this form): up to one tile per CU in all, of at least four
// super-blocks, two where four would leave more than half the CUs idle.  Above one tile per CU two workgroups of the other
// form share it and are as fast or faster.  That form / this one, with the quantizer, us: 14336 x 4096 at 48 tokens 36.5 /
// 21.4, at 128 38.4 / 28.9; 4096 x 14336 at 512 109.5 / 95; 4096^2 at 512 41.9 / 34; at 128 (four slices) 19.0 / 17.5;
// 14336 x 4096 at 256 (448 tiles) 57.8 / 57.8, at 512 84 / 111.  Nor where the other form takes three slices of tiles that cover
// little more than half the CUs here: 4352 x 12800 at 200 tokens (136 tiles) 63.5 / 72, 9600 x 13568 at 120 (150) 65.5 / 75, against
// 12288 x 12800 at 120 (192 tiles, two slices) 85 / 71; up to 64 tokens, half a tile, 9600 x 13568 at 60 63 / 52.
static uint32_t q4k_xk_slices(const ojh_device *dev, uint32_t K, uint32_t N, uint32_t m) {
    const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount, nsb = K / 256;
    const uint64_t tiles = (uint64_t)((N + 63) / 64) * ((m + 127) / 128);
    if (!dev->q4k_xk || dev->q4k_xt64 || dev->q4k_xt_split > 1 || tiles > cus) return 0;
    if (tiles * 2 > cus && m > 64 && q4k_xt_slices(dev, K, N, m) > 2) return 0;
    uint32_t z = std::min<uint32_t>((uint32_t)(cus / tiles), 8u), cap = std::max(nsb / 4, 1u);
    if (dev->q4k_xt_split == 0 || z < 2) return 1;
    if (tiles * std::min(z, cap) * 2 < cus) cap = std::max(nsb / 2, 1u);
    z = std::min(z, cap);
    return z < 2 ? 1 : ojh_gemm_sr_slices(K, z);
}
// Tokens from which that tile is taken whatever the form (measured with the rows streamed from HBM, K = 2048 .. 14336, before
// the form that has a CU to itself): the tile costs
// the same from 1 to 128 tokens, the matrix-core kernel below it doubles past 32 tokens.  So from 33 tokens; from 17
// where K is at least twice the row count (few tiles, each a long walk: 4096 x 14336 takes 38 us here against 45);
// and only from 65 for a matrix of more than one and a half 64-row tiles per CU, where two 32-token passes of the
// other kernel are still ahead (32000 x 4096 at 64 tokens: 56 us against 62).
static uint32_t q4k_xt_min_tokens(const ojh_device *dev, uint32_t K, uint32_t N) {
    if (dev->q4k_xt_min_m != 1) return dev->q4k_xt_min_m;
    const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
    if (2 * (uint64_t)((N + 63) / 64) > 3ull * cus) return 65;
    return K >= 2ull * N ? 17 : 33;
}
// The form that has a CU to itself multiplies no more than 64 tokens where no more are left, and is ahead from 17 of them,
// where the few-token kernels need a second pass of 16 (before / with it, 24 tokens, us: 14336 x 4096 22.6 / 20.7, 4096^2
// 16.7 / 12.4, 1024 x 4096 15.3 / 11.4, 4096 x 14336 35.2 / 22.3; at 12 tokens 17.7 / 20.4, 8.9 / 12.3, 8.5 / 11.4).  Not for
// short rows, where its fixed part shows (6000 x 1024 8.9 / 9.8, 4000 x 1792 10.0 / 10.4, 3500 x 2048 level, 2000 x 2048 10.9 / 9.9),
// unless more 64-row tiles than half the CUs make the few-token kernel walk two tiles a wave (8400 x 1024 11.1 / 8.6, x 2048
// 18.9 / 12.3).  Matrices of fewer rows than its slices fill half the CUs with (960 on 256) take it too, from 33 tokens also short
// ones, where the few-token kernel's row tiles leave more of them idle: 730 x 5632 at 22 tokens 20.8 / 12.4, at 64 43.9 / 12.9, 256 x 2048
// at 64 19.8 / 10.2, x 14336 at 64 105 / 17.3.  Up to 64 tokens, half a tile: more keep the sums' order of ojh_mm_noalloc, which has no
// scratch for slices.
static bool q4k_xk_early(const ojh_device *dev, uint32_t K, uint32_t N, uint32_t m) {
    const bool ahead = K > 2048 || (K == 2048 && N <= 2560) || (N + 63) / 64 * 2 > (uint32_t)dev->prop.multiProcessorCount;
    if (m > 64 && !q4k_xt_slices(dev, K, N, m)) return false;
    return (ahead || (m > 32 && K >= 1024)) && m >= 17 && dev->q4k_xt_min_m == 1 && q4k_xk_slices(dev, K, N, m);
}
// What a Q4_K product of m tokens does about that tile.  From q4k_xt_min_tokens it takes it (q4k_xt_must).  The few-token kernels need
// none of its scratch, so a product of fewer tokens, or of too few rows for that, takes it only where all of that is to be had (and
// takes none where some is not), which is asked for here, once a product.
enum { XT_ASK = -1, XT_NO, XT_TAKE, XT_SIDES };    // XT_SIDES: taken, its side arrays written by the quantizer
static bool q4k_xt_must(const ojh_device *dev, uint32_t K, uint32_t N, uint32_t m) {
    return m >= q4k_xt_min_tokens(dev, K, N) && q4k_xt_slices(dev, K, N, m);
}
static int q4k_xt_ready(ojh_device *dev, const ojh_lin *w, uint32_t m, const void *wp) {
    const uint32_t K = w->k, N = w->n;
    if (w->type != OJH_Q4_K || !dev->q4k_xt_min_m || dev->no_scratch || (uint64_t)m * K > 0xFFFFFFFFull ||
        (uint64_t)w->row_bytes * N > 0xFFFFFFFFull || (uintptr_t)wp % 16)
        return XT_NO;
    if (q4k_xt_must(dev, K, N, m)) return XT_TAKE;
    if (!q4k_xk_early(dev, K, N, m) || ensure(dev, "gemm_q8k")) return XT_NO;
    const size_t z = q4k_xk_slices(dev, K, N, m), mp = (m + 127) / 128 * 128, nsb = K / 256, tiles = (size_t)((N + 63) / 64) * (mp / 128);
    const size_t xst = nsb * mp * 4, sums = nsb * mp * 32, part = tiles * z * 32768, cnt = tiles * 4;
    ojh_buf *b;
    if (z == 1 ? !ojh_scratch_fits(dev, {{"xt_xst", xst}, {"xt_sums", sums}})
               : !ojh_scratch_fits(dev, {{"xt_xst", xst}, {"xt_sums", sums}, {"xt_part", part}, {"xt_cnt", cnt}}))
        return XT_NO;
    return (z == 1 || (!ojh_scratch_get_zeroed(dev, "xt_cnt", cnt, &b) && !ojh_scratch_spare(dev, "xt_part", part, &b))) &&
           !ojh_scratch_spare(dev, "xt_sums", sums, &b) && !ojh_scratch_spare(dev, "xt_xst", xst, &b) ? XT_TAKE : XT_NO;
}

static int xt_scratch(ojh_device *dev, const ojh_lin *w, uint32_t m, const char *name, size_t bytes, ojh_buf **out) {
    return q4k_xt_must(dev, w->k, w->n, m) ? ojh_scratch_get(dev, name, bytes, out) : ojh_scratch_spare(dev, name, bytes, out);
}

int ojh_mm_q8k_launch(ojh_device *dev, void *xq, void *xs, const ojh_lin *w, const ojh_block_format *f, void *yp,
                         const ojh_buf *bias, uint32_t m, int accum, int xt) {
    const uint32_t K = w->k, N = w->n;
    void *wp = at(w->raw, w->off);
    uint32_t grid[3] = {1, 1, 1}, block[3] = {256, 1, 1};
    std::string base = std::string("gemv_q8k_") + f->tag;
    // an output head: rows grid-stride, activations in registers
    if (m == 1 && w->type == OJH_Q6_K && dev->px && !accum && !bias && N >= 32768u && K <= 8192u) {
        uint32_t sg[3], sb[3];
        const std::string name = base + "_px";
        int rc = ojh_launch_shape(dev, name.c_str(), K, N, 1, sg, sb);
        if (rc) return rc;
        return ojh_launch(dev, name.c_str(), {xq, xs, wp, yp}, {K, N}, sg, sb);
    }
    if (m == 1) {
        int r = (accum || bias) ? 1 : pick_rows(dev, N);
        bool wide = !accum && !bias && r == 2 && N >= 32768u;
        std::string name = base + (accum ? "_accum" : bias ? "_bias" : wide ? "_wide" : r == 4 ? "" : r == 2 ? "_r2" : "_r1");
        grid[0] = (N + 4 * r - 1) / (4 * r);
        std::vector<void *> p = {xq, xs, wp, yp};
        if (bias) p.push_back(bias->ptr);
        return ojh_launch(dev, name.c_str(), p, {K, N}, grid, block);
    }
    // Q4_K rows against a prefill-sized batch: 128 x 128 tiles, the tokens copied into LDS by the memory system
    // (needs two side arrays, built by one small launch into the library's scratch — or by the quantizer itself when
    // ojh_mm quantizes: it then comes here with the side arrays ready)
    if (xt == XT_ASK) xt = q4k_xt_ready(dev, w, m, wp);
    if (xt != XT_NO) {
        int rc = ensure(dev, "gemm_q8k");
        if (rc) return rc;
        const uint32_t mp = (m + 127) / 128 * 128;
        const size_t nsb = K / 256;
        ojh_buf *xst, *sums;
        if ((rc = xt_scratch(dev, w, m, "xt_xst", nsb * mp * 4, &xst)) || (rc = xt_scratch(dev, w, m, "xt_sums", nsb * mp * 32, &sums))) return rc;
        uint32_t sg[3], sb[3];
        if (xt != XT_SIDES) {
            const char *sides = q4k_xk_slices(dev, K, N, m) ? "q8k_token_sides_h" : "q8k_token_sides";
            if ((rc = ojh_launch_shape(dev, sides, K, N, m, sg, sb))) return rc;
            if ((rc = ojh_launch(dev, sides, {xq, xs, xst->ptr, sums->ptr}, {K, m, mp}, sg, sb))) return rc;
        }
        // at most one 64-row tile per CU: the form that has a CU to itself, over K slices where that leaves CUs idle
        if (const uint32_t z = q4k_xk_slices(dev, K, N, m)) {
            const size_t tiles = (size_t)((N + 63) / 64) * (mp / 128);
            sg[0] = (N + 63) / 64; sg[1] = mp / 128; sg[2] = z;
            sb[0] = 512; sb[1] = sb[2] = 1;
            // fewer tokens may want more slices than these do, and a recorded call can ask for nothing: the places that the form
            // with two workgroups a CU would leave behind are asked for beside, where there is room
            if (const uint32_t zt = q4k_xt_slices(dev, K, N, m); zt > z && m >= q4k_xt_min_tokens(dev, K, N) && !dev->capturing) {
                ojh_buf *b;
                if (!ojh_scratch_spare(dev, "xt_part", tiles * zt * 32768, &b, true)) (void)ojh_scratch_get_zeroed(dev, "xt_cnt", tiles * 4, &b);
            }
            if (z == 1) return ojh_launch(dev, "gemm_q8k_q4k_xk64", {xq, xst->ptr, sums->ptr, wp, yp}, {K, N, m, (uint32_t)(accum != 0), mp}, sg, sb);
            ojh_buf *part, *cnt;
            if ((rc = xt_scratch(dev, w, m, "xt_part", tiles * z * 32768, &part))) return rc;
            if ((rc = ojh_scratch_get_zeroed(dev, "xt_cnt", tiles * 4, &cnt))) return rc;
            return ojh_launch(dev, "gemm_q8k_q4k_xk64_sr", {xq, xst->ptr, sums->ptr, wp, yp, part->ptr, cnt->ptr},
                              {K, N, m, (uint32_t)(accum != 0), mp, z}, sg, sb);
        }
        // too few 64-row tiles for the chip: K slices of them, summed in slice order by the last to finish
        if (const uint32_t z = q4k_xt_slices(dev, K, N, m); z > 1) {
            const size_t tiles = (size_t)((N + 63) / 64) * (mp / 128);
            ojh_buf *part, *cnt;
            if ((rc = ojh_scratch_get(dev, "xt_part", tiles * z * 32768, &part))) return rc;
            if ((rc = ojh_scratch_get_zeroed(dev, "xt_cnt", tiles * 4, &cnt))) return rc;
            sg[0] = (N + 63) / 64; sg[1] = mp / 128; sg[2] = z;
            sb[0] = 512; sb[1] = sb[2] = 1;
            return ojh_launch(dev, "gemm_q8k_q4k_xt64_sr", {xq, xst->ptr, sums->ptr, wp, yp, part->ptr, cnt->ptr},
                              {K, N, m, (uint32_t)(accum != 0), mp, z}, sg, sb);
        }
        // 128-row tiles when they give every CU one, 64-row tiles otherwise
        const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
        const char *tile = (uint64_t)((N + 127) / 128) * (mp / 128) >= cus && !dev->q4k_xt64 ? "gemm_q8k_q4k_xt" : "gemm_q8k_q4k_xt64";
        if ((rc = ojh_launch_shape(dev, tile, K, N, m, sg, sb))) return rc;
        return ojh_launch(dev, tile, {xq, xst->ptr, sums->ptr, wp, yp}, {K, N, m, (uint32_t)(accum != 0), mp}, sg, sb);
    }
    // Q4_K rows against several tokens: the int8 matrix cores, in the shape measured fastest on K = 4096 and 14336.
    // A long matrix (six 16-row tiles per CU and wave: 24576 rows on this GPU) against 2 .. 16 tokens: a wave
    // per tile, rows copied through LDS.
    if (w->type == OJH_Q4_K && dev->q4k_ml_min_m && m >= dev->q4k_ml_min_m && m <= 16 &&
        (N + 15) / 16 >= 6u * (uint32_t)dev->prop.multiProcessorCount && ojh_gemm_q8k_ml_lds(K) <= 163840 &&
        (uint64_t)w->row_bytes * N <= 0xFFFFFFFFull && (uintptr_t)wp % 16 == 0) {
        int rc = ensure(dev, "gemm_q8k");
        if (rc) return rc;
        uint32_t sg[3], sb[3];
        if ((rc = ojh_launch_shape(dev, "gemm_q8k_q4k_ml", K, N, m, sg, sb))) return rc;
        return ojh_launch(dev, "gemm_q8k_q4k_ml", {xq, xs, wp, yp}, {K, N, m, (uint32_t)(accum != 0)}, sg, sb);
    }
    // Few rows (up to a tile and a half per CU: 6144 rows) against 5 .. 16 tokens that fit LDS whole: a
    // workgroup per tile, its eight waves splitting K (a third faster than the general tiling at K = 14336).
    if (w->type == OJH_Q4_K && m >= dev->q4k_mf_min_m && m <= 16 && 2 * ((N + 15) / 16) <= 3u * (uint32_t)dev->prop.multiProcessorCount &&
        ojh_gemm_q8k_mk_lds(K, m) <= 163840 && (uintptr_t)wp % 16 == 0) {
        int rc = ensure(dev, "gemm_q8k");
        if (rc) return rc;
        uint32_t sg[3], sb[3];
        if ((rc = ojh_launch_shape(dev, "gemm_q8k_q4k_mk", K, N, m, sg, sb))) return rc;
        return ojh_launch(dev, "gemm_q8k_q4k_mk", {xq, xs, wp, yp}, {K, N, m, (uint32_t)(accum != 0)}, sg, sb);
    }
    // (from 5 tokens; from 3 on an output head, where the per-token loop of the dot kernel costs most)
    if (w->type == OJH_Q4_K && (m >= dev->q4k_mf_min_m || (m >= 3 && m + 2 >= dev->q4k_mf_min_m && N >= 32768u))) {
        int rc = ensure(dev, "gemm_q8k");
        if (rc) return rc;
        uint32_t sg[3], sb[3];
        if ((rc = ojh_launch_shape(dev, "gemm_q8k_q4k_mf", K, N, m, sg, sb))) return rc;
        uint32_t rw, rt;
        ojh_gemm_q8k_tiles(dev, K, N, m, &rw, &rt);
        return ojh_launch(dev, "gemm_q8k_q4k_mf", {xq, xs, wp, yp}, {K, N, m, (uint32_t)(accum != 0), rw, rt}, sg, sb);
    }
    const size_t w_bytes = w->row_bytes * N;
    const bool dwords_ok = (uintptr_t)wp % 4 == 0 && (w_bytes % 4 == 0 || w->off + w_bytes + 2 <= w->raw->bytes);
    // Q6_K / Q5_K rows against a batch: 128-row x 64-token tiles, scales folded into two int8 digits;
    // over K slices where the tiles alone would leave CUs idle (partial tiles in library scratch, added in slice order)
    // (from where it was measured ahead of what it replaces, rows streamed from HBM.  Q6_K: from 17 tokens on matrices of
    // more than 4096 rows or a longer K than that — 7168 x 2048 at 24 tokens 14.6 against 20.4 us for two launches of 16,
    // 730 x 5632 17.7 against 21.2, 14336 x 4096 24.2 against 39 — from 33 on the others, where two launches are level or
    // ahead (4096 x 4096: 18.2 against 17.8, 2048 x 1536 13.2 against 12.9).  Below 17 tokens Q6_K keeps the bits of
    // ojh_mm_noalloc, which has no scratch for K slices, also where 16 tokens no longer fit the few-row kernel (4096 x 14336
    // at 12 tokens: two launches of 8 take 33.4, the slices took 26.3).  Q5_K, whose few-token form is
    // the integer-dot kernel: from 5 tokens on large matrices (14336 x 4096 at 5 tokens 22.6, at 3 22.6 against 17.7 there),
    // from 9 on small ones (4096 x 4096 at 8 tokens 17.4 against 12.4, 730 x 5632 17.7 against 13.5).)
    // Below the second threshold a call takes the tile only where all it needs is to be had (a recorded call may ask for
    // nothing), and leaves its scratch to calls that cannot do without.
    const bool gs_large = N >= 8192 || K > 8192;
    const uint32_t gs_min = dev->kq_gs_min_m != 1 ? dev->kq_gs_min_m
                            : w->type == OJH_Q6_K ? (gs_large ? 17u : 33u) : (gs_large ? 5u : 9u);
    const uint32_t gs_early = dev->kq_gs_min_m != 1 || w->type != OJH_Q6_K || dev->no_scratch ? gs_min
                              : N > 4096 || K > 4096 ? 17u : 33u;
    if ((w->type == OJH_Q6_K || w->type == OJH_Q5_K) && gs_min && m >= gs_early && K % 256 == 0 &&
        (uintptr_t)xq % 16 == 0 && (w->type == OJH_Q6_K ? dwords_ok : (uintptr_t)wp % 16 == 0)) {
        int rc;
        const bool early = m < gs_min;
        const std::string gs = std::string("gemm_q8k_") + f->tag + "_gs";
        uint32_t sg[3] = {(N + 127) / 128, (m + 63) / 64, 1}, sb[3] = {256, 1, 1};
        const uint32_t z = dev->no_scratch ? 1 : ojh_gemm_q8k_gs_slices(dev, K, N, m);
        const size_t tiles = (size_t)sg[0] * sg[1], part_bytes = tiles * z * 32768, cnt_bytes = tiles * 4;
        const bool taken = !early || ((dev->modules.count("gemm_q8k") || !dev->capturing) &&
                                      (z < 2 || ojh_scratch_fits(dev, {{"gs_part", part_bytes}, {"gs_cnt", cnt_bytes}})));
        ojh_buf *part = nullptr, *cnt = nullptr;
        if (taken && z > 1) {
            rc = early ? ojh_scratch_spare(dev, "gs_part", part_bytes, &part) : ojh_scratch_get(dev, "gs_part", part_bytes, &part);
            if (!rc) rc = ojh_scratch_get_zeroed(dev, "gs_cnt", cnt_bytes, &cnt);
            if (rc && !early) return rc;
        }
        if (taken && (z < 2 || cnt)) {
            if ((rc = ensure(dev, "gemm_q8k"))) return rc;
            if (z < 2) return ojh_launch(dev, gs.c_str(), {xq, xs, wp, yp}, {K, N, m, (uint32_t)(accum != 0)}, sg, sb);
            sg[2] = z;
            return ojh_launch(dev, (gs + "_sr").c_str(), {xq, xs, wp, yp, part->ptr, cnt->ptr},
                              {K, N, m, (uint32_t)(accum != 0), z}, sg, sb);
        }
    }
    // Q6_K rows against 2 or more tokens on the int8 matrix cores (beyond 16 tokens as launches of 16 or 8:
    // each streams the rows once, which the per-token loop of the general entry does sixteen times
    // over).  Three shapes of the same tile arithmetic, picked by what was measured on K = 4096 and 14336:
    //   many rows (eight tiles per CU and wave, 32768 rows on this GPU): a wave per tile, rows copied
    //     through LDS, ahead of everything from 2 tokens;
    //   few rows (up to two tiles per CU, 8192 rows): a workgroup per tile, its waves splitting K, ahead of
    //     the integer-dot entry from 5 tokens (from 3 when K is long) and the only one that holds 8 tokens
    //     of K = 14336;
    //   between: a wave per tile with direct loads, ahead of the integer-dot entry from 5 tokens.
    if (w->type == OJH_Q6_K && m >= 2) {
        const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount, tiles = (N + 15) / 16;
        const uint32_t mc16 = m <= 8 ? m : 16;
        const bool ml_fits = dev->q6k_ml && (uint64_t)w_bytes <= 0xFFFFFFFFull && ojh_q6k_ml_lds(K, mc16) <= 163840 &&
                             (uintptr_t)wp % 16 == 0 && w->off + ((w_bytes + 15) & ~(size_t)15) <= w->raw->bytes;
        const bool mf_fits = dwords_ok && (uint64_t)(m <= 8 ? 8 : 16) * (K + 32) + K / 4 + 256 <= 69632;
        const bool mk16 = dwords_ok && ojh_q6k_mk_lds(K, mc16) <= 163840, mk8 = dwords_ok && ojh_q6k_mk_lds(K, 8) <= 163840;
        const bool mx_fits = m <= 16 && (uint64_t)m * ((K + 4095) / 4096) <= 19;
        const char *entry = nullptr;
        uint32_t step = 16;
        if (ml_fits && m >= dev->q6k_ml_min_m && tiles >= 8 * cus) {
            entry = "gemv_q8k_q6k_ml";
        } else if (tiles <= 2 * cus && (mk16 || mk8) && (m >= dev->q6k_mf_min_m || (m >= 3 && K > 8192) || !mx_fits)) {
            entry = "gemv_q8k_q6k_mk";
            step = mk16 ? 16 : 8;
        } else if (mf_fits && (m >= dev->q6k_mf_min_m || !mx_fits)) {
            entry = "gemv_q8k_q6k_mf";
        } else if (!mx_fits && (mk16 || mk8)) {
            entry = "gemv_q8k_q6k_mk";
            step = mk16 ? 16 : 8;
        } else if (!mx_fits && ml_fits) {
            entry = "gemv_q8k_q6k_ml";
        }
        if (entry) {
            const size_t nsb = K / 256;
            for (uint32_t t0 = 0; t0 < m; t0 += step) {
                const uint32_t mc = m - t0 < step ? m - t0 : step;
                uint32_t sg[3], sb[3];
                int rc = ojh_launch_shape(dev, entry, K, N, mc, sg, sb);
                if (rc) return rc;
                if ((rc = ojh_launch(dev, entry,
                                     {(char *)xq + (size_t)t0 * nsb * 256, (char *)xs + (size_t)t0 * nsb * 4, wp,
                                      (char *)yp + (size_t)t0 * N * 4},
                                     {K, N, mc, (uint32_t)(accum != 0)}, sg, sb)))
                    return rc;
            }
            return OJH_OK;
        }
    }
    // few tokens on Q6_K rows: activations staged in LDS once per workgroup, rows grid-stride
    if (w->type == OJH_Q6_K && m <= 16 && (uint64_t)m * ((K + 4095) / 4096) <= 19) {
        uint32_t sg[3], sb[3];
        int rc = ojh_launch_shape(dev, "gemv_q8k_q6k_mx", K, N, m, sg, sb);
        if (rc) return rc;
        return ojh_launch(dev, "gemv_q8k_q6k_mx", {xq, xs, wp, yp}, {K, N, m, (uint32_t)(accum != 0)}, sg, sb);
    }
    grid[0] = (N + 3) / 4;
    return ojh_launch(dev, (base + "_m").c_str(), {xq, xs, wp, yp}, {K, N, m, (uint32_t)(accum != 0)}, grid, block);
}

int ojh_mm_checks(const char *who, const ojh_lin *w, ojh_buf *y, size_t y_off, const ojh_buf *bias,
                            uint32_t m, int accum, const ojh_block_format **fmt) {
    if (!w) return ojh_fail(OJH_ERR_ARG, "%s: NULL weights", who);
    if (!m || m > 65535) return ojh_fail(OJH_ERR_ARG, "%s: m=%u out of range", who, m);
    const ojh_block_format *f = ojh_format(w->type);
    if (!f) return ojh_fail(OJH_ERR_UNSUPPORTED, "%s: GGUF type %u", who, w->type);
    if (bias && accum) return ojh_fail(OJH_ERR_UNSUPPORTED, "%s: bias and accum together", who);
    if (bias && m != 1) return ojh_fail(OJH_ERR_UNSUPPORTED, "%s: bias is a matvec (m=1) epilogue", who);
    int rc;
    if ((rc = span_ok("y", y, y_off, (size_t)m * w->n * 4, 4))) return rc;
    if (bias && (rc = span_ok("bias", bias, 0, (size_t)w->n * 4, 4))) return rc;
    if ((rc = span_ok("w", w->raw, w->off, w->row_bytes * w->n, ojh_block_align(f)))) return rc;
    *fmt = f;
    return OJH_OK;
}

extern "C" int ojh_mm_q8k(ojh_device *dev, const ojh_buf *xq, const ojh_buf *xscales, const ojh_lin *w, ojh_buf *y,
                          size_t y_off, const ojh_buf *bias, uint32_t m, int accum) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_mm_q8k: NULL device");
    const ojh_block_format *f;
    int rc = ojh_mm_checks("ojh_mm_q8k", w, y, y_off, bias, m, accum, &f);
    if (rc) return rc;
    if (ojh_float_rows(w->type))
        return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm_q8k: %s rows take f32 activations, as their CPU dot does", f->tag);
    size_t nsb = w->k / 256;
    if ((rc = span_ok("xq", xq, 0, (size_t)m * nsb * 256, 16))) return rc;
    if ((rc = span_ok("xscales", xscales, 0, (size_t)m * nsb * 4, 4))) return rc;
    if ((rc = ensure(dev, "gemv_q8k")) || (ojh_grid_type(w->type) && (rc = ensure(dev, "iq_grid")))) return rc;
    return ojh_mm_q8k_launch(dev, xq->ptr, xscales->ptr, w, f, at(y, y_off), bias, m, accum);
}

// Whether no two of a stage's outputs share a byte: otherwise its projections run one behind the other, as separate calls do.
static bool ys_apart(int count, const ojh_lin *const *ws, ojh_buf *const *ys, const size_t *y_offs) {
    for (int i = 1; i < count; i++)
        for (int j = 0; j < i; j++)
            if (overlap(at(ys[i], y_offs ? y_offs[i] : 0), (size_t)ws[i]->n * 4, at(ys[j], y_offs ? y_offs[j] : 0), (size_t)ws[j]->n * 4)) return false;
    return true;
}

extern "C" int ojh_mm_q8k_multi(ojh_device *dev, const ojh_buf *xq, const ojh_buf *xscales, int count,
                                const ojh_lin *const *ws, ojh_buf *const *ys, const size_t *y_offs) {
    if (!dev || !ws || !ys) return ojh_fail(OJH_ERR_ARG, "ojh_mm_q8k_multi: NULL argument");
    if (count < 1 || count > 4) return ojh_fail(OJH_ERR_ARG, "ojh_mm_q8k_multi: count=%d, takes 1 to 4 projections", count);
    int rc;
    bool grouped = true;
    uint64_t total = 0;
    for (int i = 0; i < count; i++) {
        const ojh_block_format *fi;
        if ((rc = ojh_mm_checks("ojh_mm_q8k_multi", ws[i], ys[i], y_offs ? y_offs[i] : 0, nullptr, 1, 0, &fi))) return rc;
        if (ojh_float_rows(ws[i]->type))
            return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm_q8k_multi: %s rows take f32 activations, as their CPU dot does", fi->tag);
        if (ws[i]->k != ws[0]->k)
            return ojh_fail(OJH_ERR_ARG, "ojh_mm_q8k_multi: projection %d has K=%u, the first has K=%u", i, ws[i]->k, ws[0]->k);
        if (ws[i]->type != OJH_Q4_K) grouped = false;
        total += ws[i]->n;
    }
    if (total > 0xFFFFFFFFull) return ojh_fail(OJH_ERR_ARG, "ojh_mm_q8k_multi: too many rows");
    size_t nsb = ws[0]->k / 256;
    if ((rc = span_ok("xq", xq, 0, nsb * 256, 16))) return rc;
    if ((rc = span_ok("xscales", xscales, 0, nsb * 4, 4))) return rc;
    if ((rc = ensure(dev, "gemv_q8k"))) return rc;
    for (int i = 0; i < count; i++)
        if (ojh_grid_type(ws[i]->type) && (rc = ensure(dev, "iq_grid"))) return rc;
    // a stage that mixes Q4_K, Q5_K and Q6_K tensors (a Q4_K_M file does): still one launch, every row in its own
    // format's arithmetic
    const bool apart = ys_apart(count, ws, ys, y_offs);
    bool kquants = count > 1 && apart;
    for (int i = 0; i < count; i++)
        if (ws[i]->type != OJH_Q4_K && ws[i]->type != OJH_Q5_K && ws[i]->type != OJH_Q6_K) kquants = false;
    if (!grouped && kquants) {
        std::vector<void *> p = {xq->ptr, xscales->ptr};
        uint32_t ends[4], run = 0, types = 0;
        for (int i = 0; i < 4; i++) {
            int j = i < count ? i : count - 1;
            p.push_back(at(ws[j]->raw, ws[j]->off));
            if (i < count) run += ws[i]->n;
            ends[i] = run;
            types |= ws[j]->type << (8 * i);
        }
        for (int i = 0; i < 4; i++) {
            int j = i < count ? i : count - 1;
            p.push_back(at(ys[j], y_offs ? y_offs[j] : 0));
        }
        uint32_t grid[3] = {(run + 3) / 4, 1, 1}, block[3] = {256, 1, 1};
        return ojh_launch(dev, "gemv_q8k_kq_x4", p, {ws[0]->k, ends[0], ends[1], ends[2], ends[3], types}, grid, block);
    }
    if (!grouped || count == 1 || !apart) {   // formats without a grouped entry, outputs over each other: one launch per projection
        for (int i = 0; i < count; i++) {
            const ojh_block_format *fi = ojh_format(ws[i]->type);
            if ((rc = ojh_mm_q8k_launch(dev, xq->ptr, xscales->ptr, ws[i], fi, at(ys[i], y_offs ? y_offs[i] : 0), nullptr, 1, 0)))
                return rc;
        }
        return OJH_OK;
    }
    std::vector<void *> p = {xq->ptr, xscales->ptr};
    uint32_t ends[4], run = 0;
    for (int i = 0; i < 4; i++) {
        int j = i < count ? i : count - 1;
        p.push_back(at(ws[j]->raw, ws[j]->off));
        if (i < count) run += ws[i]->n;
        ends[i] = run;
    }
    for (int i = 0; i < 4; i++) {
        int j = i < count ? i : count - 1;
        p.push_back(at(ys[j], y_offs ? y_offs[j] : 0));
    }
    int r = pick_rows(dev, run);
    if (r == 4) r = 2;
    uint32_t grid[3] = {(run + 4 * r - 1) / (4 * r), 1, 1}, block[3] = {256, 1, 1};
    return ojh_launch(dev, r == 2 ? "gemv_q8k_q4k_x4_r2" : "gemv_q8k_q4k_x4_r1", p,
                      {ws[0]->k, ends[0], ends[1], ends[2], ends[3]}, grid, block);
}

static bool fq_one_taken(const ojh_device *dev, const ojh_lin *w, const void *x, size_t x_bytes, const void *y);
static int fq_one_launch(ojh_device *dev, void *xp, int x_dtype, const ojh_lin *w, const ojh_block_format *f, void *yp, int accum);
static bool fq_one_alone(const ojh_device *dev, const ojh_lin *w);
// The token's codes and scales, as the two launches ask for them.
static int fq_scratch(ojh_device *dev, uint32_t K) {
    ojh_buf *b;
    int rc = ojh_scratch_get(dev, "xq", K, &b);
    return rc ? rc : ojh_scratch_get(dev, "xs", K / 64, &b);
}
// A recorded call of the two launches (more rows, or a bias) can ask for nothing: what they need is left behind by a call
// that takes one launch, some KB.
static void fq_leave_scratch(ojh_device *dev, uint32_t K) {
    ojh_buf *b;
    if (!dev->capturing && !ojh_scratch_spare(dev, "xq", K, &b, true)) (void)ojh_scratch_spare(dev, "xs", K / 64, &b, true);
}

// A workgroup's rows are one run of bytes, so workgroups lie `nrb` rows apart, and where that is close to a 128th above or below 512 KB
// or 1 MB their streams meet in the same channels: two rows more a workgroup then (us, as dealt / two more: Q4_K 26000 x 9216
// 33.3 / 27.9, 24000 x 9984 32.1 / 27.7, 52000 x 9216 56.0 / 51.3, Q5_K 38400 x 5120 34.3 / 30.4, Q6_K 23040 x 7168 35.1 / 33.2).  No
// such distance below 400 KB.
static uint32_t fq_rows_dealt(uint32_t nrb, uint32_t r, size_t row_bytes) {
    for (;; nrb += r) {
        const double apart = (double)nrb * (double)row_bytes;
        if (apart < 400e3) return nrb;
        const double off = std::fabs(apart / std::exp2(std::round(std::log2(apart))) - 1.0);
        if (std::fabs(off - 1.0 / 128) > 1.0 / 400) return nrb;
    }
}

// One stage of a decode layer in ONE launch: 1 to 4 projections of one f32 vector, the vector quantized inside the launch.
extern "C" int ojh_mm_multi(ojh_device *dev, const ojh_buf *x, size_t x_off, int count, const ojh_lin *const *ws,
                            ojh_buf *const *ys, const size_t *y_offs, int accum) {
    if (!dev || !ws || !ys) return ojh_fail(OJH_ERR_ARG, "ojh_mm_multi: NULL argument");
    if (count < 1 || count > 4) return ojh_fail(OJH_ERR_ARG, "ojh_mm_multi: count=%d, takes 1 to 4 projections", count);
    int rc;
    bool fused = true;
    uint64_t total = 0;
    for (int i = 0; i < count; i++) {
        const ojh_block_format *fi;
        if ((rc = ojh_mm_checks("ojh_mm_multi", ws[i], ys[i], y_offs ? y_offs[i] : 0, nullptr, 1, accum, &fi))) return rc;
        if (ojh_float_rows(ws[i]->type))
            return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm_multi: %s rows take f32 activations and need no quantizer: call ojh_mm", fi->tag);
        if (ws[i]->k != ws[0]->k)
            return ojh_fail(OJH_ERR_ARG, "ojh_mm_multi: projection %d has K=%u, the first has K=%u", i, ws[i]->k, ws[0]->k);
        if (ws[i]->type != OJH_Q4_K) fused = false;
        total += ws[i]->n;
    }
    if (total > 0xFFFFFFFFull) return ojh_fail(OJH_ERR_ARG, "ojh_mm_multi: too many rows");
    const uint32_t K = ws[0]->k;
    if ((rc = span_ok("ojh_mm_multi: x", x, x_off, (size_t)K * 4, 16))) return rc;
    if ((rc = ensure(dev, "gemv_q8k"))) return rc;
    for (int i = 0; i < count; i++)
        if (ojh_grid_type(ws[i]->type) && (rc = ensure(dev, "iq_grid"))) return rc;
    // The single launch against two (quantizer, matvec), us a stage in a recorded chain, weights from HBM: 6144 x 1024 5.7 / 4.5, 28672 x
    // 4096 15.7 / 14.8, 6144 x 8192 10.8 / 8.8, 4096 x 14336 11.2 / 10.1, 36000 x 5120 23.8 / 22.2, 65536 x 2048 17.4 / 16.7.  Beyond, the plain
    // matvec's thousands of small workgroups keep more bytes in flight: 49152 x 4096 23.0 / 23.1, x 8192 41.6 / 43.2, 65536 x
    // 4096 29.0 / 29.9; a long token for few rows is quantized too often: 600 x 14336 6.9 / 7.1.  Not where an output lies
    // over x: a workgroup may store its rows before another has read the token; nor where two lie over each other: they are
    // added to, or set, in order.  OJAS_HIP_FQ_MULTI = 0 never takes it, 2 at every size.
    const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
    const bool small_stage = total <= (uint64_t)(K <= 2048u ? 256u : 144u) * cus && (K <= 12288u || total >= 6ull * cus);
    // (the larger of these have two launches' scratch behind them all the same: a limit or a recording that has none refuses
    // them, and a recorded call that takes two launches finds it)
    const bool alone = total * K <= 32u * 1024u * 1024u && K <= 4096u;
    if (!ys_apart(count, ws, ys, y_offs)) fused = false;
    for (int i = 0; i < count; i++)
        if (overlap(at(x, x_off), (size_t)K * 4, at(ys[i], y_offs ? y_offs[i] : 0), (size_t)ws[i]->n * 4)) fused = false;
    if (count == 1 && !fused && dev->fq_multi && fq_one_taken(dev, ws[0], at(x, x_off), (size_t)K * 4, at(ys[0], y_offs ? y_offs[0] : 0)))
        return !fq_one_alone(dev, ws[0]) && (rc = fq_scratch(dev, K)) ? rc : fq_one_launch(dev, at(x, x_off), OJH_X_F32, ws[0], ojh_format(ws[0]->type), at(ys[0], y_offs ? y_offs[0] : 0), accum);
    if (!fused || K > 16384 || dev->fq_multi == 0 || (dev->fq_multi == 1 && !small_stage)) {   // quantize once, then the per-format launches
        size_t nsb = K / 256;
        ojh_buf *xq, *xs;
        if ((rc = ojh_scratch_get(dev, "xq", nsb * 256, &xq))) return rc;
        if ((rc = ojh_scratch_get(dev, "xs", nsb * 4, &xs))) return rc;
        if ((rc = ojh_quant_q8k_launch(dev, at(x, x_off), OJH_X_F32, 1, K, xq->ptr, xs->ptr))) return rc;
        if (!accum) return ojh_mm_q8k_multi(dev, xq, xs, count, ws, ys, y_offs);
        for (int i = 0; i < count; i++)
            if ((rc = ojh_mm_q8k_launch(dev, xq->ptr, xs->ptr, ws[i], ojh_format(ws[i]->type), at(ys[i], y_offs ? y_offs[i] : 0),
                                        nullptr, 1, 1)))
                return rc;
        return OJH_OK;
    }
    std::vector<void *> p = {at(x, x_off)};
    uint32_t ends[4], run = 0;
    for (int i = 0; i < 4; i++) {
        int j = i < count ? i : count - 1;
        p.push_back(at(ws[j]->raw, ws[j]->off));
        if (i < count) run += ws[i]->n;
        ends[i] = run;
    }
    for (int i = 0; i < 4; i++) {
        int j = i < count ? i : count - 1;
        p.push_back(at(ys[j], y_offs ? y_offs[j] : 0));
    }
    // Every workgroup repeats the quantization (as many vector instructions as the dots of some twenty rows), so the
    // launch takes few, large workgroups — `fq_blocks_per_cu` per CU, `fq_threads` threads each — and deals the rows
    // evenly between them.
    if (alone || dev->fq_multi == 2) fq_leave_scratch(dev, K);
    else if ((rc = fq_scratch(dev, K))) return rc;
    int r = dev->fq_rows ? dev->fq_rows : 2;
    uint32_t want = cus * dev->fq_multi_blocks;
    uint32_t nrb = (run + want - 1) / want;
    nrb = fq_rows_dealt((nrb + (uint32_t)r - 1) / (uint32_t)r * (uint32_t)r, (uint32_t)r, ws[0]->row_bytes);
    uint32_t grid[3] = {(run + nrb - 1) / nrb, 1, 1}, block[3] = {dev->fq_threads, 1, 1};
    return ojh_launch(dev, r == 2 ? "gemv_fq8k_q4k_x4_r2" : "gemv_fq8k_q4k_x4_r1", p,
                      {K, ends[0], ends[1], ends[2], ends[3], nrb, (uint32_t)(accum != 0)}, grid, block);
}

// A batch on plain f16 rows: the format's rows decoded into scratch and the activations converted in one launch, then the
// tile whose operands the memory system copies (`gemm_f16d_*`) — the same weights (dequant_to_f16's bits) and f16 activations
// as the tile that decodes on the way into LDS, sums in another order.  That tile's loaders fetch a row's block piecemeal,
// 64 weights a step (a 210-byte Q6_K block is touched in four cache lines four times over), and decode every weight once per
// 128 or 256 tokens; the pass reads and writes everything once.  Which is ahead is a matter of rounds of workgroups over the
// CUs more than of rows or tokens, so both are priced, in us: K steps on the busiest CU times what a step takes (a part
// that does not depend on how many CUs are busy, and one that grows with them), the atomics that K slices meet in, the
// pass.  The prices are fitted to 39000 timed calls (14 formats, 128 - 152064 rows, K 512 - 14336, 129 - 2048 tokens) with the
// copying tile on four waves: what they choose was on average within 0.8 % of the faster route, and 4 % or more behind the
// decoding tile in one call of 90 (by tokens and rows alone 1.7 %, and one of 40).  On eight waves that tile takes some 5 % less
// than it is priced at, so that near the line a call may stay with the decoding one.  Both routes measured then, decoding tile /
// pass + copying tile:
//   Q6_K   6914 x 2816 at 333 tokens 60 / 37, 14336 x 4096 at 130 79 / 71, 4096 x 4096 at 700 83 / 45
//   IQ4_NL 5330 x 11776 at 333 95 / 85, 8192 x 14336 at 333 162 / 215 (decoded rows beyond 112 MB: read back from memory)
//   Q5_0   8576 x 4096 at 257 106 / 51, MXFP4 8192 x 14336 at 512 188 / 249, Q4_1 8192 x 1024 at 512 26 / 32
static uint32_t f16d_tile(const ojh_device *dev, uint32_t N, uint32_t m) {   // 0: 128 x 128, 1: 256 x 128, 2: 256 x 256 tokens x rows
    // rounds of workgroups over the chip times a K step of the tile, fitted over 6650 timed calls with all three on four waves
    // (launch, decode pass and stores apart: 0.49 / 0.83 / 1.37 us with every CU busy; within 0.13 % of the fastest of the three on
    // average): 14336 x 4096 at 512 tokens 108 / 100 / 122 us, at 2048 308 / 294 / 262; 4096 x 14336 at 2048 334 / 279 / 388; 6914 x
    // 2816 at 333 35 / 51 / 76.  Where the first two run on eight waves (f16d_eight_waves) they take 6 - 8 % less, which these
    // weights do not know
    const uint64_t cus = (uint64_t)dev->prop.multiProcessorCount;
    auto rounds = [&](uint32_t bm, uint32_t bn) { return ((uint64_t)((N + bn - 1) / bn) * ((m + bm - 1) / bm) + cus - 1) / cus; };
    if (dev->f16d_tile > 0) return (uint32_t)dev->f16d_tile - 1u;
    const uint64_t c1 = 8 * rounds(128, 128), c2 = 13 * rounds(256, 128), c3 = 23 * rounds(256, 256);
    return c3 <= c1 && c3 <= c2 ? 2u : c2 < c1 ? 1u : 0u;
}
// Whether that tile (0 or 1) runs on eight waves, which pay for their sums' meeting by filling each other's gaps.  Whole calls on four
// / eight, mean and worst of random ones beyond 256 tokens: 128 x 128 from K = 2304 0.96 / 0.98 in one round of workgroups over the CUs
// as in several, below that 1.00 - 1.03 / 1.08 in several; 256 x 128 in one round 0.94 / 1.03 from K = 1024, in several 1.04 / 1.10 at
// K = 1024, 1.00 / 1.03 at 1280, 0.95 - 0.98 / 1.02 from 1536.  Up to 256 tokens a row of weights meets two tiles or one, and what
// fetches it bounds: 0.96 / 1.05 up to three quarters of the CUs (128 x 128; 256 x 128 where the decoded rows stay in the caches, 0.93 -
// 0.95), 1.01 - 1.08 / 1.11 otherwise.  us: Q8_0 4096 x 2816 at 1900 tokens 57.2 / 54.1, Q6_K 9500 x 8192 at 200 101 / 96, IQ3_XXS 23484 x
// 7936 at 251 252 / 277, IQ4_NL 26621 x 1024 at 1241 116 / 126.
static bool f16d_eight_waves(const ojh_device *dev, uint32_t N, uint32_t K, uint32_t m, uint32_t tile) {
    const uint64_t cus = (uint64_t)dev->prop.multiProcessorCount, bm = tile ? 256 : 128, tiles = (uint64_t)((N + 127) / 128) * ((m + bm - 1) / bm);
    if (tile ? K < 1536 && tiles > cus : K < 2304) return false;
    return m > 256 || (4 * tiles <= 3 * cus && (!tile || (uint64_t)N * K <= 56u << 20));
}
// whether the tile that decodes on the way into LDS is 128 tokens tall instead of 256
static bool gemm_mm_m128(const ojh_device *dev, uint32_t N, uint32_t m, bool decoded) {
    const uint64_t t256 = (uint64_t)((N + 127) / 128) * ((m + 255) / 256);
    return dev->gemm_m128 && (m <= (uint32_t)dev->gemm_m128 || 2 * t256 <= (uint32_t)dev->prop.multiProcessorCount || decoded);
}
static bool f16d_pays(const ojh_device *dev, const ojh_lin *w, uint32_t m, bool decoded) {
    const uint32_t K = w->k, N = w->n;
    const double cus = dev->prop.multiProcessorCount, mi = (double)N * K / (1 << 20);
    auto walk = [&](uint32_t bm, uint32_t bn, uint32_t most, double round, double fill) {
        const uint64_t tiles = (uint64_t)((N + bn - 1) / bn) * ((m + bm - 1) / bm);
        const uint32_t z = dev->gemm_sr ? 1u : ojh_gemm_slices(dev, tiles, most);
        const double per_cu = tiles * z / cus;
        return (K / 64 + z - 1) / z * (round * ceil(per_cu) + fill * per_cu) + (z > 1 ? 2.2 * z * m * N / (1 << 20) : 0.0);
    };
    const uint32_t tile = f16d_tile(dev, N, m);
    const double copied = tile == 2 ? 2.75 + walk(256, 256, 1, 1.14, 0.15) : tile == 1 ? 4.0 + walk(256, 128, 1, 0.66, 0.15)
                                                                                   : 0.75 + walk(128, 128, K / 512, 0.28, 0.19);
    // (a format that is decoded first in any case: the same pass, conversion included only where its decoder does that)
    if (decoded) return copied < (ojh_grid_type(w->type) ? 0.75 : 2.75) + walk(128, 128, K / 256, 0.40, 0.20);
    // a K step of 128 x 128 and of 256 x 128 on the loader
    double s128 = 0.76, s256 = 1.16;
    switch (w->type) {
    case OJH_IQ4_NL: case OJH_Q4_0: case OJH_Q8_0: s128 = 0.74; s256 = 1.10; break;
    case OJH_Q4_1: s128 = 0.82; s256 = 1.27; break;
    case OJH_Q5_0: case OJH_Q6_K: s128 = 1.00; s256 = 1.47; break;
    default: break;
    }
    const double loaded = gemm_mm_m128(dev, N, m, false) ? walk(128, 128, K / 256, s128, 0.0) : 3.5 + walk(256, 128, K / 256, s256, 0.0);
    return 0.42 * mi + (mi > 56 ? 0.5 * (mi - 56) : 0.0) + copied < loaded;
}
// Q4_K rows have tiles that dequantize straight into the matrix operand, far cheaper loaders than the other formats': decoding
// first pays where those tiles leave CUs idle or K slices have to meet through atomics, mostly below 3000 rows, and where a
// long K amortizes the pass.  Both priced as above, the terms fitted to 3031 pairs of timed calls (512 - 32768 rows, K 1024 -
// 14336, 200 - 2048 tokens; median error 2 - 5 %), and taken where ahead by a twentieth: 652 of the pairs, on average 16 %
// faster, six of them more than 3 % slower.  Tiles / pass + copying tile, us: 1088 x 2304 at 1944 tokens 39.8 / 26.9, 2752 x
// 6912 at 768 78.7 / 54.7, 4096 x 4096 at 1024 56.7 / 49.4, 6914 x 2816 at 333 39.2 / 33.1;
// kept: 14336 x 4096 at 512 70 / 93, at 2048 235 / 255, 28534 x 12288 at 241 202 / 427.  The pass forms the tiles' weights
// (dequant_q4kl_f16_x: f16 q qa + qb).
// Not beyond K = 8192: what the pass wrote has to come from the caches, and in the first call after other work it does not.
// Repeated / first call, us: 4096 x 14336 at 2048 263 -> 250 / 282 -> 294, at 1536 218 -> 210 / 221 -> 275, at 1024 150 -> 158 / 164 -> 192,
// 4096 x 11008 at 1024 120 -> 125 / 135 -> 135; against 4096 x 8192 at 2048 178 -> 150 / 197 -> 160, at 1024 93 -> 87 / 110 -> 107, 2048 x
// 8192 at 1536 86 -> 74 / 101 -> 90.
static bool f16d_pays_q4k(const ojh_device *dev, uint32_t N, uint32_t K, uint32_t m) {
    const double cus = dev->prop.multiProcessorCount, mi = (double)N * K / (1 << 20), mk = (double)m * K / (1 << 20), mn = (double)m * N / (1 << 20);
    struct Price { double fixed, acts, round, fill, meet, out, start; };
    auto price = [&](uint32_t bm, uint32_t bn, uint32_t most, const Price &p) {
        const uint64_t tiles = (uint64_t)((N + bn - 1) / bn) * ((m + bm - 1) / bm);
        const uint32_t z = most ? ojh_gemm_slices(dev, tiles, most) : 1u;
        const double per_cu = tiles * z / cus, steps = (K / 64 + z - 1) / z;
        return p.fixed + p.acts * mk + steps * (p.round * ceil(per_cu) + p.fill * per_cu) + (z > 1 ? p.meet * z * mn : 0.0) + p.out * mn + p.start * ceil(per_cu);
    };
    const double over = mi > 56 ? mi - 56 : 0.0;
    const uint32_t tile = f16d_tile(dev, N, m);
    const double copied = tile == 2   ? 0.345 * mi + 0.481 * over + price(256, 256, 0, {2.2, 0.24, 0.827, 0.802, 0.0, 0.50, 8.9})
                          : tile == 1 ? 0.263 * mi + 0.735 * over + price(256, 128, 0, {6.5, 0.06, 0.306, 0.547, 0.0, 0.68, 5.8})
                                      : 0.422 * mi + 0.684 * over + price(128, 128, K / 512, {7.5, 0.77, 0.173, 0.218, 3.59, 1.92, 0.35});
    // the tile that ojh_mm takes otherwise (1024 <= K <= 8192 here)
    const uint64_t t256 = (uint64_t)((N + 255) / 256) * ((m + 255) / 256), t128 = (uint64_t)((N + 255) / 256) * ((m + 127) / 128);
    const uint32_t z128 = (uint32_t)((uint64_t)cus / t128);
    const bool tall = t256 >= (uint64_t)cus || (2 * t256 >= (uint64_t)cus && K >= 8192);
    const double loaded = !tall && z128 >= 2 ? price(128, 64, K / 1024, {4.4, 1.26, 0.215, 0.037, 3.01, 1.33, 4.7})
                          : tall ? price(256, 256, K / 256, {5.3, 0.64, 1.059, 0.683, 2.29, 0.39, 5.2})
                                 : price(128, 256, K / 256, {11.4, 0.75, 0.436, 0.509, 2.24, 0.15, 0.0});
    return 1.05 * copied < loaded;
}
static bool f16d_taken(const ojh_device *dev, const ojh_lin *w, uint32_t m, int act_mode, bool decoded) {
    const bool q4kl = w->type == OJH_Q4_K && !dev->gemm_exact && act_mode != OJH_ACT_FLOAT_EXACT;   // (tiles of its own, other weight bits)
    if (!dev->deq_big_m || dev->no_scratch || dev->gemm_split_override || (uint64_t)w->n * w->k > 0x7FFFFFFFull) return false;
    if (q4kl && (dev->deq_big_m != 1 || dev->gemm_bdk != 1 || dev->gemm_sr || m < 257 || w->n < 512 || w->k < 1024 || w->k > 8192 || !f16d_pays_q4k(dev, w->n, w->k, m))) return false;
    // while a graph is recorded nothing can be loaded or grown: what is not there yet leaves the call on the tile it has
    if (dev->capturing) {
        const auto slot = dev->scratch.find("wdeq");
        if (!dev->modules.count("gemm_f16") || !dev->modules.count(ojh_grid_type(w->type) ? "iq_grid" : "dequant") ||
            slot == dev->scratch.end() || !slot->second || slot->second->bytes < (size_t)w->n * w->k * 2)
            return false;
    }
    if (dev->deq_big_m > 1 && !decoded) {   // asked for: Q6_K and, from twice as many tokens, Q5_K / Q8_0 rows of large matrices
        const bool kq = w->type == OJH_Q6_K || w->type == OJH_Q5_K || w->type == OJH_Q8_0;
        if (w->type == OJH_Q4_K || (kq && (uint64_t)w->n * w->k < (32ull << 20))) return false;
        return m >= (w->type == OJH_Q5_K || w->type == OJH_Q8_0 ? 2 * dev->deq_big_m : dev->deq_big_m);
    }
    if (q4kl) return true;                                     // (priced above)
    // (129 to 256 tokens are two tiles of 128, the second part empty: the two routes are within the prices' error of each
    // other there for the lighter loaders, whose rows then need no scratch)
    return m >= (decoded || w->type == OJH_Q6_K ? 129u : 257u) && f16d_pays(dev, w, m, decoded);
}
// Whether all the route needs is there.  What every form of the call needs comes first, so that the decoded rows' scratch,
// which a format with a loader can do without, never takes its room: the activations' scratch, and the family of the tiles
// that a recorded call of fewer tokens, or one that finds no room for its decoded rows, would take (nothing can be loaded then).
static int f16d_ready(ojh_device *dev, const ojh_lin *w, uint32_t m, bool decoded, bool q4kl, bool *ready) {
    int rc;
    ojh_buf *b;
    *ready = false;
    if ((rc = ensure(dev, "glue")) || (!dev->capturing && (rc = ensure(dev, q4kl ? "gemm_xl" : "gemm")))) return rc;
    if ((rc = ojh_scratch_get(dev, "xh", (size_t)m * w->k * 2, &b))) return rc;
    *ready = !ensure(dev, ojh_grid_type(w->type) ? "iq_grid" : "dequant") && !ensure(dev, "gemm_f16") &&
             !(decoded ? ojh_scratch_get(dev, "wdeq", (size_t)w->n * w->k * 2, &b) : ojh_scratch_spare(dev, "wdeq", (size_t)w->n * w->k * 2, &b));
    return OJH_OK;
}
static int f16d_launch(ojh_device *dev, void *xp, int x_dtype, const ojh_lin *w, const ojh_block_format *f, void *yp, uint32_t m,
                       int accum, bool q4kl) {
    const uint32_t K = w->k, N = w->n, tile = f16d_tile(dev, N, m);
    const bool grid_fmt = ojh_grid_type(w->type);
    int rc;
    ojh_buf *xh, *wdeq;
    if ((rc = ojh_scratch_get(dev, "xh", (size_t)m * K * 2, &xh))) return rc;
    if ((rc = ojh_scratch_spare(dev, "wdeq", (size_t)N * K * 2, &wdeq))) return rc;   // (there: f16d_ready)
    const bool kw = f16d_eight_waves(dev, N, K, m, tile);
    const char *name = tile == 2 ? "gemm_f16d_256" : tile == 1 ? (kw ? "gemm_f16d_256x128_kw" : "gemm_f16d_256x128") : kw ? "gemm_f16d_128_kw" : "gemm_f16d_128";
    uint32_t sg[3], sb[3];
    bool sk = false;
    if (!tile) {
        if ((rc = ojh_launch_shape(dev, "gemm_f16d_128_sk", K, N, m, sg, sb))) return rc;
        sk = sg[1] > 1 && !dev->gemm_sr;
        if (sk) name = "gemm_f16d_128_sk";
    }
    if (!sk && (rc = ojh_launch_shape(dev, name, K, N, m, sg, sb))) return rc;
    const uint32_t n_el = m * K, nz = sk && !accum ? m * N : 0, nb = (uint32_t)((uint64_t)N * K / f->weights);
    const uint32_t cb = (uint32_t)(((uint64_t)n_el / 8 + nz / 4 + 255) / 256 + 1);
    uint32_t dg[3], db[3];
    const std::string dq = std::string("dequant_") + f->tag + (q4kl ? "l_f16" : "_f16");
    if (!grid_fmt) {
        if ((rc = ojh_launch_shape(dev, (dq + "_x").c_str(), cb, nb, 0, dg, db))) return rc;
        if ((rc = ojh_launch(dev, (dq + "_x").c_str(), {at(w->raw, w->off), wdeq->ptr, xp, xh->ptr, yp},
                             {nb, n_el, nz, cb, (uint32_t)(x_dtype == OJH_X_BF16)}, dg, db)))
            return rc;
    } else {
        // (their decoders convert nothing beside: activations and zero fill in one launch; in two, 512 x 1024 at 130 tokens
        // took 14 us instead of 12)
        const uint32_t conv_blocks = (n_el / 8 + 255) / 256 + 1;
        uint32_t block[3] = {256, 1, 1}, cg[3] = {nz ? conv_blocks + (nz / 4 + 255) / 256 + 1 : conv_blocks, 1, 1};
        const std::string copy = std::string(x_dtype == OJH_X_BF16 ? "copy_bf16_half" : "copy_f32_half");
        if ((rc = ojh_launch_shape(dev, dq.c_str(), 0, nb, 0, dg, db))) return rc;
        if ((rc = ojh_launch(dev, dq.c_str(), {at(w->raw, w->off), wdeq->ptr}, {nb}, dg, db))) return rc;
        if ((rc = nz ? ojh_launch(dev, (copy + "_zero").c_str(), {xp, xh->ptr, yp}, {n_el, nz, conv_blocks}, cg, block)
                     : ojh_launch(dev, copy.c_str(), {xp, xh->ptr}, {n_el}, cg, block)))
            return rc;
    }
    if (sk) return ojh_launch(dev, name, {xh->ptr, wdeq->ptr, yp}, {K, N, m, sg[1]}, sg, sb);
    return ojh_launch(dev, name, {xh->ptr, wdeq->ptr, yp}, {K, N, (uint32_t)(accum != 0), m}, sg, sb);
}

// One K-quant projection of one token: quantizer and matvec in one launch.  Two launches / one, call to call, us:
//   Q5_K   600 x 4096 5.7 / 4.8, 4096^2 6.8 / 6.0, 9000 x 4096 11.4 / 10.1, 30000 x 8192 42.1 / 34.5, 128256 x 2560 66.9 / 58.0: everywhere
//   Q4_K   1024 x 4096 5.8 / 4.3, 9000 x 5120 10.8 / 9.6, 5300 x 14336 15.0 / 12.3, 30000 x 4096 16.3 / 16.0; output heads have a form of their
//          own that keeps more bytes in flight, so from 32768 rows only a short K: 65536 x 1792 16.8 / 15.8, x 4096 29.1 / 30.9
//   Q6_K   four lanes take a super-block, sixteen super-blocks a step.  Up to sixteen rows a CU, one a wave: 4096^2 7.7 / 6.4, 4096 x 11008
//          14.2 / 12.2, 2500 x 14336 13.5 / 11.5, but 1024 x 14336 8.4 / 8.9.  Beyond, the waves take pairs of rows.  Four units a wave
//          (gemv_fq8k_ring) are ahead, 12000 x 5120 17.4 / 16.6, 30000 x 9984 62.5 / 56.7, 50000 x 1024 31.3 / 19.2 (output heads have a form
//          of their own, a step of which is mostly idle at a short K), but not where one step is full, 30000 x 4096 25.6 / 25.8, 50000 x
//          4096 36.5 / 39.0.  Fewer: from 28 rows a CU, where fewer would leave waves without a pair, and rows of fifteen super-blocks,
//          7500 x 3840 9.7 / 9.5, x 5120 13.7 / 13.4, not 7500 x 3072 9.2 / 9.3; from 500 super-blocks a CU with less, 5300 x 6144 12.1 / 11.7,
//          4608 x 9984 15.5 / 15.1, not 6144 x 5120 11.6 / 11.9; one step up to 64, 16000 x 4096 level, 24000 x 4096 21.2 / 21.5.
// Not where y lies over x: a workgroup may store its rows before another has read the token.
static bool fq_one_taken(const ojh_device *dev, const ojh_lin *w, const void *x, size_t x_bytes, const void *y) {
    const uint32_t K = w->k, N = w->n, cus = (uint32_t)dev->prop.multiProcessorCount;
    if ((w->type != OJH_Q4_K && w->type != OJH_Q5_K && w->type != OJH_Q6_K) || overlap(x, x_bytes, y, (size_t)N * 4) || K > 16384u) return false;
    if (dev->fq_one != 1) return dev->fq_one == 2;
    if (w->type == OJH_Q4_K) return (N < 32768u || K <= 2048u) && (K <= 12288u || N >= 5u * cus);
    if (w->type == OJH_Q5_K) return K <= 8192u || N >= (K <= 12288u ? 5u : 16u) * cus;
    const uint32_t nsb = K / 256, steps = (nsb + 15) / 16, nrb = (N + cus - 1) / cus;
    if (nrb <= 16u) return K <= 8192u || nrb >= 5u;
    if ((nrb + 31) / 32 * steps >= 4u) return steps > 1 || nsb <= 12;
    return nsb >= 15 && (nrb >= 28u ? steps > 1 || nrb <= 64u : nrb * nsb >= 500u);
}
// Those that need nothing but themselves; the others ask for the two launches' scratch although they do without, so what a limit on
// scratch or a recording refuses does not depend on the route, and a recorded call that takes two launches finds it.
static bool fq_one_alone(const ojh_device *dev, const ojh_lin *w) {
    const uint32_t K = w->k, mi = (uint32_t)(((uint64_t)w->n * K + (1u << 20) - 1) >> 20);
    if (dev->fq_one == 2) return true;
    if (w->n >= 32768u || K > 8192u) return false;
    if (w->type != OJH_Q6_K && K <= 4096u) return mi <= (w->type == OJH_Q5_K ? 56u : 32u);
    if (w->n > 16u * (uint32_t)dev->prop.multiProcessorCount) return false;
    return mi <= (w->type == OJH_Q6_K ? (K <= 4096u ? 16u : 8u) : w->type == OJH_Q4_K ? 18u : K <= 6144u ? 14u : 8u);
}
static int fq_one_launch(ojh_device *dev, void *xp, int x_dtype, const ojh_lin *w, const ojh_block_format *f, void *yp, int accum) {
    const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
    // A workgroup of sixteen waves per CU; two rows a wave where it has more than one, and where a row alone is several steps (us,
    // one row a wave / two: Q4_K 1024 x 2560 4.5 / 4.8, x 8192 5.9 / 5.6, x 14336 7.9 / 7.3, Q5_K 1500 x 8192 6.2 / 6.9, x 14336 10.2 / 9.2)
    uint32_t nrb = (w->n + cus - 1) / cus;
    const bool steps = w->type == OJH_Q4_K ? w->k >= 8192u : w->type == OJH_Q5_K && w->k > 8192u && w->n >= 5u * cus;
    const uint32_t r = dev->fq_rows ? (uint32_t)dev->fq_rows : nrb > 16 || steps ? 2 : 1;
    nrb = fq_rows_dealt((nrb + r - 1) / r * r, r, w->row_bytes);
    const uint32_t grid[3] = {(w->n + nrb - 1) / nrb, 1, 1}, block[3] = {1024, 1, 1};
    const std::string name = std::string("gemv_fq8k_") + f->tag + (x_dtype == OJH_X_BF16 ? "_one_bf16_r" : "_one_r") + (r == 2 ? "2" : "1");
    int rc = ensure(dev, "gemv_q8k");
    fq_leave_scratch(dev, w->k);
    return rc ? rc : ojh_launch(dev, name.c_str(), {xp, at(w->raw, w->off), yp}, {w->k, w->n, nrb, (uint32_t)(accum != 0)}, grid, block);
}

extern "C" int ojh_mm(ojh_device *dev, const ojh_buf *x, size_t x_off, int x_dtype, const ojh_lin *w, ojh_buf *y,
                      size_t y_off, const ojh_buf *bias, uint32_t m, int accum, int act_mode) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_mm: NULL device");
    const ojh_block_format *f;
    int rc = ojh_mm_checks("ojh_mm", w, y, y_off, bias, m, accum, &f);
    if (rc) return rc;
    if (x_dtype != OJH_X_F32 && x_dtype != OJH_X_BF16)
        return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm: activations must be f32 or bf16");
    const uint32_t K = w->k, N = w->n;
    size_t esz = x_dtype == OJH_X_BF16 ? 2 : 4;
    if ((rc = span_ok("ojh_mm: x", x, x_off, (size_t)m * K * esz, 16))) return rc;

    void *wp = at(w->raw, w->off), *yp = at(y, y_off);
    uint32_t grid[3] = {1, 1, 1}, block[3] = {256, 1, 1};

    // Q8_0 rows on the reference GPU decode path's arithmetic: activations quantized per 32 (quantize_q8_1), integer
    // dots against the blocks as the file stores them (crates/ojas-cuda/src/kernels/gemv_q8.rs:152-215), token by token.
    if (act_mode == OJH_ACT_Q8_1) {
        if (w->type != OJH_Q8_0) return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm: OJH_ACT_Q8_1 serves Q8_0 rows, not %s", f->tag);
        if (x_dtype != OJH_X_F32) return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm: OJH_ACT_Q8_1 takes f32 activations");
        if ((rc = ensure(dev, "q80_dp4a"))) return rc;
        const size_t nblk = K / 32;
        ojh_buf *q8, *d8, *d8s;
        if ((rc = ojh_scratch_get(dev, "q81_q", (size_t)m * K, &q8))) return rc;
        if ((rc = ojh_scratch_get(dev, "q81_d", (size_t)m * nblk * 4, &d8))) return rc;
        if ((rc = ojh_scratch_get(dev, "q81_s", (size_t)m * nblk * 4, &d8s))) return rc;
        const char *name = accum ? "gemv_q80_dp4a_accum" : bias ? "gemv_q80_dp4a_bias" : "gemv_q80_dp4a";
        if (accum && bias) return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm: OJH_ACT_Q8_1 adds a bias or accumulates, not both");
        uint32_t qg[3] = {(K + 255) / 256, 1, 1}, gg[3] = {(N + 7) / 8, 1, 1};
        for (uint32_t t = 0; t < m; t++) {
            void *tq = (char *)q8->ptr + (size_t)t * K, *td = (char *)d8->ptr + (size_t)t * nblk * 4;
            if ((rc = ojh_launch(dev, "quantize_q8_1", {(char *)at(x, x_off) + (size_t)t * K * 4, tq, td, (char *)d8s->ptr + (size_t)t * nblk * 4},
                                 {K}, qg, block)))
                return rc;
            std::vector<void *> p = {wp, tq, td, (char *)yp + (size_t)t * N * 4};
            if (bias && !accum) p.push_back(bias->ptr);
            if ((rc = ojh_launch(dev, name, p, {K, N}, gg, block))) return rc;
        }
        return OJH_OK;
    }

    // Q5_K: the CPU path's arithmetic (dot_q5k over int8 activations) unless floating-point activations are
    // asked for, which run on the f32-activation matvecs; from the tile crossover both that request and
    // OJH_ACT_AUTO take the f16 tile (dequant_to_f16 bits), as Q6_K and Q8_0 do.
    // Where OJH_ACT_AUTO hands over from the int8 kernels to the f16 tile: 32 tokens (OJAS_HIP_GEMM_MIN_M); for Q6_K and
    // Q5_K rows later — their int8 tile is ahead of their f16 tile up to 128 / 64 tokens (measured, 14336 x 4096 at 64
    // tokens: Q6_K 34.5 against 45.9 us, Q5_K 31.9 against 38.7; a 151936-row head at 32 tokens 164 against 341).
    uint32_t tile_min = dev->gemm_min_m;
    if (act_mode == OJH_ACT_AUTO && dev->kq_gs_min_m && K % 256 == 0 && (w->type == OJH_Q6_K || w->type == OJH_Q5_K)) {
        const uint32_t later = w->type == OJH_Q6_K ? 129u : 65u;
        if (tile_min < later) tile_min = later;
    }
    // Q8_0 rows have no few-token kernel on the matrix cores: their f32-activation matvec walks the rows once per token
    // (14336 x 4096 at 8 tokens 84 us, a 128256-row head 810), and the 128-token f16 tile — the contract the reference's
    // own GPU path switches to from 8 rows (crates/ojas-models/src/decoder/dispatch.rs:70-75) — takes 38 and 251: under
    // OJH_ACT_AUTO from 4 tokens on large matrices, 6 on small ones (4096 x 4096: 12.3 against 17.0 at 4, 21.4 at 8).
    if (act_mode == OJH_ACT_AUTO && w->type == OJH_Q8_0 && dev->q80_tile_min_m) {
        const uint32_t early = dev->q80_tile_min_m != 1 ? dev->q80_tile_min_m : (uint64_t)N * K >= (32ull << 20) ? 4u : 6u;
        if (tile_min > early) tile_min = early;
    }
    const bool q5_tile = w->type == OJH_Q5_K && act_mode != OJH_ACT_Q8K && m >= tile_min && K % 64 == 0 &&
                         (uint64_t)m * K < 0x7FFFFFFFull && (uint64_t)m * N < 0x7FFFFFFFull;
    const bool q5_float = w->type == OJH_Q5_K && !q5_tile && (act_mode == OJH_ACT_FLOAT || act_mode == OJH_ACT_FLOAT_EXACT);
    if (w->type == OJH_Q5_K && !q5_float && !q5_tile) act_mode = OJH_ACT_Q8K;

    // IQ4_NL / IQ4_XS (dot_iq4nl / dot_iq4xs), Q4_0 / Q4_1 / Q5_0 / Q5_1 and Q2_K / Q3_K: f32 activations against the raw
    // rows at every token count; no int8-activation form and no MFMA tile read them.
    // The grid-codebook formats likewise have no MFMA tile; IQ2_XXS and IQ3_XXS take int8 activations unless f32
    // ones are asked for (dot_iq2xxs_q8k / dot_iq3xxs_q8k under matvec_kq, dot_iq2xxs / dot_iq3xxs under dot_iq).
    const bool grid_fmt = ojh_grid_type(w->type);
    const bool iq4 = ojh_float_only(w->type) || q5_float;   // (the IQ4 types, the legacy 32-weight blocks, Q2_K, Q3_K, ...)
    if (iq4 && act_mode == OJH_ACT_Q8K)
        return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm: %s rows take f32 activations only (OJH_ACT_FLOAT or OJH_ACT_AUTO)", f->tag);

    // Above the crossover the MFMA tile wins over streaming the weights once per few tokens
    // (the reference switches at 8 rows, crates/ojas-models/src/decoder/dispatch.rs:70-75).
    const int act_asked = act_mode;
    if (grid_fmt && !iq4 && act_mode == OJH_ACT_AUTO) act_mode = OJH_ACT_Q8K;
    if (grid_fmt && (rc = ensure(dev, "iq_grid"))) return rc;
    // Formats without a tile of their own (the IQ4 types, the legacy 32-weight blocks, Q2_K / Q3_K, MXFP4, the grid
    // codebooks) against a batch: their matvec walks the rows once per token (14336 x 4096: 8 us a token, 1 ms at 128
    // tokens).  From `deq_min_m` tokens the rows are decoded once into library scratch (`dequant_<fmt>_f16`:
    // dequant_to_f16's bits) and the batch runs on the f16 tile — what the reference does at load time for every
    // tensor it cannot keep in place (crates/ojas-cuda/src/qwen35.rs:174-201), without holding the f16 copy.
    // (from where the decode pass plus the tile beat the matvec that walks the rows once per four tokens: measured with
    // the decoders at 22 - 31 us for 14336 x 4096, pass + tile 50 - 56 us flat against 37 - 41 / 66 / 98 us at 4 / 8 / 12
    // tokens; on 4096 x 4096 28 against 13 / 22 / 31 / 39 at 4 / 8 / 12 / 16)
    const uint32_t deq_min = dev->deq_min_m != 1 ? dev->deq_min_m : (uint64_t)N * K >= (32ull << 20) ? 5u : 9u;
    // IQ4_NL / IQ4_XS rows have loaders in the tile: short of the long batches they skip the decode pass (14336 x 4096:
    // 53 - 62 -> 32 - 42 us up to 128 tokens; 4096 x 4096 at 16 tokens 29 -> 14; beyond, f16d_pays weighs the pass again) and
    // take the tile from 5 tokens on every shape (the matvec that walks the rows once per four tokens: 13 / 22 us at 4 / 8
    // tokens on 4096 x 4096)
    // (the legacy 32-weight blocks, MXFP4, Q2_K and Q3_K likewise)
    const bool own_loader = w->type == OJH_IQ4_NL || (w->type == OJH_IQ4_XS && K % 256 == 0) || w->type == OJH_Q4_0 ||
                            w->type == OJH_Q4_1 || w->type == OJH_Q5_0 || w->type == OJH_Q5_1 || w->type == OJH_MXFP4 ||
                            ((w->type == OJH_Q2_K || w->type == OJH_Q3_K) && K % 256 == 0);
    const bool iq4_own = dev->iq4_tile && own_loader &&
                         act_asked != OJH_ACT_Q8K && m >= dev->iq4_tile &&
                         (w->type != OJH_Q3_K || m <= dev->iq4_tile_cap) &&   // (Q3_K: eight loads at 2-byte alignment per thread and step, 55 against 68 us at 128 tokens, 86 against 82 at 256)
                         K % 64 == 0;
    const bool deq_tile = ((iq4 || grid_fmt) && !iq4_own && !q5_float && act_asked != OJH_ACT_Q8K && deq_min && m >= deq_min) &&
                          !dev->no_scratch && K % 64 == 0 && (uint64_t)N * K / f->weights <= 0x7FFFFFFFu / 64;
    const bool tile_fits = K % 64 == 0 && (uint64_t)m * K < 0x7FFFFFFFull && (uint64_t)m * N < 0x7FFFFFFFull;
    const bool tile_taken = (deq_tile || iq4_own || (m >= tile_min && act_mode != OJH_ACT_Q8K && !iq4 && !grid_fmt)) && tile_fits;
    const bool q4kl = w->type == OJH_Q4_K && !dev->gemm_exact && act_mode != OJH_ACT_FLOAT_EXACT;
    // (Q4_K rows not where y lies over x: the pass may clear y while it converts x, which their own tiles, whole, do not)
    if (tile_taken && f16d_taken(dev, w, m, act_mode, deq_tile) && !(q4kl && overlap(at(x, x_off), (size_t)m * K * esz, yp, (size_t)m * N * 4))) {
        bool ready;
        if ((rc = f16d_ready(dev, w, m, deq_tile, q4kl, &ready))) return rc;
        if (ready) return f16d_launch(dev, at(x, x_off), x_dtype, w, f, yp, m, accum, q4kl);
    }
    void *tile_w = wp;
    if (deq_tile) {
        ojh_buf *wdeq;
        if ((rc = ojh_scratch_get(dev, "wdeq", (size_t)N * K * 2, &wdeq))) return rc;
        if ((rc = ensure(dev, grid_fmt ? "iq_grid" : "dequant"))) return rc;
        const std::string dq = std::string("dequant_") + f->tag + "_f16";
        const uint32_t nb = (uint32_t)((uint64_t)N * K / f->weights);
        uint32_t dg[3], db[3];
        if ((rc = ojh_launch_shape(dev, dq.c_str(), 0, nb, 0, dg, db))) return rc;
        if ((rc = ojh_launch(dev, dq.c_str(), {wp, wdeq->ptr}, {nb}, dg, db))) return rc;
        tile_w = wdeq->ptr;
    }
    if (tile_taken) {
        // Q4_K takes the 256-wide tile with the reference GPU kernel's arithmetic (f16 qa*q + qb)
        // unless the tile that reproduces dequant_to_f16 bit for bit is asked for.
        const bool xl = w->type == OJH_Q4_K && !dev->gemm_exact && act_mode != OJH_ACT_FLOAT_EXACT &&
                        (uint64_t)w->row_bytes * N <= 0xFFFFFFFFull;  // 32-bit row offsets in that tile
        if ((rc = ensure(dev, "glue")) || (rc = ensure(dev, xl ? "gemm_xl" : "gemm"))) return rc;
        // (the few-token kernel below reads the tokens' f16 copy in the order of its lanes where there is room for whole
        // groups of sixteen tokens, row by row otherwise; with the growing room that a recorded batch of a few more may count on)
        const uint32_t few_tg = m <= 16 ? 1 : m <= 32 ? 2 : 4;
        ojh_buf *xh;
        const bool few_frag = !xl && !deq_tile && dev->gemm_few && m <= dev->gemm_few && m <= 64 && K % 128 == 0 && (own_loader || w->type == OJH_Q8_0) &&
                              !ojh_scratch_spare(dev, "xh", (size_t)16 * few_tg * K * 2, &xh, true);
        if (!few_frag && (rc = ojh_scratch_get(dev, "xh", (size_t)m * K * 2, &xh))) return rc;
        const uint32_t n_el = m * K, conv_blocks = (n_el / 8 + 255) / 256 + 1;
        std::string base = std::string("gemm_mm_") + (deq_tile ? "f16" : w->type == OJH_Q8_0 ? "q8_0" : f->tag);
        // (the tile that shares the dequantized weights through LDS is 256 tokens tall; its 128-token form up to 128 tokens
        // and wherever the taller one would give at most half of the CUs a tile — 14336 x 4096 at 256 tokens: Q8_0 78 ->
        // 55 us, Q6_K 100 -> 77 — and for plain f16 rows, 322 -> 288 us at 2048 tokens)
        if (!xl && gemm_mm_m128(dev, N, m, deq_tile)) base += "_m128";
        if (xl) {
            // 256-token tiles when they give every CU a tile, or half of them with a K long enough
            // to split in two without the slices' fixed costs showing (measured on MI355X);
            // 128-token tiles, which dequantize every weight for half as many MFMAs, otherwise — in the form that
            // dequantizes straight into the B registers (5-17 % ahead of the form that shares the f16 tile through LDS).
            uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
            uint32_t t256 = ((N + 255) / 256) * ((m + 255) / 256);
            bool tall = m > 128 && (t256 >= cus || (2 * t256 >= cus && K >= 8192));
            base = tall ? "gemm_mm_q4kl" : "gemm_mm_q4kl_bd";
            // 128-token tiles of 256 rows too few to fill the chip: 64-row tiles whose four waves split K between them
            // and meet in LDS — four times the tiles before any K slice has to meet another through atomics
            // (measured: gate/up at 128 tokens 26 against 42 us, down at 512 tokens 74 against 88, 4096 x 4096 at 512
            // tokens 33 against 51 with the conversion)
            // — wherever the 256-row tiles would have to split K in two or more (from four slices when K is long: there
            // the longer loop pays more for the waves' separate activation copies than two slices' atomics cost)
            const uint32_t t_bd = ((N + 255) / 256) * ((m + 127) / 128), z_bd = t_bd ? cus / t_bd : 0;
            if (!tall && K >= 1024 && (dev->gemm_bdk == 2 || (dev->gemm_bdk == 1 && z_bd >= 2 && (K <= 8192 || z_bd >= 4))))
                base = "gemm_mm_q4kl_bdk";
        }
        // A few tokens on the formats whose 32 weights per thread come out of one or two wide loads: 16 (or 64) rows per
        // workgroup with the weights decoded straight into the matrix operand, no LDS staging, no barrier per K step
        // (`gemm_few_*`; 14336 x 4096 at 8 / 16 / 32 tokens, kernel alone: IQ4_XS 14 / 15 / 23 us against 30 of the tile,
        // Q8_0 26 / 28 / 32 against 36; 4096 x 4096 IQ4_XS 7 / 9 / 11 against 12 .. 14).  Four row groups per workgroup where
        // that still gives most CUs a workgroup: the tokens' bytes, re-read by every workgroup, are most of its traffic.
        // (with 16 rows per workgroup a long K costs more, and below 2048 rows there are few of them: up to 16 tokens there, and
        // none for Q8_0, twice the bytes per weight, nor more for Q3_K, eight loads at 2-byte alignment.  Tile / this kernel
        // beyond, us: 4096 x 14336 at 24 tokens IQ4_XS 29.1 / 18.4, at 30 Q4_0 30.3 / 23.4, Q5_1 31.6 / 21.4, Q2_K 32.1 / 21.8, MXFP4
        // 29.7 / 21.3, Q3_K 40.7 / 40.4; 2048 x 8192 IQ4_XS at 24 13.9 / 12.8; 1024 x 8192 at 24 Q4_0 13.4 / 14.6, Q2_K 13.9 / 15.5;
        // Q8_0 4096^2 at 32 16.9 / 12.2, 2048 x 4096 at 32 13.0 / 11.8, 1024 x 4096 at 24 10.7 / 11.5, 2048 x 8192 at 12 14.4 / 17.5)
        const uint32_t cus = (uint32_t)dev->prop.multiProcessorCount;
        const bool r4 = (uint64_t)(N + 63) / 64 * 4 >= 3ull * cus;
        const bool few_long = N >= 2048 ? w->type != OJH_Q3_K || K <= 4096 : w->type != OJH_Q8_0 && K <= 4096;
        const uint32_t few_cap = r4 ? dev->gemm_few : w->type == OJH_Q8_0 && K > 4096 ? 0u : few_long ? dev->gemm_few : std::min(dev->gemm_few, 16u);
        if (dev->gemm_few && !xl && !deq_tile && (own_loader || w->type == OJH_Q8_0) && m <= few_cap && m <= 64 && K % 128 == 0) {
            const std::string few = std::string("gemm_few_") + (w->type == OJH_Q8_0 ? "q8_0" : f->tag) + (r4 ? "_r4" : "") +
                                    (m <= 16 ? "_t1" : m <= 32 ? "_t2" : "_t4");
            uint32_t fg[3], fb[3], eg[3] = {few_frag ? K / 128 * few_tg : conv_blocks, 1, 1};
            if ((rc = ojh_launch_shape(dev, few.c_str(), K, N, m, fg, fb))) return rc;
            if ((rc = few_frag ? ojh_launch(dev, x_dtype == OJH_X_BF16 ? "few_x_bf16" : "few_x_f32", {at(x, x_off), xh->ptr}, {K, m, few_tg}, eg, block)
                               : ojh_launch(dev, x_dtype == OJH_X_BF16 ? "copy_bf16_half" : "copy_f32_half", {at(x, x_off), xh->ptr}, {n_el}, eg, block)))
                return rc;
            return ojh_launch(dev, few.c_str(), {xh->ptr, wp, yp}, {K, N, (few_frag ? 2u : 0u) | (uint32_t)(accum != 0), m}, fg, fb);
        }
        uint32_t sg[3], sb[3];
        if ((rc = ojh_launch_shape(dev, (base + "_sk").c_str(), K, N, m, sg, sb))) return rc;
        // (a forced split counts before the tile is chosen, so that what follows sees the split that will run)
        if (dev->gemm_split_override > 0) sg[2] = (uint32_t)dev->gemm_split_override;
        if (dev->gemm_sr && base == "gemm_mm_q4kl_bdk" && sg[2] > 1) {   // reproducible bits asked for: its K slices meet in atomics
            base = "gemm_mm_q4kl_bd";
            if ((rc = ojh_launch_shape(dev, (base + "_sk").c_str(), K, N, m, sg, sb))) return rc;
            if (dev->gemm_split_override > 0) sg[2] = (uint32_t)dev->gemm_split_override;
        }
        // ... and tiles without a slice-ordered form (the LDS-shared Q4_K tile, Q6_K, Q8_0) keep K whole under that request:
        // their slices could only meet in f32 atomics, in arrival order
        if (dev->gemm_sr && sg[2] > 1 && !(xl && (base == "gemm_mm_q4kl_bd" || (base == "gemm_mm_q4kl" &&
                (uint64_t)sg[0] * sg[1] * sg[2] >= (uint32_t)dev->prop.multiProcessorCount))))
            sg[2] = 1;
        // 256-token tiles that fill the chip: the form that dequantizes into the B registers (same grid).  Its step
        // time does not grow with the number of busy CUs as the LDS-shared tile's does (measured: 2.2 us per K step
        // at 224 and at 448 workgroups against 2.0 and 2.4).
        if (xl && base == "gemm_mm_q4kl" && (uint64_t)sg[0] * sg[1] * sg[2] >= (uint32_t)dev->prop.multiProcessorCount)
            base = "gemm_mm_q4kl_bd256";
        // On request (OJAS_HIP_GEMM_SR=1) the K slices of the tiles that dequantize into the B registers meet in
        // scratch, the last slice of a tile to finish adding them in slice order: bits that do not depend on arrival, no
        // zero fill.  Measured slower than the atomics (one workgroup per tile reads every slice back from behind the
        // L2: gate/up at 128 tokens 60 against 45 us, down 142 against 46), so it is not the default.
        if (sg[2] > 1 && xl && (base == "gemm_mm_q4kl_bd" || base == "gemm_mm_q4kl_bd256") && dev->gemm_sr && !dev->no_scratch) {
            uint32_t eg[3] = {conv_blocks, 1, 1};
            if ((rc = ojh_launch(dev, x_dtype == OJH_X_BF16 ? "copy_bf16_half" : "copy_f32_half", {at(x, x_off), xh->ptr},
                                 {n_el}, eg, block)))
                return rc;
            const size_t tiles = (size_t)sg[0] * sg[1], bm = base == "gemm_mm_q4kl_bd256" ? 256 : 128;
            ojh_buf *part, *cnt;
            if ((rc = ojh_scratch_get(dev, "gemm_part", tiles * ojh_gemm_sr_slices(K, sg[2]) * bm * 256 * 4, &part))) return rc;
            if ((rc = ojh_scratch_get_zeroed(dev, "gemm_cnt", tiles * 4, &cnt))) return rc;
            return ojh_launch(dev, (base + "_sr").c_str(), {xh->ptr, wp, yp, part->ptr, cnt->ptr},
                              {K, N, m, sg[2], (uint32_t)(accum != 0)}, sg, sb);
        }
        // activations to f16 — and, ahead of K slices that add into y, the zero fill of y in the same launch
        if (sg[2] > 1 && !accum) {
            uint32_t n_y = m * N, cg[3] = {conv_blocks + (n_y / 4 + 255) / 256 + 1, 1, 1};
            if ((rc = ojh_launch(dev, x_dtype == OJH_X_BF16 ? "copy_bf16_half_zero" : "copy_f32_half_zero",
                                 {at(x, x_off), xh->ptr, yp}, {n_el, n_y, conv_blocks}, cg, block)))
                return rc;
        } else {
            uint32_t eg[3] = {conv_blocks, 1, 1};
            if ((rc = ojh_launch(dev, x_dtype == OJH_X_BF16 ? "copy_bf16_half" : "copy_f32_half", {at(x, x_off), xh->ptr},
                                 {n_el}, eg, block)))
                return rc;
        }
        if (sg[2] > 1) return ojh_launch(dev, (base + "_sk").c_str(), {xh->ptr, tile_w, yp}, {K, N, m, sg[2]}, sg, sb);
        sg[2] = 1;
        return ojh_launch(dev, base.c_str(), {xh->ptr, tile_w, yp}, {K, N, (uint32_t)(accum != 0), m}, sg, sb);
    }

    bool q8k = !ojh_float_rows(w->type) && act_mode != OJH_ACT_FLOAT && act_mode != OJH_ACT_FLOAT_EXACT;
    if (grid_fmt && act_mode == OJH_ACT_FLOAT_EXACT)
        return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_mm: %s rows have no MFMA tile; OJH_ACT_FLOAT runs their f32-activation matvec", f->tag);
    // Opt-in: one token, f32 in, plain store through the launch that quantizes x itself
    // (bit-identical results).  Measured slower than quantize + matvec at every decode shape on
    // MI355X — each block repeats the quantization and reads x through LDS — so it is off by default.
    if (q8k && m == 1 && !accum && !bias && x_dtype == OJH_X_F32 && w->type == OJH_Q4_K && K <= 16384 &&
        dev->fused_quant) {
        if ((rc = ensure(dev, "gemv_q8k"))) return rc;
        int r = pick_rows(dev, N);
        if (r > 2) r = 2;
        const char *name = (r == 2 && N >= 32768u) ? "gemv_fq8k_q4k_wide" : r == 2 ? "gemv_fq8k_q4k_r2" : "gemv_fq8k_q4k_r1";
        // rows per block: every block re-quantizes x, so give it enough rows that this stays a
        // small share, but keep several blocks per CU
        uint32_t unit = 4u * (uint32_t)r, cus = (uint32_t)dev->prop.multiProcessorCount;
        uint32_t nrb = (N + cus * dev->fq_blocks_per_cu - 1) / (cus * dev->fq_blocks_per_cu);
        nrb = ((nrb + unit - 1) / unit) * unit;
        if (nrb < unit) nrb = unit;
        grid[0] = (N + nrb - 1) / nrb;
        return ojh_launch(dev, name, {at(x, x_off), wp, yp}, {K, N, nrb}, grid, block);
    }
    if (q8k && m == 1 && !bias && fq_one_taken(dev, w, at(x, x_off), K * esz, yp))
        return !fq_one_alone(dev, w) && (rc = fq_scratch(dev, K)) ? rc : fq_one_launch(dev, at(x, x_off), x_dtype, w, f, yp, accum);
    if (q8k) {
        if ((rc = ensure(dev, "gemv_q8k"))) return rc;
        size_t nsb = K / 256;
        ojh_buf *xq, *xs;
        if ((rc = ojh_scratch_get(dev, "xq", (size_t)m * nsb * 256, &xq))) return rc;
        if ((rc = ojh_scratch_get(dev, "xs", (size_t)m * nsb * 4, &xs))) return rc;
        // ahead of the 128-token int8 tile the quantizer writes that tile's side arrays too (one launch less)
        const int xt = q4k_xt_ready(dev, w, m, wp);
        if (xt != XT_NO) {
            if ((rc = ensure(dev, "gemm_q8k"))) return rc;
            const uint32_t mp = (m + 127) / 128 * 128;
            ojh_buf *xst, *sums;
            if ((rc = xt_scratch(dev, w, m, "xt_xst", nsb * mp * 4, &xst)) || (rc = xt_scratch(dev, w, m, "xt_sums", nsb * mp * 32, &sums))) return rc;
            uint32_t qg[3] = {K / 256 * (mp / 4), 1, 1};
            const std::string quant = std::string(x_dtype == OJH_X_BF16 ? "quantize_q8k_bf16_sides" : "quantize_q8k_sides") +
                                      (q4k_xk_slices(dev, K, N, m) ? "_h" : "");
            if ((rc = ojh_launch(dev, quant.c_str(),
                                 {at(x, x_off), xq->ptr, xs->ptr, xst->ptr, sums->ptr}, {K, m, mp}, qg, block)))
                return rc;
            return ojh_mm_q8k_launch(dev, xq->ptr, xs->ptr, w, f, yp, bias, m, accum, XT_SIDES);
        }
        if ((rc = ojh_quant_q8k_launch(dev, at(x, x_off), x_dtype, m, K, xq->ptr, xs->ptr))) return rc;
        return ojh_mm_q8k_launch(dev, xq->ptr, xs->ptr, w, f, yp, bias, m, accum, xt);
    }

    // floating-point activations: the matvec kernels read f32
    void *xp = at(x, x_off);
    if (x_dtype == OJH_X_BF16) {
        if ((rc = ensure(dev, "glue"))) return rc;
        ojh_buf *xf;
        if ((uint64_t)m * K > 0xFFFFFFFFull) return ojh_fail(OJH_ERR_ARG, "ojh_mm: %u x %u bf16 activations exceed 2^32 elements", m, K);
        if ((rc = ojh_scratch_get(dev, "xf", (size_t)m * K * 4, &xf))) return rc;
        uint32_t n_el = m * K, eg[3] = {(n_el / 8 + 255) / 256 + 1, 1, 1};
        if ((rc = ojh_launch(dev, "copy_bf16_f32", {xp, xf->ptr}, {n_el}, eg, block))) return rc;
        xp = xf->ptr;
    }
    if (!grid_fmt && (rc = ensure(dev, "gemv"))) return rc;
    std::string base = std::string("gemv_nat_") + f->tag;
    // Q8_0 rows from a few thousand up: activations in registers, rows copied into LDS by the
    // memory system (needs 16-byte aligned rows and a K that chunks)
    if (m == 1 && w->type == OJH_Q8_0 && dev->q80_lds && N >= dev->q80_lds_min_n && ojh_q80_lds_kc(K) &&
        (uintptr_t)wp % 16 == 0 && (uintptr_t)xp % 16 == 0) {
        uint32_t sg[3], sb[3];
        if ((rc = ojh_launch_shape(dev, "gemv_nat_q80_lds", K, N, 1, sg, sb))) return rc;
        std::vector<void *> p = {xp, wp, yp};
        if (bias) p.push_back(bias->ptr);
        return ojh_launch(dev, accum ? "gemv_nat_q80_lds_accum" : bias ? "gemv_nat_q80_lds_bias" : "gemv_nat_q80_lds", p,
                          {K, N, ojh_q80_lds_kc(K)}, sg, sb);
    }
    // an output head (K-quant or IQ4 rows): rows grid-stride, the wave's f32 activations in registers
    if (m == 1 && w->type != OJH_Q8_0 && dev->px && !accum && !bias && N >= 32768u && K <= 4096u) {
        uint32_t sg[3], sb[3];
        if ((rc = ojh_launch_shape(dev, (base + "_px").c_str(), K, N, 1, sg, sb))) return rc;
        return ojh_launch(dev, (base + "_px").c_str(), {xp, wp, yp}, {K, N}, sg, sb);
    }
    // the sub-block-per-lane form of IQ2_XXS / IQ2_S / IQ3_XXS / IQ3_S also wins on mid-sized projections, with fewer
    // workgroups (a wave needs a few row pairs to pay for the 64 activations it keeps): 14336 x 4096 IQ3_S 17.1 -> 15.9 us,
    // IQ2_XXS 17.4 -> 13.2 us at 512 workgroups
    if (m == 1 && dev->px && !accum && !bias && N >= 8192u && K <= 4096u &&
        (w->type == OJH_IQ2_XXS || w->type == OJH_IQ2_S || w->type == OJH_IQ3_XXS || w->type == OJH_IQ3_S)) {
        uint32_t sg[3] = {std::min(std::max(N / 28u / 64u * 64u, 256u), 2048u), 1, 1};
        return ojh_launch(dev, (base + "_px").c_str(), {xp, wp, yp}, {K, N}, sg, block);
    }
    if (m == 1) {
        // rows per wave for the f32-activation kernels (measured on Q4_K and Q6_K, K = 4096 and 14336): the
        // activation fragment is 4 bytes per weight, so sharing it pays earlier than for int8 activations —
        // two rows everywhere, four from 8192 Q4_K rows; one row only when told to
        int r = (accum || bias) ? 4 : dev->gemv_rows_override ? pick_rows(dev, N) : (w->type == OJH_Q4_K && N >= 8192u) ? 4 : 2;
        std::string name = base + (accum ? "_accum" : bias ? "_bias" : r == 4 ? "" : r == 2 ? "_r2" : "_r1");
        grid[0] = (N + 4 * r - 1) / (4 * r);
        std::vector<void *> p = {xp, wp, yp};
        if (bias) p.push_back(bias->ptr);
        return ojh_launch(dev, name.c_str(), p, {K, N}, grid, block);
    }
    // (waves that share rows where a row is many steps of 512 weights: two tokens from the fifth, more, also beyond four, from the
    // third; both sides at gemv_nat_ms_body)
    const bool shared = ojh_shares_rows(w->type) && K > (m == 2 ? 2048u : 1024u);
    grid[0] = (N + 3) / 4;
    return ojh_launch(dev, (base + (shared ? "_ms" : "_m")).c_str(), {xp, wp, yp}, {K, N, m, (uint32_t)(accum != 0)}, grid, block);
}

// ---- row-int8 path -------------------------------------------------------------------------------
extern "C" int ojh_q8rows_from_f16(ojh_device *dev, const ojh_buf *w16, size_t w_off, uint32_t n, uint32_t k,
                                   ojh_buf *q, ojh_buf *scale) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_q8rows_from_f16: NULL device");
    if (!n || !k) return ojh_fail(OJH_ERR_ARG, "ojh_q8rows_from_f16: n=%u k=%u", n, k);
    int rc;
    if ((rc = span_ok("q8rows: w16", w16, w_off, (size_t)n * k * 2, 2))) return rc;
    if ((rc = span_ok("q8rows: q", q, 0, (size_t)n * k, 16))) return rc;
    if ((rc = span_ok("q8rows: scale", scale, 0, (size_t)n * 4, 4))) return rc;
    if ((rc = ensure(dev, "rowq8"))) return rc;
    uint32_t grid[3] = {n, 1, 1}, block[3] = {256, 1, 1};
    return ojh_launch(dev, "rows_q8_from_f16", {at(w16, w_off), q->ptr, scale->ptr}, {k, n}, grid, block);
}

extern "C" int ojh_matmul_q8(ojh_device *dev, const ojh_buf *x, size_t x_off, const ojh_buf *wq, const ojh_buf *wscale,
                             const ojh_buf *bias, ojh_buf *y, size_t y_off, uint32_t n, uint32_t k, uint32_t m) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_matmul_q8: NULL device");
    if (!n || !k || !m || m > 65535) return ojh_fail(OJH_ERR_ARG, "ojh_matmul_q8: n=%u k=%u m=%u out of range", n, k, m);
    if (k % 16) return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_matmul_q8: K=%u must be a multiple of 16", k);
    int rc;
    if ((rc = span_ok("matmul_q8: x", x, x_off, (size_t)m * k * 4, 4))) return rc;
    if ((rc = span_ok("matmul_q8: wq", wq, 0, (size_t)n * k, 16))) return rc;
    if ((rc = span_ok("matmul_q8: wscale", wscale, 0, (size_t)n * 4, 4))) return rc;
    if (bias && (rc = span_ok("matmul_q8: bias", bias, 0, (size_t)n * 4, 4))) return rc;
    if ((rc = span_ok("matmul_q8: y", y, y_off, (size_t)m * n * 4, 4))) return rc;
    if ((rc = ensure(dev, "rowq8"))) return rc;
    ojh_buf *xq, *sx;
    if ((rc = ojh_scratch_get(dev, "q8_xq", (size_t)m * k, &xq))) return rc;
    if ((rc = ojh_scratch_get(dev, "q8_sx", (size_t)m * 4, &sx))) return rc;
    uint32_t block[3] = {256, 1, 1}, gq[3], bq[3], gm[3] = {(n + 3) / 4, 1, 1};
    if ((rc = ojh_launch_shape(dev, "quant_rows_i8", k, 0, m, gq, bq))) return rc;
    if ((rc = ojh_launch(dev, "quant_rows_i8", {at(x, x_off), xq->ptr, sx->ptr}, {k, m}, gq, bq))) return rc;
    // a batch: the integer sums on the int8 matrix instruction (the same bits; the per-row kernel reads a row once per
    // 8 tokens, so its time grows with the tokens)
    const uint32_t mt_min = dev->q8row_mt_min_m != 1 ? dev->q8row_mt_min_m : 9u;
    if (mt_min && m >= mt_min) {
        uint32_t gt[3] = {(n + 127) / 128, (m + 63) / 64, 1};
        void *bp = bias ? bias->ptr : nullptr;
        // 128 tokens a tile where that still leaves a tile and a half per CU
        const bool many = (uint64_t)gt[0] * ((m + 127) / 128) * 2 >= (uint64_t)3 * dev->prop.multiProcessorCount;
        const uint32_t t128 = dev->q8row_t128_min_m != 1 ? dev->q8row_t128_min_m : many ? 129u : 0u;
        if (t128 && m >= t128) {
            gt[1] = (m + 127) / 128;
            return ojh_launch(dev, "matmul_q8row_mt128", {xq->ptr, sx->ptr, wq->ptr, wscale->ptr, at(y, y_off), bp}, {k, n, m}, gt, block);
        }
        const uint32_t z = dev->no_scratch ? 1 : ojh_matmul_q8row_slices(dev, k, n, m);
        if (z > 1) {
            const size_t tiles = (size_t)gt[0] * gt[1];
            ojh_buf *part, *cnt;
            if ((rc = ojh_scratch_get(dev, "q8r_part", tiles * z * 32768, &part))) return rc;
            if ((rc = ojh_scratch_get_zeroed(dev, "q8r_cnt", tiles * 4, &cnt))) return rc;
            gt[2] = z;
            return ojh_launch(dev, "matmul_q8row_mt_sr", {xq->ptr, sx->ptr, wq->ptr, wscale->ptr, at(y, y_off), bp, part->ptr, cnt->ptr},
                              {k, n, m, z}, gt, block);
        }
        return ojh_launch(dev, "matmul_q8row_mt", {xq->ptr, sx->ptr, wq->ptr, wscale->ptr, at(y, y_off), bp}, {k, n, m}, gt, block);
    }
    if (dev->q8row_dec && m <= 8 && (size_t)m * k <= 131072) {
        const char *name = (size_t)m * k <= 65536 ? "matmul_q8row_dec" : "matmul_q8row_dec_l";
        uint32_t gd[3], bd[3];
        if ((rc = ojh_launch_shape(dev, name, k, n, m, gd, bd))) return rc;
        return ojh_launch(dev, name, {xq->ptr, sx->ptr, wq->ptr, wscale->ptr, at(y, y_off), bias ? bias->ptr : nullptr}, {k, n, m}, gd, bd);
    }
    if (bias)
        return ojh_launch(dev, "matmul_q8row_bias", {xq->ptr, sx->ptr, wq->ptr, wscale->ptr, at(y, y_off), bias->ptr},
                          {k, n, m}, gm, block);
    return ojh_launch(dev, "matmul_q8row", {xq->ptr, sx->ptr, wq->ptr, wscale->ptr, at(y, y_off)}, {k, n, m}, gm, block);
}

// ---- decode-layer epilogues around the matvec ----------------------------------------------------
extern "C" int ojh_rmsnorm_quant_q8k(ojh_device *dev, const ojh_buf *x, size_t x_off, const ojh_buf *gamma, float eps,
                                     uint32_t m, uint32_t k, ojh_buf *q, ojh_buf *scales, ojh_buf *xn) {
    if (!dev) return ojh_fail(OJH_ERR_ARG, "ojh_rmsnorm_quant_q8k: NULL device");
    if (!m || !k || k > 16384 || m > 65535) return ojh_fail(OJH_ERR_ARG, "rmsnorm_quant_q8k: m=%u k=%u out of range (k <= 16384)", m, k);
    size_t nsb = (k + 255) / 256;
    int rc;
    if ((rc = span_ok("rmsnorm_quant_q8k: x", x, x_off, (size_t)m * k * 4, 4))) return rc;
    if ((rc = span_ok("rmsnorm_quant_q8k: gamma", gamma, 0, (size_t)k * 4, 4))) return rc;
    if ((rc = span_ok("rmsnorm_quant_q8k: q", q, 0, (size_t)m * nsb * 256, 16))) return rc;
    if ((rc = span_ok("rmsnorm_quant_q8k: scales", scales, 0, (size_t)m * nsb * 4, 4))) return rc;
    if (xn && (rc = span_ok("rmsnorm_quant_q8k: xn", xn, 0, (size_t)m * k * 4, 4))) return rc;
    if ((rc = ensure(dev, "gemv_q8k"))) return rc;
    uint32_t eps_bits;
    memcpy(&eps_bits, &eps, 4);
    // a few rows: sixteen waves, a segment each up to 4096 values (the launch is one dependent chain of latencies);
    // many rows: four, so that several rows share a CU
    uint32_t grid[3] = {m, 1, 1}, block[3] = {dev->rms_threads ? dev->rms_threads : (m <= 64 ? 1024u : 256u), 1, 1};
    return ojh_launch(dev, "rmsnorm_q8k", {at(x, x_off), gamma->ptr, q->ptr, scales->ptr, xn ? xn->ptr : q->ptr},
                      {k, m, eps_bits, (uint32_t)(xn != nullptr)}, grid, block);
}

extern "C" int ojh_ffn_gu_q8k(ojh_device *dev, const ojh_buf *xq, const ojh_buf *xscales, const ojh_lin *gate,
                              const ojh_lin *up, ojh_buf *out, size_t out_off, int act) {
    if (!dev || !gate || !up) return ojh_fail(OJH_ERR_ARG, "ojh_ffn_gu_q8k: NULL argument");
    auto kq = [](uint32_t t) { return t == OJH_Q4_K || t == OJH_Q5_K || t == OJH_Q6_K; };
    if (!kq(gate->type) || !kq(up->type))
        return ojh_fail(OJH_ERR_UNSUPPORTED, "ojh_ffn_gu_q8k: gate and up must be Q4_K, Q5_K or Q6_K (got %u, %u)", gate->type, up->type);
    if (gate->n != up->n || gate->k != up->k)
        return ojh_fail(OJH_ERR_ARG, "ojh_ffn_gu_q8k: gate is %ux%u, up is %ux%u", gate->n, gate->k, up->n, up->k);
    if (act != 0 && act != 1) return ojh_fail(OJH_ERR_ARG, "ojh_ffn_gu_q8k: act=%d (0 = SiLU, 1 = GELU)", act);
    const uint32_t N = gate->n, K = gate->k;
    size_t nsb = K / 256;
    int rc;
    if ((rc = span_ok("ffn_gu: xq", xq, 0, nsb * 256, 16))) return rc;
    if ((rc = span_ok("ffn_gu: xscales", xscales, 0, nsb * 4, 4))) return rc;
    if ((rc = span_ok("ffn_gu: out", out, out_off, (size_t)N * 4, 4))) return rc;
    if ((rc = span_ok("ffn_gu: gate", gate->raw, gate->off, gate->row_bytes * N, ojh_block_align(ojh_format(gate->type))))) return rc;
    if ((rc = span_ok("ffn_gu: up", up->raw, up->off, up->row_bytes * N, ojh_block_align(ojh_format(up->type))))) return rc;
    if ((rc = ensure(dev, "gemv_q8k"))) return rc;
    uint32_t grid[3] = {(N + 3) / 4, 1, 1}, block[3] = {256, 1, 1};
    if (gate->type != OJH_Q4_K || up->type != OJH_Q4_K)   // every row in its own format's arithmetic
        return ojh_launch(dev, "ffn_gu_q8k_kq", {xq->ptr, xscales->ptr, at(gate->raw, gate->off), at(up->raw, up->off), at(out, out_off)},
                          {K, N, (uint32_t)act, gate->type | (up->type << 8)}, grid, block);
    return ojh_launch(dev, "ffn_gu_q8k_q4k", {xq->ptr, xscales->ptr, at(gate->raw, gate->off), at(up->raw, up->off), at(out, out_off)},
                      {K, N, (uint32_t)act}, grid, block);
}
