"""Each mechanism of the Lazolix design alone: the HIP kernel behind its one-sequence C entry (csrc/capi_stream32.hip) against the float64 oracle.
Where random inputs would hide a fault -- a far key among hundreds, a window's edge, a sink -- one query / key pair is scaled so that one score stands out."""
import ctypes as C

import numpy as np
import pytest

import lazolix_oracle as O
from uzu_amd import _ffi

pytestmark = pytest.mark.gpu


def ptr(a):
    return None if a is None else a.ctypes.data_as(C.c_void_p)


def f32(a):
    return np.ascontiguousarray(a, dtype=np.float32)


def linear(ctx, x, w, bias=None, residual=None, batch=1, act=0, bf16=0, form=0):
    rows = x.shape[0]
    n, k = w.shape[-2], w.shape[-1]
    y = np.empty((rows, n * batch), dtype=np.float32)
    wb, bb = O.bf16_bits(w), None if bias is None else O.bf16_bits(bias)
    _ffi.call("uzu_hip_s32_linear", ctx._h, ptr(f32(x)), ptr(wb), ptr(bb), ptr(None if residual is None else f32(residual)), ptr(y), C.c_uint32(rows), C.c_uint32(n), C.c_uint32(k),
              C.c_uint32(batch), C.c_uint32(act), C.c_uint32(bf16), C.c_uint32(form))
    return y


@pytest.mark.parametrize("rows,n,k", [(1, 7, 24), (3, 33, 40), (16, 64, 72), (17, 5, 9), (70, 130, 100), (129, 64, 64), (300, 96, 136)])
def test_linear_true_f32_every_row_count(hip_ctx, rows, n, k):
    rng = np.random.default_rng(rows)
    x, w, b, res = rng.standard_normal((rows, k)), O.to_bf16(rng.standard_normal((n, k))), O.to_bf16(rng.standard_normal(n)), rng.standard_normal((rows, n))
    want = np.maximum(f32(x).astype(np.float64) @ w.T.astype(np.float64) + b, 0) ** 2 + f32(res)
    got = linear(hip_ctx, x, w, b, res, act=1)
    assert np.abs(got - want).max() <= 2e-5 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("rows,n,k,batch", [(32, 64, 64, 1), (200, 200, 72, 1), (130, 48, 24, 3), (257, 128, 320, 1), (64, 320, 128, 2), (1000, 130, 136, 1)])
def test_linear_matrix_core_form_equals_the_plain_form(hip_ctx, rows, n, k, batch):
    """bf16 products: the matrix-core tiles against the same products without the matrix cores, every tile shape, ragged edges, the batched per-head form"""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((rows, k * batch))
    w = O.to_bf16(rng.standard_normal((batch, n, k)))
    b = O.to_bf16(rng.standard_normal(n)) if batch == 1 else None
    res = rng.standard_normal((rows, n)) if batch == 1 else None
    a = linear(hip_ctx, x, w, b, res, batch=batch, act=0, bf16=1, form=1)
    c = linear(hip_ctx, x, w, b, res, batch=batch, act=0, bf16=1, form=2)
    xb = O.to_bf16(x).astype(np.float64)
    want = np.concatenate([xb[:, z * k:(z + 1) * k] @ w[z].T.astype(np.float64) for z in range(batch)], axis=1)
    if batch == 1:
        want = want + b + f32(res)
    assert np.isfinite(a).all()
    assert np.abs(a - want).max() <= 3e-5 * max(1.0, np.abs(want).max()) and np.abs(c - want).max() <= 3e-5 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("rows,n,k,bf16", [(257, 128, 320, 0), (257, 128, 320, 1), (64, 70, 1024, 0), (17, 64, 64, 0)])
def test_linear_without_the_matrix_cores(hip_ctx, rows, n, k, bf16):
    """Form 2 keeps off the matrix cores at sizes where the dispatch takes them for f32 products as well: its 64 x 64 tiles add f32 product after f32 product in the order of k, which gives
    the same bits here (a fused multiply-add: the product is exact in 64 bits; the sum's second rounding on the way to f32 can differ once in 2^29)."""
    rng = np.random.default_rng(rows + k)
    x, w = f32(rng.standard_normal((rows, k))), O.to_bf16(rng.standard_normal((n, k)))
    got = linear(hip_ctx, x, w, act=0, bf16=bf16, form=2)
    xb = O.to_bf16(x) if bf16 else x
    want = np.zeros((rows, n), dtype=np.float32)
    for c in range(k):
        want = (want + np.multiply.outer(xb[:, c].astype(np.float64), w[:, c].astype(np.float64))).astype(np.float32)
    assert np.mean(got == want) > 1 - 1e-4


@pytest.mark.parametrize("rows,n,k,act", [(129, 8200, 1024, 0), (1000, 1025, 1024, 1), (255, 16400, 256, 0), (513, 8192, 256, 0), (2050, 4100, 128, 1), (128, 4100, 2048, 0), (33, 1024, 1024, 1), (300, 700, 2048, 0)])
def test_linear_prompt_sized_form(hip_ctx, rows, n, k, act):
    """Prompt-sized products (both operands by LDS DMA): every tile form and buffer count, ragged last tiles in both directions, two k-steps and many, bias, activation and a residual
    in place; f32 sums of bf16 products, so the bound of the other matrix-core form holds."""
    rng = np.random.default_rng(rows + n)
    x, w = rng.standard_normal((rows, k), dtype=np.float32), O.to_bf16(rng.standard_normal((n, k), dtype=np.float32))
    b, res = O.to_bf16(rng.standard_normal(n)), rng.standard_normal((rows, n), dtype=np.float32)
    got = linear(hip_ctx, x, w, b, res, act=act, bf16=1, form=1)
    want = O.to_bf16(x).astype(np.float64) @ w.T.astype(np.float64) + b
    want = (np.maximum(want, 0) ** 2 if act else want) + res
    assert np.abs(got - want).max() <= 3e-5 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("rows,n,k,act", [(17, 1500, 1024, 0), (33, 1025, 832, 1), (17, 70, 256, 0), (129, 4101, 64, 0), (300, 1024, 2048, 1), (64, 64, 8192, 0), (1025, 4100, 128, 0), (2050, 4100, 64, 0)])
def test_linear_f32_from_three_bf16_parts(hip_ctx, rows, n, k, act):
    """f32 products of many rows (each operand number as three bf16 numbers): against 64 bits, with numbers of mixed sizes; every tile form, the product cut along k, ragged last
    tiles.  f32 accumulation of 3 k exact products: each addition rounds a partial sum that is at most sum |x w| by 2^-24, and errors of k steps add like sqrt(k) (factor 4 of room)."""
    rng = np.random.default_rng(rows + n)
    x = f32(rng.standard_normal((rows, k)) * np.exp2(rng.integers(-12, 13, (rows, k))))
    w, b, res = O.to_bf16(rng.standard_normal((n, k), dtype=np.float32)), O.to_bf16(rng.standard_normal(n)), rng.standard_normal((rows, n), dtype=np.float32)
    got = linear(hip_ctx, x, w, b, res, act=act, bf16=0)
    lin = x.astype(np.float64) @ w.T.astype(np.float64) + b
    mass = np.abs(x.astype(np.float64)) @ np.abs(w.T.astype(np.float64)) + np.abs(b)
    bound = 4 * 2.0 ** -24 * np.sqrt(3 * k) * mass
    if act:
        bound = 2 * np.maximum(lin, 0) * bound + bound ** 2 + 2.0 ** -23 * lin ** 2
    want = (np.maximum(lin, 0) ** 2 if act else lin) + res
    assert (np.abs(got - want) <= bound + 2.0 ** -23 * (np.abs(want) + np.abs(res))).all()


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("rows,n,k,act", [(65, 129, 1024, 0), (129, 385, 4096, 1), (20, 64, 1152, 0), (513, 2049, 512, 0), (1030, 3900, 128, 1), (2048, 2048, 320, 0), (700, 1030, 1088, 0), (700, 765, 4096, 1)])
def test_linear_on_eight_waves_a_tile(hip_ctx, rows, n, k, act, bf16):
    """At most a 128 x 128 tile a CU (csrc/k_linear_mfma.hip: eight_wave_splits): whole and cut into two to eight shares with uneven counts of k-steps, fewer steps than buffers, ragged last
    tiles, all 256 tiles.  Against 64 bits, with the bound of the products above (bf16 products: k of them)."""
    rng = np.random.default_rng(rows + n + k)
    x = rng.standard_normal((rows, k), dtype=np.float32)
    w, b, res = O.to_bf16(rng.standard_normal((n, k), dtype=np.float32)), O.to_bf16(rng.standard_normal(n)), rng.standard_normal((rows, n), dtype=np.float32)
    got = linear(hip_ctx, x, w, b, res, act=act, bf16=bf16)
    xr = O.to_bf16(x).astype(np.float64) if bf16 else x.astype(np.float64)
    lin = xr @ w.T.astype(np.float64) + b
    bound = 4 * 2.0 ** -24 * np.sqrt((1 if bf16 else 3) * k) * (np.abs(xr) @ np.abs(w.T.astype(np.float64)) + np.abs(b))
    if act:
        bound = 2 * np.maximum(lin, 0) * bound + bound ** 2 + 2.0 ** -23 * lin ** 2
    want = (np.maximum(lin, 0) ** 2 if act else lin) + res
    assert (np.abs(got - want) <= bound + 2.0 ** -23 * (np.abs(want) + np.abs(res))).all()


@pytest.mark.parametrize("rows,n,k", [(300, 700, 2048), (1025, 4100, 128), (17, 70, 256), (600, 4100, 1024)])
@pytest.mark.parametrize("power", [-118, -123])
def test_linear_f32_parts_of_tiny_numbers(hip_ctx, rows, n, k, power):
    """... numbers whose last bits lie below the smallest bf16 number: the parts carry them all the same, in whole products and in ones cut along k inside a part.  The bound of the test
    above; the results themselves are normal numbers (weights of 2^20)."""
    rng = np.random.default_rng(rows + n)
    x = f32(rng.uniform(1.0, 4.0, (rows, k)) * rng.choice([-1.0, 1.0], (rows, k)) * 2.0 ** power)
    w = O.to_bf16(rng.standard_normal((n, k)) * 2.0 ** 20)
    got = linear(hip_ctx, x, w, act=0, bf16=0).astype(np.float64)
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    mass = np.abs(x.astype(np.float64)) @ np.abs(w.T.astype(np.float64))
    assert (np.abs(got - want) <= 4 * 2.0 ** -24 * np.sqrt(3 * k) * mass).all()
    assert np.linalg.norm((got - want) / 2.0 ** power) <= 2.0 ** -21 * np.linalg.norm(want / 2.0 ** power)


@pytest.mark.parametrize("rows,n,k", [(40, 700, 1024), (2050, 4100, 64), (600, 4100, 128), (1100, 8200, 64)])
def test_linear_f32_parts_with_weights_that_are_no_numbers(hip_ctx, rows, n, k):
    """An infinite weight makes an infinity of every non-zero operand, whichever of its parts are zero, and a NaN of zero; a NaN weight NaNs: in products cut along k and in every tile form."""
    rng = np.random.default_rng(rows)
    x = O.to_bf16(rng.standard_normal((rows, k), dtype=np.float32) + np.float32(3.0) * rng.choice([-1, 1], (rows, k)).astype(np.float32))  # (one part)
    x[::2] = f32(x[::2] * np.float32(1.001))  # (three)
    w = O.to_bf16(rng.standard_normal((n, k), dtype=np.float32))
    w[3, 5], w[n - 1, k - 1], w[n // 2, 0] = np.inf, -np.inf, np.nan
    w[7, 1], w[7, 2] = np.inf, np.inf
    x[5, 5], x[rows - 1, k - 1], x[9, 1] = 0.0, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.T.astype(np.float64)
    got = linear(hip_ctx, x, w, act=0, bf16=0)
    ok = np.isfinite(want)
    assert np.array_equal(got[~ok], want[~ok].astype(np.float32), equal_nan=True) and np.isfinite(got[ok]).all()
    assert np.abs(got[ok] - want[ok]).max() <= 3e-5 * np.abs(want[ok]).max()


def test_f32_experts_with_weights_that_are_no_numbers(hip_ctx):
    """... in the grouped products of the experts, the gated one and the one behind it: infinities and NaNs where 64 bits have them."""
    rng = np.random.default_rng(6)
    rows, routed, top, ff, d = 50, 4, 2, 256, 320
    x, wr = O.to_bf16(rng.standard_normal((rows, d))).astype(np.float32), O.to_bf16(rng.standard_normal((routed, d)) * 0.5)
    w13 = O.to_bf16(rng.standard_normal((routed, 2 * ff, d)) / np.sqrt(d))
    w2 = O.to_bf16(rng.standard_normal((routed, d, ff)) / np.sqrt(ff))
    w13[1, 4, 7], w13[2, ff + 9, 3], w2[0, 11, 2] = np.inf, np.inf, -np.inf  # up, gate, down
    corr, res = np.zeros(routed, np.float32), np.zeros((rows, d), np.float32)
    y, ids, wts = np.empty((rows, d), dtype=np.float32), np.empty((rows, top), dtype=np.int32), np.empty((rows, top), dtype=np.float32)
    _ffi.call("uzu_hip_s32_moe", hip_ctx._h, ptr(x), ptr(O.bf16_bits(wr)), ptr(corr), ptr(O.bf16_bits(w13)), ptr(O.bf16_bits(w2)), ptr(res), ptr(y), ptr(ids), ptr(wts), C.c_uint32(rows),
              C.c_uint32(d), C.c_uint32(ff), C.c_uint32(routed), C.c_uint32(0), C.c_uint32(top), C.c_uint32(3))
    want = np.zeros((rows, d))
    with np.errstate(invalid="ignore", over="ignore"):
        for r in range(rows):
            for e, wt in zip(ids[r], wts[r].astype(np.float64)):
                up, gate = np.split(w13[e].astype(np.float64) @ x[r].astype(np.float64), 2)
                want[r] += wt * (w2[e].astype(np.float64) @ (gate / (1 + np.exp(-gate)) * up))
    ok = np.isfinite(want)
    assert (~ok).any() and np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(y[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    assert np.abs(y[ok] - want[ok]).max() <= 2e-5 * np.abs(want[ok]).max()


def test_linear_f32_parts_keep_infinities_and_nans(hip_ctx):
    rng = np.random.default_rng(3)
    x, w = rng.standard_normal((40, 1024), dtype=np.float32), O.to_bf16(np.abs(rng.standard_normal((700, 1024), dtype=np.float32)) + 0.5)
    x[3, 5], x[7, 900], x[11, 0], x[20, 1] = np.inf, -np.inf, np.nan, 3.4e38
    w[:, 1] = 1.0
    got = linear(hip_ctx, x, w, act=0, bf16=0)
    assert np.isposinf(got[3]).all() and np.isneginf(got[7]).all() and np.isnan(got[11]).all() and np.isfinite(np.delete(got, [3, 7, 11], 0)).all()
    assert np.abs(got[20] - 3.4e38).max() <= 3.4e38 * 2.0 ** -22


@pytest.mark.parametrize("rows,start", [(1, 0), (1, 5), (6, 0), (9, 3)])
def test_dyn_tanh_and_token_shift_with_state(hip_ctx, rows, start):
    rng = np.random.default_rng(rows + start)
    d = 70
    x, w, b, mu, prev = rng.standard_normal((rows, d)) * 2, 1 + 0.2 * rng.standard_normal(d), 0.1 * rng.standard_normal(d), rng.random(d), rng.standard_normal(d)
    alpha = 0.7
    h = O.dyn_tanh(f32(x), f32(w), f32(b), np.float32(alpha))
    want, last = O.token_shift(h, f32(mu), prev=f32(prev) if start else None)
    out, state = np.empty((rows, d), dtype=np.float32), f32(prev).copy()
    _ffi.call("uzu_hip_s32_dyn_tanh", hip_ctx._h, ptr(f32(x)), ptr(f32(w)), ptr(f32(b)), C.c_float(alpha), ptr(f32(mu)), ptr(state), C.c_uint32(start), ptr(out), C.c_uint32(rows),
              C.c_uint32(d))
    assert np.abs(out - want).max() < 5e-6 and np.abs(state - last).max() < 5e-6   # position 0 ignores what the state row held
    plain = np.empty((rows, d), dtype=np.float32)
    _ffi.call("uzu_hip_s32_dyn_tanh", hip_ctx._h, ptr(f32(x)), ptr(f32(w)), None, C.c_float(alpha), None, None, C.c_uint32(0), ptr(plain), C.c_uint32(rows), C.c_uint32(d))
    assert np.abs(plain - O.dyn_tanh(f32(x), f32(w), None, np.float32(alpha))).max() < 5e-6


def test_depth_mix(hip_ctx):
    rng = np.random.default_rng(5)
    slots, w = f32(rng.standard_normal((4, 7, 33))), f32(rng.standard_normal(4))
    out = np.empty((7, 33), dtype=np.float32)
    _ffi.call("uzu_hip_s32_depth_mix", hip_ctx._h, ptr(slots), ptr(w), C.c_uint32(4), ptr(out), C.c_uint32(7), C.c_uint32(33))
    assert np.abs(out - O.depth_mix(list(slots.astype(np.float64)), w)).max() < 1e-5


@pytest.mark.parametrize("bf16", [0, 1])
def test_latent_norm_append_keeps_earlier_rows(hip_ctx, bf16):
    rng = np.random.default_rng(6)
    start, rows, rank = 5, 4, 40
    cache = f32(O.to_bf16(rng.standard_normal((start + rows, rank))))
    before = cache.copy()
    u, g = f32(rng.standard_normal((rows, rank)) * 3), f32(1 + 0.2 * rng.standard_normal(rank))
    _ffi.call("uzu_hip_s32_latent_norm_append", hip_ctx._h, ptr(u), ptr(g), C.c_float(1e-3), ptr(cache), C.c_uint32(bf16), C.c_uint32(start), C.c_uint32(rows), C.c_uint32(rank))
    want = O.rms_latent(u.astype(np.float64), g, 1e-3)
    assert np.array_equal(cache[:start], before[:start])
    assert np.abs(cache[start:] - want).max() <= (2e-2 if bf16 else 5e-6)


def core(ctx, qlat, cache, sinks, rows, start, heads, rank, window, scale, bf16, form):
    out = np.empty((rows, heads * rank), dtype=np.float32)
    _ffi.call("uzu_hip_s32_latent_attention", ctx._h, ptr(f32(qlat)), ptr(f32(cache)), ptr(None if sinks is None else f32(sinks)), ptr(out), C.c_uint32(rows), C.c_uint32(start),
              C.c_uint32(heads), C.c_uint32(rank), C.c_uint32(window), C.c_float(scale), C.c_uint32(bf16), C.c_uint32(form))
    return out


FORMS = [(0, 1), (1, 1), (1, 2), (1, 3)]  # (bf16 cache, form): f32 simple, bf16 simple, bf16 tiled, bf16 tiled with the keys split over workgroups


@pytest.mark.parametrize("bf16,form", FORMS)
@pytest.mark.parametrize("rows,start,heads,rank,window", [(1, 0, 3, 40, 0), (7, 0, 3, 40, 4), (1, 9, 5, 24, 4), (40, 3, 3, 72, 9), (5, 130, 2, 128, 0), (150, 0, 8, 128, 33), (33, 64, 16, 256, 32), (3, 2, 2, 1100, 0), (2, 6, 3, 320, 5)])
def test_latent_core_against_the_oracle(hip_ctx, bf16, form, rows, start, heads, rank, window):
    rng = np.random.default_rng(rows * 7 + start)
    if form >= 2 and (rank > 256 or rank % 8):  # the matrix-core form refuses what it does not cover (the dispatcher then takes the simple form)
        with pytest.raises(_ffi.UzuHipError):
            core(hip_ctx, np.zeros((rows, heads * rank)), np.zeros((start + rows, rank)), None, rows, start, heads, rank, window, 1.0, bf16, form)
        return
    cache = O.to_bf16(rng.standard_normal((start + rows, rank)))
    qlat = O.to_bf16(rng.standard_normal((rows, heads * rank)) * 1.5)   # bf16-representable queries: the tiled form's rounding of them is then exact
    sinks = rng.standard_normal(heads) if rows % 2 else None
    got = core(hip_ctx, qlat, cache, sinks, rows, start, heads, rank, window, rank ** -0.5, bf16, form)
    want = O.latent_core(qlat, cache, heads, rank ** -0.5, window, sinks, start)
    assert np.isfinite(got).all() and np.abs(got - want).max() < (2e-4 if form >= 2 else 2e-5)


@pytest.mark.parametrize("bf16,form", FORMS)
@pytest.mark.parametrize("rows,start", [(1, 299), (300, 0), (45, 255)])   # decoding alone, a whole prompt, a portion behind a prefix
def test_latent_core_one_key_stands_out_at_every_edge(hip_ctx, bf16, form, rows, start):
    """The last row's query is aligned with ONE key.  Just inside the window (and at a block border, and far back without a window) the output must be that key's
    latent; just outside, the key must leave no trace."""
    rng = np.random.default_rng(9)
    heads, rank, T = 2, 64, start + rows
    t = T - 1
    for window, j, inside in [(40, t - 39, True), (40, t - 40, False), (0, 3, True), (200, t - 199, True), (200, t - 200, False), (33, t - 32, True), (1, t, True), (1, t - 1, False),
                              (64, t - 63, True), (65, t - 64, True), (64, t - 64, False)]:
        cache = O.to_bf16(rng.standard_normal((T, rank)))
        qlat = O.to_bf16(rng.standard_normal((rows, heads * rank)) * 0.3)
        qlat[-1, :rank] = O.to_bf16(cache[j] * 4.0)                       # head 0 of the last row: score ~ 4 * 64 * scale above everything else
        got = core(hip_ctx, qlat, cache, np.zeros(heads), rows, start, heads, rank, window, 0.5, bf16, form)
        want = O.latent_core(qlat, cache, heads, 0.5, window, np.zeros(heads), start)
        assert np.abs(got - want).max() < 3e-4, (window, j)
        hit = np.abs(got[-1, :rank] - cache[j]).max() < 1e-2
        assert hit == inside, (window, j, inside)


@pytest.mark.parametrize("bf16,form", FORMS)
def test_latent_core_sink_takes_weight_and_first_tokens(hip_ctx, bf16, form):
    rng = np.random.default_rng(10)
    heads, rank = 4, 32
    cache, qlat = O.to_bf16(rng.standard_normal((6, rank))), O.to_bf16(rng.standard_normal((6, heads * rank)))
    sinks = np.array([-30.0, 0.0, 5.0, 30.0])
    got = core(hip_ctx, qlat, cache, sinks, 6, 0, heads, rank, 3, 0.2, bf16, form)
    assert np.abs(got - O.latent_core(qlat, cache, heads, 0.2, 3, sinks)).max() < 2e-4
    assert np.abs(got[0, :rank] - cache[0]).max() < 1e-3        # position 0, a negligible sink: the only key gets all the weight
    assert np.abs(got[:, 3 * rank:]).max() < 1e-6               # a dominant sink: (almost) nothing is left for the keys
    no_sink = core(hip_ctx, qlat, cache, None, 6, 0, heads, rank, 3, 0.2, bf16, form)
    assert np.abs(no_sink[0].reshape(heads, rank) - cache[0]).max() < 1e-3


@pytest.mark.parametrize("routed,identity,top,ff", [(4, 0, 1, 16), (3, 2, 2, 24), (1, 1, 2, 8), (0, 3, 2, 0), (9, 1, 4, 40), (5, 1, 4, 3200)])
def test_score_routed_experts(hip_ctx, routed, identity, top, ff):
    rng = np.random.default_rng(routed * 10 + top)
    rows, d = 13, 48
    x = f32(rng.standard_normal((rows, d)))
    wr = O.to_bf16(rng.standard_normal((routed + identity, d)) * 0.5)
    corr = f32(0.3 * rng.standard_normal(routed + identity))
    experts = [tuple(O.to_bf16(rng.standard_normal(s) / np.sqrt(s[1])) for s in ((ff, d), (ff, d), (d, ff))) for _ in range(routed)]
    w13 = np.stack([np.concatenate([O.bf16_bits(u), O.bf16_bits(g)]) for g, u, _ in experts]) if routed else None
    w2 = np.stack([O.bf16_bits(dn) for _, _, dn in experts]) if routed else None
    res = f32(rng.standard_normal((rows, d)))
    y, ids, wts = np.empty((rows, d), dtype=np.float32), np.empty((rows, top), dtype=np.int32), np.empty((rows, top), dtype=np.float32)
    _ffi.call("uzu_hip_s32_moe", hip_ctx._h, ptr(x), ptr(O.bf16_bits(wr)), ptr(corr), ptr(w13), ptr(w2), ptr(res), ptr(y), ptr(ids), ptr(wts), C.c_uint32(rows), C.c_uint32(d),
              C.c_uint32(ff), C.c_uint32(routed), C.c_uint32(identity), C.c_uint32(top), C.c_uint32(0))
    want_ids, want_w = O.route(x.astype(np.float64), wr, corr, top)
    assert np.array_equal(ids, want_ids) and np.abs(wts - want_w).max() < 1e-5
    want = res + O.moe_mlp(x.astype(np.float64), wr, corr, experts, top)
    assert np.abs(y - want).max() < 3e-5 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("rows,routed,identity,top,ff,d", [(64, 4, 1, 2, 32, 64), (300, 3, 0, 1, 40, 72), (257, 8, 2, 3, 64, 128), (100, 5, 1, 2, 24, 48)])
def test_grouped_expert_form_equals_the_per_row_form(hip_ctx, rows, routed, identity, top, ff, d):
    """prefill-sized row counts, bf16 products: buckets per expert through the matrix-core linear against the per-row kernels and the oracle on rounded operands"""
    rng = np.random.default_rng(rows)
    x = f32(rng.standard_normal((rows, d)))
    wr = O.to_bf16(rng.standard_normal((routed + identity, d)) * 0.5)
    corr = f32(0.1 * rng.standard_normal(routed + identity))
    experts = [tuple(O.to_bf16(rng.standard_normal(s) / np.sqrt(s[1])) for s in ((ff, d), (ff, d), (d, ff))) for _ in range(routed)]
    w13 = np.stack([np.concatenate([O.bf16_bits(u), O.bf16_bits(g)]) for g, u, _ in experts])
    w2 = np.stack([O.bf16_bits(dn) for _, _, dn in experts])
    res = f32(rng.standard_normal((rows, d)))
    outs = []
    for mode in (1, 2):
        y, ids, wts = np.empty((rows, d), dtype=np.float32), np.empty((rows, top), dtype=np.int32), np.empty((rows, top), dtype=np.float32)
        _ffi.call("uzu_hip_s32_moe", hip_ctx._h, ptr(x), ptr(O.bf16_bits(wr)), ptr(corr), ptr(w13), ptr(w2), ptr(res), ptr(y), ptr(ids), ptr(wts), C.c_uint32(rows), C.c_uint32(d),
                  C.c_uint32(ff), C.c_uint32(routed), C.c_uint32(identity), C.c_uint32(top), C.c_uint32(mode))
        outs.append(y)
    assert np.isfinite(outs[1]).all() and np.abs(outs[0] - outs[1]).max() < 2e-4 * max(1.0, np.abs(outs[0]).max())


@pytest.mark.parametrize("rows,routed,identity,top,ff,d", [(700, 5, 1, 2, 1088, 1024), (1030, 64, 0, 1, 1024, 1024)])
def test_grouped_expert_form_prompt_sized(hip_ctx, rows, routed, identity, top, ff, d):
    """... at sizes whose operands go by LDS DMA: the gated product in the first product's epilogue, odd and many buckets (the most that form takes), a hidden width that is no whole
    tile.  The forms sum in other orders, so a hidden value h can round to the neighbouring bf16: a result then moves by 2^-8 |h| |w| of its down weight, a few of which may meet."""
    rng = np.random.default_rng(rows)
    x, wr = f32(rng.standard_normal((rows, d))), O.to_bf16(rng.standard_normal((routed + identity, d)) * 0.5)
    corr, res = f32(0.1 * rng.standard_normal(routed + identity)), f32(rng.standard_normal((rows, d)))
    w13 = O.to_bf16(rng.standard_normal((routed, 2 * ff, d), dtype=np.float32) / np.float32(np.sqrt(d)))
    w2 = O.to_bf16(rng.standard_normal((routed, d, ff), dtype=np.float32) / np.float32(np.sqrt(ff)))
    b13, b2, outs = O.bf16_bits(w13), O.bf16_bits(w2), []
    for mode in (1, 2):
        y, ids, wts = np.empty((rows, d), dtype=np.float32), np.empty((rows, top), dtype=np.int32), np.empty((rows, top), dtype=np.float32)
        _ffi.call("uzu_hip_s32_moe", hip_ctx._h, ptr(x), ptr(O.bf16_bits(wr)), ptr(corr), ptr(b13), ptr(b2), ptr(res), ptr(y), ptr(ids), ptr(wts), C.c_uint32(rows), C.c_uint32(d),
                  C.c_uint32(ff), C.c_uint32(routed), C.c_uint32(identity), C.c_uint32(top), C.c_uint32(mode))
        outs.append(y)
    up, gate = np.split(O.to_bf16(x[:64]) @ w13[0].T, 2, axis=1)
    h = np.abs(gate / (1 + np.exp(-gate)) * up).max()
    assert np.isfinite(outs[1]).all() and np.abs(outs[0] - outs[1]).max() < 2 * 2.0 ** -8 * h * np.abs(w2).max()
    assert np.linalg.norm(outs[0] - outs[1]) < 1e-4 * np.linalg.norm(outs[0])


@pytest.mark.parametrize("rows,n,k,batch,act", [(3, 4097, 64, 1, 0), (5, 15, 128, 1, 1), (8, 70, 1024, 1, 0), (16, 4100, 2048, 1, 1), (7, 48, 192, 3, 0), (15, 2048, 4096, 1, 0), (17, 33, 64, 1, 1),
                                                (31, 1030, 1024, 1, 0), (32, 8191, 320, 1, 0), (9, 2100, 64, 2, 0), (20, 300, 4096, 1, 0), (24, 8200, 1024, 1, 1), (8, 70, 448, 1, 0), (6, 1990, 1024, 1, 0)])
def test_linear_of_a_few_rows(hip_ctx, rows, n, k, batch, act):
    """bf16 products of 3 to 32 rows: ragged rows and outputs, one chunk of the contraction and many (fewer than waves, no multiple of them), the per-head form, bias, activation and
    residual; f32 sums of bf16 products, the bound of the other matrix-core forms"""
    rng = np.random.default_rng(rows + n)
    x, w = f32(rng.standard_normal((rows, k * batch))), O.to_bf16(rng.standard_normal((batch, n, k)))
    b = O.to_bf16(rng.standard_normal(n)) if batch == 1 else None
    res = f32(rng.standard_normal((rows, n))) if batch == 1 else None
    got = linear(hip_ctx, x, w, b, res, batch=batch, act=act, bf16=1)
    xb = O.to_bf16(x).astype(np.float64)
    want = np.concatenate([xb[:, z * k:(z + 1) * k] @ w[z].T.astype(np.float64) for z in range(batch)], axis=1)
    if batch == 1:
        want = (np.maximum(want + b, 0) ** 2 if act else want + b) + res
    assert np.abs(got - want).max() <= 3e-5 * max(1.0, np.abs(want).max())


def test_experts_of_a_few_rows_refuse_a_row_that_fits_no_workgroup(hip_ctx):
    """A width that one row's step refuses (its input does not fit the workgroup's LDS) is refused for a few rows as well: a model is served at every row count or not at all."""
    d, ff = 12352, 64
    x, w = np.ones((2, d), np.float32), np.zeros((1, 2 * ff, d), np.uint16)
    y, ids, wts = np.empty((2, d), np.float32), np.empty((2, 1), np.int32), np.empty((2, 1), np.float32)
    for rows in (1, 2):
        with pytest.raises(_ffi.UzuHipError, match="LDS row"):
            _ffi.call("uzu_hip_s32_moe", hip_ctx._h, ptr(x), ptr(w), ptr(np.zeros(1, np.float32)), ptr(w), ptr(w), ptr(x), ptr(y), ptr(ids), ptr(wts), C.c_uint32(rows), C.c_uint32(d),
                      C.c_uint32(ff), C.c_uint32(1), C.c_uint32(0), C.c_uint32(1), C.c_uint32(1))


@pytest.mark.parametrize("rows,n,k", [(3, 4112, 1024), (8, 2048, 4096), (16, 520, 2048), (24, 1024, 2048), (12, 300, 1024), (16, 520, 512), (12, 300, 256), (12, 1500, 2048)])
def test_linear_of_a_few_rows_sums(hip_ctx, rows, n, k):
    """How far the f32 sums are from 64 bits, held to the sums a wave per column makes (64 lanes that add every 64th product one by one, then in pairs; products of bf16 numbers are
    exact): no further, with 5 % for the chance of the inputs."""
    rng = np.random.default_rng(rows + n + k)
    x, w = O.to_bf16(rng.standard_normal((rows, k))).astype(np.float32), O.to_bf16(rng.standard_normal((n, k))).astype(np.float32)
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    lanes = np.zeros((rows, n, 64), dtype=np.float32)
    for at in range(0, k, 64):
        lanes += x[:, None, at:at + 64] * w[None, :, at:at + 64]
    while lanes.shape[-1] > 1:
        lanes = lanes[..., ::2] + lanes[..., 1::2]
    got = linear(hip_ctx, x, w, act=0, bf16=1)
    assert np.linalg.norm(got - want) <= 1.05 * np.linalg.norm(lanes[..., 0] - want)


@pytest.mark.parametrize("rows,routed,identity,top,ff,d", [(2, 8, 0, 2, 64, 64), (3, 70, 2, 4, 128, 192), (16, 4, 1, 3, 320, 64), (33, 2, 1, 1, 64, 1024), (63, 3, 0, 3, 192, 128), (61, 16, 3, 16, 64, 64),
                                                           (2, 8, 0, 2, 1984, 2112), (3, 70, 2, 4, 640, 704), (16, 4, 1, 3, 512, 64)])
def test_experts_of_a_few_rows(hip_ctx, rows, routed, identity, top, ff, d):
    """bf16 products of 2 to 63 rows: fewer (row, slot) pairs than experts and more, an expert with more pairs than a tile holds, every pair on one expert, identity experts; against 64 bits
    with the router's choice.  A hidden value near the middle of two bf16 numbers may round to the other: a result then moves by 2^-8 |h| |w|, a few of which may meet."""
    rng = np.random.default_rng(rows)
    x, wr = f32(rng.standard_normal((rows, d))), O.to_bf16(rng.standard_normal((routed + identity, d)) * 0.5)
    corr, res = f32(0.1 * rng.standard_normal(routed + identity)), f32(rng.standard_normal((rows, d)))
    w13 = O.to_bf16(rng.standard_normal((routed, 2 * ff, d), dtype=np.float32) / np.float32(np.sqrt(d)))
    w2 = O.to_bf16(rng.standard_normal((routed, d, ff), dtype=np.float32) / np.float32(np.sqrt(ff)))
    y, ids, wts = np.empty((rows, d), dtype=np.float32), np.empty((rows, top), dtype=np.int32), np.empty((rows, top), dtype=np.float32)
    _ffi.call("uzu_hip_s32_moe", hip_ctx._h, ptr(x), ptr(O.bf16_bits(wr)), ptr(corr), ptr(O.bf16_bits(w13)), ptr(O.bf16_bits(w2)), ptr(res), ptr(y), ptr(ids), ptr(wts), C.c_uint32(rows),
              C.c_uint32(d), C.c_uint32(ff), C.c_uint32(routed), C.c_uint32(identity), C.c_uint32(top), C.c_uint32(1))
    want, h_max, xb = res.astype(np.float64), 0.0, O.to_bf16(x).astype(np.float64)
    for r in range(rows):
        for e, wt in zip(ids[r], wts[r].astype(np.float64)):
            if e >= routed:
                want[r] += wt * x[r]
                continue
            up, gate = np.split(w13[e].astype(np.float64) @ xb[r], 2)
            h = gate / (1 + np.exp(-gate)) * up
            h_max = max(h_max, np.abs(h).max())
            want[r] += wt * (w2[e].astype(np.float64) @ O.to_bf16(h.astype(np.float32)).astype(np.float64))
    err = np.abs(y - want)
    assert err.max() <= 2 * 2.0 ** -8 * h_max * np.abs(w2).max() + 1e-5 and np.linalg.norm(err) < 1e-4 * np.linalg.norm(want)
