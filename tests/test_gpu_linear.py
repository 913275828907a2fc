"""GPU parity of qa_linear / qa_mlp_fused against the oracle.

Every case calls the product through the C ABI (csrc/libqa.so) on an MI355X
and compares with oracle/ (the CPU restatement of src/cpu_tensor.rs /
src/cpu_decoder.rs / src/audio_encoder.rs linear semantics) on identical 16-bit
inputs.  Tolerance (north star, f16 outputs): max relative error <= 1e-2 with
the max(|r|, 1e-3 max|r|) floor, mean absolute error <= 1e-3.  In addition,
above that floor every output must be within 1 ulp of the f64-exact oracle:
one rounding of an f32 accumulator whose error is far below half an ulp.
SiLU.up rounds three times (g, u, then the product): g and u may each land
one ulp (plus the f32 summation error) away from the exactly rounded value,
and that perturbation, propagated through silu(g)*u, bounds each output
elementwise (conftest.silu_mul_bound); in bf16 (ulp 2^-7 relative) its
relative bound is 0.03.  bf16 composites (the MLP block) are gated per stage
on identical inputs, as the reference's per-op rounding contract states.
"""
from __future__ import annotations

import os

import numpy as np
import pytest

from conftest import MAE_TOL, REL_TOL, assert_parity, assert_silu_mul, parity_stats

pytestmark = pytest.mark.gpu

SILU_REL = {0: 1e-2, 1: 0.03}


def _h16(orc, x, dtype):
    return orc.h16_from_f32(np.asarray(x, np.float32), dtype)


def _run(ctx, pkg, dtype, a, w, c0, *, flags=0, bias=None, m=None, n=None, k=None, **kw):
    m = a.shape[0] if m is None else m
    k = a.shape[1] if k is None else k
    if n is None:
        n = w.shape[1] if flags & pkg.TRANSB else w.shape[0]
    da, dw, dc = ctx.to_device(a), ctx.to_device(w), ctx.to_device(c0)
    db = ctx.to_device(bias) if bias is not None else None
    ctx.linear(pkg.linear_desc(dtype, m, n, k, da, dw, dc, flags=flags, bias=db,
                               ldc=c0.shape[-1], **kw))
    out = ctx.download(dc, c0.shape)
    for b in (da, dw, dc, db):
        if b is not None:
            b.free()
    return out


def _case(rng, orc, dtype, m, n, k, *, w_std=0.02, transb=False):
    a = _h16(orc, rng.standard_normal((m, k)), dtype)
    wshape = (k, n) if transb else (n, k)
    w = _h16(orc, w_std * rng.standard_normal(wshape), dtype)
    return a, w


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
def test_config1_up_projection(ctx, pkg, orc, dtype):
    """x [256,1024] ~ N(0,1), W [3072,1024] ~ N(0,0.02), seed 0."""
    rng = np.random.default_rng(0)
    a, w = _case(rng, orc, dtype, 256, 3072, 1024)
    c0 = np.zeros((256, 3072), np.uint16)
    got = _run(ctx, pkg, dtype, a, w, c0)
    want = orc.linear(dtype, a, w, c0.copy())
    exact = orc.linear(dtype, a, w, c0.copy(), flags=orc.EXACT)
    s = assert_parity(got, want, orc, dtype)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)
    assert s["identical"] > 0.9, s


SHAPES = [
    (1, 128, 64), (7, 384, 16), (64, 384, 1024), (100, 136, 200), (129, 256, 72),
    (255, 512, 320), (300, 1024, 4320 // 8 * 8), (513, 640, 192),
]


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_plain_ragged_shapes(ctx, pkg, orc, dtype, m, n, k):
    rng = np.random.default_rng(m * 7 + n + k)
    a, w = _case(rng, orc, dtype, m, n, k)
    c0 = np.zeros((m, n), np.uint16)
    got = _run(ctx, pkg, dtype, a, w, c0)
    exact = orc.linear(dtype, a, w, c0.copy(), flags=orc.EXACT)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("epi", ["bias", "acc", "bias_acc", "gelu", "bias_gelu"])
def test_epilogues(ctx, pkg, orc, dtype, epi):
    rng = np.random.default_rng(11)
    m, n, k = 200, 384, 256
    a, w = _case(rng, orc, dtype, m, n, k)
    bias = _h16(orc, 0.01 * rng.standard_normal(n) * 10, dtype) if "bias" in epi else None
    flags = 0
    if "acc" in epi:
        flags |= pkg.ACCUMULATE
        c0 = _h16(orc, rng.standard_normal((m, n)), dtype)
    else:
        c0 = np.zeros((m, n), np.uint16)
    if "gelu" in epi:
        flags |= pkg.EPI_GELU
    got = _run(ctx, pkg, dtype, a, w, c0, flags=flags, bias=bias)
    exact = orc.linear(dtype, a, w, c0.copy(), flags=flags | orc.EXACT, bias=bias)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,inter,hidden", [(1, 64, 64), (37, 192, 128), (512, 3072, 1024)])
def test_silu_mul_epilogue(ctx, pkg, orc, dtype, m, inter, hidden):
    rng = np.random.default_rng(5)
    a = _h16(orc, rng.standard_normal((m, hidden)), dtype)
    w = _h16(orc, 0.05 * rng.standard_normal((2 * inter, hidden)), dtype)
    c0 = np.zeros((m, inter), np.uint16)
    got = _run(ctx, pkg, dtype, a, w, c0, flags=pkg.EPI_SILU_MUL)
    want = orc.linear(dtype, a, w, c0.copy(), flags=orc.EPI_SILU_MUL)
    exact = orc.linear(dtype, a, w, c0.copy(), flags=orc.EPI_SILU_MUL | orc.EXACT)
    gu_exact = orc.linear(dtype, a, w, np.zeros((m, 2 * inter), np.uint16), flags=orc.EXACT)
    assert_parity(got, want, orc, dtype, rel_tol=SILU_REL[dtype])
    assert_silu_mul(got, exact, a, w, gu_exact, orc, dtype, hidden, rel_tol=SILU_REL[dtype])


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("flags_name", ["plain", "bias_rows_gelu"])
def test_transb_conv_operand(ctx, pkg, orc, dtype, flags_name):
    """gemm_conv form: C[ch, pos] = Wconv[ch, K] . col[K, pos] (transb)."""
    rng = np.random.default_rng(3)
    m, n, k = 192, 520, 144  # channels, positions, 16*9 taps
    a = _h16(orc, 0.05 * rng.standard_normal((m, k)), dtype)
    w = _h16(orc, rng.standard_normal((k, n)), dtype)
    flags, bias = pkg.TRANSB, None
    if flags_name == "bias_rows_gelu":
        flags |= pkg.BIAS_ROWS | pkg.EPI_GELU
        bias = _h16(orc, 0.1 * rng.standard_normal(m), dtype)
    c0 = np.zeros((m, n), np.uint16)
    got = _run(ctx, pkg, dtype, a, w, c0, flags=flags, bias=bias)
    exact = orc.linear(dtype, a, w, c0.copy(), flags=flags | orc.EXACT, bias=bias)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
def test_batched(ctx, pkg, orc, dtype):
    rng = np.random.default_rng(9)
    batch, m, n, k = 3, 70, 128, 96
    a = _h16(orc, rng.standard_normal((batch, m, k)), dtype)
    w = _h16(orc, 0.1 * rng.standard_normal((batch, n, k)), dtype)
    c0 = np.zeros((batch, m, n), np.uint16)
    got = _run(ctx, pkg, dtype, a.reshape(batch * m, k), w.reshape(batch * n, k),
               c0.reshape(batch * m, n), m=m, n=n, k=k, batch=batch, bsa=m * k, bsb=n * k,
               bsc=m * n)
    want = orc.linear(dtype, a, w, c0.copy(), flags=orc.EXACT, m=m, n=n, k=k, batch=batch,
                      bsa=m * k, bsb=n * k, bsc=m * n)
    assert_parity(got.reshape(batch, m, n), want, orc, dtype, ulp_tol=1)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
def test_batched_long_k_is_never_split(ctx, pkg, orc, dtype):
    """A batched call whose shape alone would make the planner split K (few
    tiles, long K) runs unsplit instead of failing with QA_EUNSUPPORTED: the
    planner, not the caller's valid shape, decides the split."""
    rng = np.random.default_rng(19)
    batch, m, n, k = 3, 64, 128, 4096
    a = _h16(orc, rng.standard_normal((batch, m, k)), dtype)
    w = _h16(orc, 0.02 * rng.standard_normal((batch, n, k)), dtype)
    c0 = np.zeros((batch, m, n), np.uint16)
    got = _run(ctx, pkg, dtype, a.reshape(batch * m, k), w.reshape(batch * n, k),
               c0.reshape(batch * m, n), m=m, n=n, k=k, batch=batch, bsa=m * k, bsb=n * k,
               bsc=m * n)
    want = orc.linear(dtype, a, w, c0.copy(), flags=orc.EXACT, m=m, n=n, k=k, batch=batch,
                      bsa=m * k, bsb=n * k, bsc=m * n)
    assert_parity(got.reshape(batch, m, n), want, orc, dtype, ulp_tol=1)
    # a split forced through the environment is not applied to a batched call either
    os.environ["QA_SPLITS"] = "4"
    try:
        got2 = _run(ctx, pkg, dtype, a.reshape(batch * m, k), w.reshape(batch * n, k),
                    c0.reshape(batch * m, n), m=m, n=n, k=k, batch=batch, bsa=m * k,
                    bsb=n * k, bsc=m * n)
    finally:
        del os.environ["QA_SPLITS"]
    assert np.array_equal(got2, got)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 5, 6, 7, 9])
@pytest.mark.parametrize("splits", [1, 2, 3, 5])
def test_forced_tiles_and_splits(ctx, pkg, orc, tile, splits, dtype):
    """Every tile shape, with and without split-K (incl. uneven k ranges), in
    both formats: bias + residual, bias + GELU, and SiLU.up."""
    rng = np.random.default_rng(tile * 10 + splits + 100 * dtype)
    m, n, k = 300, 512, 1216
    a, w = _case(rng, orc, dtype, m, n, k)
    c0 = _h16(orc, rng.standard_normal((m, n)), dtype)
    bias = _h16(orc, 0.1 * rng.standard_normal(n), dtype)
    os.environ["QA_TILE"], os.environ["QA_SPLITS"] = str(tile), str(splits)
    try:
        got = _run(ctx, pkg, dtype, a, w, c0, flags=pkg.ACCUMULATE, bias=bias)
        again = _run(ctx, pkg, dtype, a, w, c0, flags=pkg.ACCUMULATE, bias=bias)
        gelu = _run(ctx, pkg, dtype, a, w, np.zeros_like(c0), flags=pkg.EPI_GELU, bias=bias)
        gu_w = _h16(orc, 0.05 * rng.standard_normal((2 * 256, k)), dtype)
        act = _run(ctx, pkg, dtype, a, gu_w, np.zeros((m, 256), np.uint16), flags=pkg.EPI_SILU_MUL)
    finally:
        del os.environ["QA_TILE"], os.environ["QA_SPLITS"]
    exact = orc.linear(dtype, a, w, c0.copy(), flags=orc.ACCUMULATE | orc.EXACT, bias=bias)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)
    assert np.array_equal(got, again), "split-K reduction must be deterministic"
    gelu_exact = orc.linear(dtype, a, w, np.zeros_like(c0), flags=orc.EPI_GELU | orc.EXACT,
                            bias=bias)
    assert_parity(gelu, gelu_exact, orc, dtype, ulp_tol=1)
    act_exact = orc.linear(dtype, a, gu_w, np.zeros((m, 256), np.uint16),
                           flags=orc.EPI_SILU_MUL | orc.EXACT)
    gu_exact = orc.linear(dtype, a, gu_w, np.zeros((m, 512), np.uint16), flags=orc.EXACT)
    assert_silu_mul(act, act_exact, a, gu_w, gu_exact, orc, dtype, k, rel_tol=SILU_REL[dtype])


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("tile", [10, 11])
@pytest.mark.parametrize("splits", [1, 3])
def test_forced_32_row_tiles(ctx, pkg, orc, tile, splits, dtype):
    """The 32-row tiles as the others above (11 has no SiLU.up: 10 takes it)."""
    test_forced_tiles_and_splits(ctx, pkg, orc, tile, splits, dtype)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("tile", [10, 11])
@pytest.mark.parametrize("m,n,k", [(1, 4, 8), (31, 36, 72), (33, 60, 120), (32, 64, 128), (65, 100, 1544)])
def test_32_row_tile_edges(ctx, pkg, orc, tile, m, n, k, dtype):
    """Rows, columns and k at the edges of the 32-row tiles: k ranges inside
    one 16-deep slice group, one plane, one stage, and past the ring; residual
    and bias (the preloaded words) and plain."""
    rng = np.random.default_rng(m * n + k + tile + dtype)
    a, w = _case(rng, orc, dtype, m, n, k, w_std=0.1)
    c0 = _h16(orc, rng.standard_normal((m, n)), dtype)
    bias = _h16(orc, 0.1 * rng.standard_normal(n), dtype)
    os.environ["QA_TILE"] = str(tile)
    try:
        got = _run(ctx, pkg, dtype, a, w, c0, flags=pkg.ACCUMULATE, bias=bias)
        plain = _run(ctx, pkg, dtype, a, w, c0)
    finally:
        del os.environ["QA_TILE"]
    exact = orc.linear(dtype, a, w, c0.copy(), flags=orc.ACCUMULATE | orc.EXACT, bias=bias)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)
    assert_parity(plain, orc.linear(dtype, a, w, np.zeros_like(c0), flags=orc.EXACT), orc, dtype, ulp_tol=1)


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
@pytest.mark.parametrize("group_m", [1, 3, 5, 8, 1000])
@pytest.mark.parametrize("tile,splits", [(4, 1), (0, 1), (3, 2), (5, 1), (6, 1), (7, 1), (7, 3),
                                         (9, 1), (9, 2)])
def test_tile_enumeration_bands(ctx, pkg, orc, group_m, tile, splits, dtype):
    """Every band height of the tile enumeration (including ones that do not
    divide the tile grid, and more than its height) maps blocks onto tiles
    one to one: C starts as noise and must end equal to the exactly rounded
    result everywhere (a tile computed twice leaves another one untouched).
    Plain, bias + GELU and SiLU.up epilogues, both formats."""
    rng = np.random.default_rng(40 + group_m + 10 * tile + 1000 * dtype)
    m, n, k = 600, 1472, 640   # ragged in m and n for every tile shape
    a, w = _case(rng, orc, dtype, m, n, k)
    c0 = _h16(orc, rng.standard_normal((m, n)), dtype)
    bias = _h16(orc, 0.1 * rng.standard_normal(n), dtype)
    os.environ.update(QA_TILE=str(tile), QA_SPLITS=str(splits), QA_GROUP_M=str(group_m))
    try:
        got = _run(ctx, pkg, dtype, a, w, c0)
        gelu = _run(ctx, pkg, dtype, a, w, c0, flags=pkg.EPI_GELU, bias=bias)
        gu_w = _h16(orc, 0.05 * rng.standard_normal((2 * 736, k)), dtype)
        act = _run(ctx, pkg, dtype, a, gu_w, np.zeros((m, 736), np.uint16), flags=pkg.EPI_SILU_MUL)
    finally:
        for key in ("QA_TILE", "QA_SPLITS", "QA_GROUP_M"):
            del os.environ[key]
    exact = orc.linear(dtype, a, w, np.zeros_like(c0), flags=orc.EXACT)
    assert_parity(got, exact, orc, dtype, ulp_tol=1)
    gelu_exact = orc.linear(dtype, a, w, np.zeros_like(c0), flags=orc.EPI_GELU | orc.EXACT,
                            bias=bias)
    assert_parity(gelu, gelu_exact, orc, dtype, ulp_tol=1)
    act_exact = orc.linear(dtype, a, gu_w, np.zeros((m, 736), np.uint16),
                           flags=orc.EPI_SILU_MUL | orc.EXACT)
    gu_exact = orc.linear(dtype, a, gu_w, np.zeros((m, 1472), np.uint16), flags=orc.EXACT)
    assert_silu_mul(act, act_exact, a, gu_w, gu_exact, orc, dtype, k, rel_tol=SILU_REL[dtype])


@pytest.mark.parametrize("dtype", [0, 1], ids=["f16", "bf16"])
def test_mlp_fused_config2(ctx, pkg, orc, dtype):
    """out = down(SiLU(x Wg^T) * (x Wu^T)) + x, M=512."""
    rng = np.random.default_rng(2)
    m, hid, inter = 512, 1024, 3072
    x = _h16(orc, rng.standard_normal((m, hid)), dtype)
    wgu = _h16(orc, 0.02 * rng.standard_normal((2 * inter, hid)), dtype)
    wd = _h16(orc, 0.02 * rng.standard_normal((hid, inter)), dtype)
    dx, dgu, dwd = ctx.to_device(x), ctx.to_device(wgu), ctx.to_device(wd)
    dact = ctx.alloc(m * inter * 2)
    ctx.mlp_fused(pkg.MlpDesc(dtype=dtype, flags=0, m=m, hidden=hid, inter=inter, x=dx.ptr,
                              w_gu=dgu.ptr, w_down=dwd.ptr, act=dact.ptr, h=dx.ptr))
    got = ctx.download(dx, (m, hid))
    got_act = ctx.download(dact, (m, inter))
    for b in (dx, dgu, dwd, dact):
        b.free()
    act = orc.linear(dtype, x, wgu, np.zeros((m, inter), np.uint16), flags=orc.EPI_SILU_MUL)
    assert_parity(got_act, act, orc, dtype, rel_tol=SILU_REL[dtype])
    if dtype == 0:
        # f16: the whole block against the CPU path.  A one-ulp difference in
        # an act element (a rounding tie under a different f32 summation
        # order) reaches h as an absolute error of ~1e-4 through 3072 down
        # weights; where x + mlp(x) cancels to near zero that is a large
        # relative error, so the end-to-end relative floor is 1e-2 max|r|
        # (the per-stage checks above and below keep the 1e-3 floor).
        want = orc.linear(dtype, act, wd, x.copy(), flags=orc.ACCUMULATE)
        s = parity_stats(got, want, orc, dtype)
        assert s["mae"] <= MAE_TOL, s
        g, r = orc.h16_to_f32(got, dtype), orc.h16_to_f32(want, dtype)
        rel = np.abs(g - r) / np.maximum(np.abs(r), 1e-2 * np.abs(r).max())
        assert rel.max() <= REL_TOL, (rel.max(), s)
    # both formats: the down projection on the GPU's own act (identical inputs)
    want = orc.linear(dtype, got_act, wd, x.copy(), flags=orc.ACCUMULATE | orc.EXACT)
    assert_parity(got, want, orc, dtype, ulp_tol=1)


def test_fused_qkv_columns_match_separate(ctx, pkg, orc):
    """[q|k|v] fused rows (src/decoder.rs:840-871): fused output columns equal
    the separate projections, which is what the CPU decoder runs
    (src/cpu_decoder.rs:456-458)."""
    rng = np.random.default_rng(4)
    m, hid = 160, 1024
    x = _h16(orc, rng.standard_normal((m, hid)), 0)
    wq = _h16(orc, 0.02 * rng.standard_normal((2048, hid)), 0)
    wk = _h16(orc, 0.02 * rng.standard_normal((1024, hid)), 0)
    wv = _h16(orc, 0.02 * rng.standard_normal((1024, hid)), 0)
    fused = _run(ctx, pkg, 0, x, np.concatenate([wq, wk, wv]), np.zeros((m, 4096), np.uint16))
    for lo, wpart in ((0, wq), (2048, wk), (3072, wv)):
        sep = orc.linear(0, x, wpart, np.zeros((m, wpart.shape[0]), np.uint16))
        assert_parity(fused[:, lo:lo + wpart.shape[0]], sep, orc, 0)


def test_zero_rows_is_a_noop(ctx, pkg, orc):
    a = np.zeros((8, 64), np.uint16)
    w = np.zeros((128, 64), np.uint16)
    c0 = np.full((8, 128), 0x3C00, np.uint16)
    got = _run(ctx, pkg, 0, a, w, c0, m=0)
    assert np.array_equal(got, c0)


def test_accumulate_with_zero_a_keeps_c(ctx, pkg, orc):
    rng = np.random.default_rng(8)
    m, n, k = 64, 256, 128
    a = np.zeros((m, k), np.uint16)
    w = _h16(orc, rng.standard_normal((n, k)), 0)
    c0 = _h16(orc, rng.standard_normal((m, n)), 0)
    got = _run(ctx, pkg, 0, a, w, c0, flags=pkg.ACCUMULATE)
    assert np.array_equal(got, c0)


def test_time_next_launch_stamps_the_kernel(ctx, pkg, orc):
    """qa_time_next_launch: the next GEMM's dispatch records its start and end
    into the caller's HIP events (a positive interval below the whole
    launch-to-sync time), the result is the same as without the events, and
    the launch after it records nothing (the events are taken over once)."""
    import ctypes
    import time

    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float), ctypes.c_void_p,
                                        ctypes.c_void_p]
    hip.hipEventDestroy.argtypes = [ctypes.c_void_p]
    ev = [ctypes.c_void_p(), ctypes.c_void_p()]
    for e in ev:
        assert hip.hipEventCreate(ctypes.byref(e)) == 0
    rng = np.random.default_rng(12)
    m, n, k = 1024, 1024, 2048
    a = _h16(orc, rng.standard_normal((m, k)), 0)
    w = _h16(orc, 0.02 * rng.standard_normal((n, k)), 0)
    c0 = np.zeros((m, n), np.uint16)
    plain = _run(ctx, pkg, 0, a, w, c0)
    da, dw, dc = ctx.to_device(a), ctx.to_device(w), ctx.to_device(c0)
    desc = pkg.linear_desc(0, m, n, k, da, dw, dc)
    try:
        ctx.sync()
        t = time.perf_counter()
        pkg.check(pkg.lib().qa_time_next_launch(ctx.handle, ev[0], ev[1]))
        ctx.linear(desc)
        ctx.sync()
        wall_ms = (time.perf_counter() - t) * 1e3
        ms = ctypes.c_float()
        assert hip.hipEventElapsedTime(ctypes.byref(ms), ev[0], ev[1]) == 0
        assert 0.0 < ms.value < wall_ms, (ms.value, wall_ms)
        stamped = ctx.download(dc, c0.shape)
        ctx.linear(desc)  # no events: the hook was cleared by the launch above
        ctx.sync()
        again = ctx.download(dc, c0.shape)
    finally:
        for b in (da, dw, dc):
            b.free()
        for e in ev:
            hip.hipEventDestroy(e)
    assert np.array_equal(stamped, plain)
    assert np.array_equal(again, plain)


def test_time_next_launch_spans_the_split_k_reduce(ctx, pkg, orc):
    """With K split, the GEMM kernel's dispatch stamps the start event and the
    split-K reduce kernel's the stop event: a positive interval, and the
    result (GEMM + reduce + residual) within 1 ulp of the exactly rounded one."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float), ctypes.c_void_p,
                                        ctypes.c_void_p]
    hip.hipEventDestroy.argtypes = [ctypes.c_void_p]
    ev = [ctypes.c_void_p(), ctypes.c_void_p()]
    for e in ev:
        assert hip.hipEventCreate(ctypes.byref(e)) == 0
    rng = np.random.default_rng(13)
    m, n, k = 512, 1024, 3072
    a = _h16(orc, rng.standard_normal((m, k)), 0)
    w = _h16(orc, 0.02 * rng.standard_normal((n, k)), 0)
    c0 = _h16(orc, rng.standard_normal((m, n)), 0)
    da, dw, dc = ctx.to_device(a), ctx.to_device(w), ctx.to_device(c0)
    desc = pkg.linear_desc(0, m, n, k, da, dw, dc, flags=pkg.ACCUMULATE)
    os.environ["QA_SPLITS"] = "2"
    try:
        pkg.check(pkg.lib().qa_time_next_launch(ctx.handle, ev[0], ev[1]))
        ctx.linear(desc)
        ctx.sync()
        ms = ctypes.c_float()
        assert hip.hipEventElapsedTime(ctypes.byref(ms), ev[0], ev[1]) == 0
        assert ms.value > 0.0, ms.value
        got = ctx.download(dc, c0.shape)
    finally:
        del os.environ["QA_SPLITS"]
        for b in (da, dw, dc):
            b.free()
        for e in ev:
            hip.hipEventDestroy(e)
    exact = orc.linear(0, a, w, c0.copy(), flags=orc.ACCUMULATE | orc.EXACT)
    assert_parity(got, exact, orc, 0, ulp_tol=1)


def test_stamped_per_launch_timer(ctx, pkg, orc):
    """qah_time_linears_stamped (the benchmark's kernel-only per-launch
    figures): positive per launch, and each launch's kernel time is at most
    the event-to-event interval of the same back-to-back launches (which adds
    the gap between them), compared on medians; unsplit and split-K."""
    from qwen3_aligner_wgpu_amd import host

    rng = np.random.default_rng(14)
    m, n, k = 512, 1024, 3072
    a = _h16(orc, rng.standard_normal((m, k)), 0)
    w = _h16(orc, 0.02 * rng.standard_normal((n, k)), 0)
    da, dw, dc = ctx.to_device(a), ctx.to_device(w), ctx.alloc(m * n * 2)
    desc = pkg.linear_desc(0, m, n, k, da, dw, dc)
    try:
        for splits in ("1", "2"):
            os.environ["QA_SPLITS"] = splits
            try:
                kern = host.time_linears_stamped(ctx, [desc], 5, 40)
                each = host.time_linears_each(ctx, [desc], 5, 40)
            finally:
                del os.environ["QA_SPLITS"]
            assert (kern > 0).all(), kern
            assert np.median(kern) <= np.median(each) * 1.05, (splits, np.median(kern),
                                                               np.median(each))
    finally:
        for b in (da, dw, dc):
            b.free()


@pytest.mark.parametrize("seed", [1, 2])
def test_silu_f16_packed_arithmetic_is_f32_then_f16(ctx, pkg, seed):
    """The f16 SiLU.up epilogue's packed arithmetic (v_fma_mix on f16 operands,
    paired conversions) gives, bit for bit, silu_mul in f32 followed by one
    round-to-nearest-even to f16 (the reference shader's order, src/shaders.rs:
    1411-1450), on 16.7 M inputs per seed: special values (+-0, subnormals, f16
    overflow), random f32 bit patterns and ordinary values."""
    from qwen3_aligner_wgpu_amd import host

    assert host.check_silu_f16x2(ctx, 1 << 23, seed) == 0


def test_gelu_epilogue_rounds_like_the_exact_gelu(ctx, pkg, orc):
    """GELU of every 16-bit value from 2^-10 to 10 in size (w picks one
    element of the row, so the sum is the value itself).  Near zero an f32
    evaluation with relative error d moves a result over one of f16's rounding
    boundaries for a share d * 2^11 of the values at most: 3.1e-4 for the
    1.5e-7 that gelu_erf keeps up to 0.1.  A bf16 result is within an ulp of the
    exact one down to -7, where the tail's relative error is 8e-4 (ulp 4e-3)."""
    from scipy.special import erfc
    for dtype in (0, 1):
        with np.errstate(invalid="ignore"):  # the NaN patterns
            x = orc.h16_to_f32(np.arange(1 << 16, dtype=np.uint16), dtype).astype(np.float64)
        keep = np.isfinite(x) & (np.abs(x) >= 2.0 ** -10) & (np.abs(x) <= 10.0)
        bits, x = np.flatnonzero(keep).astype(np.uint16), x[keep]
        a = np.zeros((len(bits), 8), np.uint16)
        a[:, 0] = bits
        w = _h16(orc, np.eye(1, 8).repeat(4, 0), dtype)
        got = _run(ctx, pkg, dtype, a, w, np.zeros((len(bits), 4), np.uint16), flags=pkg.EPI_GELU)
        assert (got == got[:, :1]).all()
        exact = 0.5 * x * erfc(-x / np.sqrt(2.0))
        if dtype == 0:
            small = np.abs(x) <= 0.1
            assert (got[small, 0] != exact[small].astype(np.float16).view(np.uint16)).mean() <= 5e-4
        else:
            part = x >= -7.0
            v = orc.h16_to_f32(got[part, 0].copy(), dtype).astype(np.float64)
            assert (np.abs(v - exact[part]) <= 2.0 ** (np.floor(np.log2(np.abs(exact[part]))) - 7)).all()
